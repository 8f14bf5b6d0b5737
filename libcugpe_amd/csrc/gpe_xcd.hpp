// Whole runs of steps of a small lattice in one kernel on one XCD.
//
// A lattice of a few ten thousand points is bound by latency: the four to ten
// passes of a step each take 4-7 us from launch to drained stores, and the
// host spends 2.5-4 us on each launch, while the state streams through an L2
// in well under a microsecond.  Here workgroups of one XCD stay for all steps
// of a launch and walk the same passes (zwave_tile, plane_tile, the turn-around
// tiles of lean_body: the same arithmetic, so the same bits) with a barrier
// between them.  They share the XCD's L2, so a pass's stores need only to have
// reached it (vmcnt 0) before the barrier, and the next pass's loads only to
// pass the CU's own L1 by (ld_l2); nothing is written back to memory or
// invalidated (an agent acquire fence per barrier took a 32^3 complex64 step
// from 20 to 61 us).  Of its 14.6 us, the four barriers take 0.9 us each, the x
// turn-arounds 1.9 and the planes about 3.5: chains of one wave's
// instructions, so the tasks of a pass go to the CUs before their SIMDs.
//
// Who takes part: the grid covers every CU, each workgroup reads its XCC_ID,
// and those of the wanted XCD register.  The first to register closes the
// registration when `want` workgroups are in or after a bounded wait, and
// publishes their number; a workgroup that comes later leaves.  The barriers
// count registered workgroups only.  Those are all running, so every wait
// ends whatever else occupies the GPU, and no launch order, grid size or
// residency is relied on.  If no workgroup ran on the wanted XCD, the last
// one to leave does the whole run alone.
#pragma once

#include "gpe_plane.hpp"

namespace gpe {

// queue words, all zero at launch; the run clears the words of the next one
constexpr unsigned kXqState = 0, kXqLeft = 32, kXqBar = 64, kXqGroup = 96, kXqWords = 128;
constexpr unsigned kXqClosed = 1u << 31;

template <typename T>
struct XcdArgs {
    PassArgs<T> a;                                  // physics, tables, psi, vbuf, scal, partials
    cplx<T>* B;                                     // predictor array
    const cplx<T>*twx, *twlox, *twy, *twloy, *twz, *twloz;
    int nt;
    unsigned *q, *qnext;
    unsigned xcd, want;
};

constexpr int kXcdMaxLen = 64;
constexpr bool xcd_length(int N) {
    return N == 8 || N == 12 || N == 16 || N == 24 || N == 32 || N == 48 || N == 64;
}

__device__ __forceinline__ unsigned xq_load(const unsigned* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned xq_add(unsigned* p, unsigned v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// columns of a turn-around tile: about 1024 points, one wave or two of butterflies
template <typename T, int N>
constexpr int xcd_wd() {
    const int w = tile_w<T, N>() * N / 1024;
    return w > 0 ? w : 1;
}

template <typename T, int NZ>
struct XcdLds {
    static constexpr int ZX = ZW<T, NZ>::WAVES * ZW<T, NZ>::WAVE;
    static constexpr int TX = 2048;  // covers every turn-around tile with its pad
    TwE<T> twz[NZ], twy[kXcdMaxLen], twx[kXcdMaxLen];
    T vz[NZ];
    cplx<T> x[ZX > TX ? ZX : TX];
    double red[kThreads / 64];
    double scal[2];
    unsigned idx, group;
};

template <typename T>
__device__ __forceinline__ void xcd_table(TwE<T>* t, const cplx<T>* tw, const cplx<T>* lo, int n) {
    for (int i = threadIdx.x; i < n; i += kThreads) {
        if constexpr (sizeof(T) == 4) {
            const cplx<float> h = tw[i], l = lo[i];
            t[i].t = make_float4(h.x, h.y, l.x, l.y);
        } else {
            t[i].t = tw[i];
        }
    }
}

// a value of threadIdx.x the compiler cannot carry over the step loop: what
// is derived from it is recomputed per tile instead of held in registers
__device__ __forceinline__ int xcd_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// barrier over the registered workgroups; target counts all arrivals so far
__device__ __forceinline__ void xcd_barrier(unsigned* q, unsigned group, unsigned& target) {
    target += group;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        (void)xq_add(q + kXqBar, 1u);
        while (xq_load(q + kXqBar) < target) __builtin_amdgcn_s_sleep(1);
    }
    __syncthreads();
}

// turn-around of axis AX (0 x, 1 y) on buf, tiles idx, idx + group, ...
template <typename T, int N, int AX>
__device__ __forceinline__ void xcd_turn_n(const XcdArgs<T>& g, cplx<T>* buf, cplx<T>* lds, const TwE<T>* tw,
                                           unsigned idx, unsigned group) {
    constexpr int WD = xcd_wd<T, N>();
    constexpr unsigned W = (unsigned)lean_w<T, N, WD>();
    static_assert(lds_elems<T, N, (int)W, false>() <= 2048, "tile fits the exchange area");
    PassArgs<T> a = g.a;
    a.M = a.n1 / (unsigned)N;
    a.src = buf;
    a.dst = buf;
    const unsigned tiles = (a.M + W - 1) / W;
    for (unsigned t = idx; t < tiles; t += group) {
        lean_body<T, N, false, -1, 1, WD, MK_SEP, AX, 0, true>(a, lds, tw, nullptr, t, []() {}, xcd_tid());
        __syncthreads();
    }
}
template <typename T, int AX>
__device__ __forceinline__ void xcd_turn(const XcdArgs<T>& g, cplx<T>* buf, cplx<T>* lds, const TwE<T>* tw,
                                         unsigned idx, unsigned group) {
    switch (AX == 0 ? g.a.ph.nx : g.a.ph.ny) {
    case 8: xcd_turn_n<T, 8, AX>(g, buf, lds, tw, idx, group); break;
    case 12: xcd_turn_n<T, 12, AX>(g, buf, lds, tw, idx, group); break;
    case 16: xcd_turn_n<T, 16, AX>(g, buf, lds, tw, idx, group); break;
    case 24: xcd_turn_n<T, 24, AX>(g, buf, lds, tw, idx, group); break;
    case 32: xcd_turn_n<T, 32, AX>(g, buf, lds, tw, idx, group); break;
    case 48: xcd_turn_n<T, 48, AX>(g, buf, lds, tw, idx, group); break;
    default: xcd_turn_n<T, 64, AX>(g, buf, lds, tw, idx, group); break;
    }
}

template <typename T, int NZ>
__device__ __forceinline__ unsigned xcd_ztasks(const XcdArgs<T>& g) {
    return (g.a.n1 / (unsigned)NZ + ZW<T, NZ>::PW - 1) / ZW<T, NZ>::PW;
}

// z pass over the workgroup's wave tasks; with sums, a task's FP64 sum goes to partials[task]
template <typename T, int NZ, int SHAPE, int LM, int MM, bool SUM>
__device__ __forceinline__ void xcd_z(const XcdArgs<T>& g, XcdLds<T, NZ>& S, const cplx<T>* src, cplx<T>* dst,
                                      int flags, unsigned idx, unsigned group) {
    PassArgs<T> a = g.a;
    a.M = a.n1 / (unsigned)NZ;
    a.src = src;
    a.dst = dst;
    a.load_mode = LM;
    a.mid_mode = MM;
    a.store_mode = dst ? STORE_PLAIN : STORE_NONE;
    a.flags = flags;
    a.scal = S.scal;
    // wave tasks go to the workgroups first, then to their waves: a pass with
    // fewer tasks than waves uses every CU
    const unsigned tasks = xcd_ztasks<T, NZ>(g);
    for (unsigned t = idx + group * (threadIdx.x >> 6); t < tasks; t += group * (kThreads / 64)) {
        double acc[3] = {0.0, 0.0, 0.0};
        zwave_tile<T, NZ, SHAPE, LM, MM, true>(a, S.twz, S.vz, S.x, t, acc, xcd_tid());
        if constexpr (SUM) {
            double s = acc[0];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
            if ((threadIdx.x & 63) == 0) g.a.partials[t] = s;
        }
    }
}

// scal[1] = sqrt(npart / sum) by every workgroup for itself, from the tasks'
// sums added in the order of the passes (the four waves of a workgroup's tile,
// then finalize_kernel's)
template <typename T, int NZ>
__device__ __forceinline__ void xcd_norm(const XcdArgs<T>& g, XcdLds<T, NZ>& S) {
    const unsigned tasks = xcd_ztasks<T, NZ>(g);
    double acc = 0.0;
    for (unsigned b = threadIdx.x; b * 4 < tasks; b += kThreads) {
        double s = 0.0;
        for (unsigned t = 4 * b; t < 4 * b + 4 && t < tasks; t++) s += ld_l2(g.a.partials + t);
        acc += s;
    }
    const double sum = block_sum(acc, S.red);
    if (threadIdx.x == 0) {
        S.scal[0] = sum;
        S.scal[1] = sqrt(g.a.ph.npart / sum);
    }
    __syncthreads();
}

// registration of the workgroup: its number among the group's (~0: not in it)
template <typename T>
__device__ __forceinline__ void xcd_join(const XcdArgs<T>& g, unsigned& sidx, unsigned& sgroup) {
    unsigned* q = g.q;
    if (threadIdx.x == 0) {
        // hardware register 20, XCC_ID: bits 0..3
        const unsigned xcc = (unsigned)__builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 15u;
        unsigned idx = ~0u, group = 0;
        if (xcc == g.xcd) {
            const unsigned old = xq_add(q + kXqState, 1u);
            if (!(old & kXqClosed)) {
                idx = old;
                if (old == 0) {
                    for (int i = 0; i < 400 && xq_load(q + kXqState) < g.want; i++) __builtin_amdgcn_s_sleep(2);
                    group = __hip_atomic_fetch_or(q + kXqState, kXqClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(q + kXqGroup, group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    while ((group = xq_load(q + kXqGroup)) == 0) __builtin_amdgcn_s_sleep(1);
                }
            }
        }
        if (idx == ~0u && xq_add(q + kXqLeft, 1u) == gridDim.x - 1) {
            idx = 0;
            group = 1;
        }
        sidx = idx;
        sgroup = group;
    }
    __syncthreads();
    if (sidx == 0)
        for (unsigned i = threadIdx.x; i < kXqWords; i += kThreads) g.qnext[i] = 0u;
}

template <typename T, int NZ, bool ITE>
__global__ __launch_bounds__(kThreads) void xcd_steps_kernel(const XcdArgs<T> g) {
    __shared__ XcdLds<T, NZ> S;
    unsigned* q = g.q;
    xcd_join<T>(g, S.idx, S.group);
    const unsigned idx = __builtin_amdgcn_readfirstlane(S.idx), group = __builtin_amdgcn_readfirstlane(S.group);
    if (idx == ~0u) return;
    {
        PassArgs<T> az = g.a;
        az.tw = g.twz;
        az.twlo = g.twloz;
        zwave_stage<T, NZ>(az, S.twz, S.vz);
    }
    xcd_table<T>(S.twy, g.twy, g.twloy, g.a.ph.ny);
    xcd_table<T>(S.twx, g.twx, g.twlox, g.a.ph.nx);
    __syncthreads();

    cplx<T>*A = g.a.psiA, *B = g.B;
    unsigned bar = 0;
    xcd_z<T, NZ, SHAPE_F, LOAD_PSI0, MID_NONE, false>(g, S, nullptr, B, F_VSTEP1, idx, group);
    for (int s = 0; s < g.nt; s++) {
        const bool last = (s == g.nt - 1);
        // half 0: predictor on B, half 1: corrector on psi
        for (int half = 0; half < 2; half++) {
            cplx<T>* buf = half ? A : B;
            xcd_barrier(q, group, bar);
            xcd_turn<T, 1>(g, buf, S.x, S.twy, idx, group);
            xcd_barrier(q, group, bar);
            xcd_turn<T, 0>(g, buf, S.x, S.twx, idx, group);
            xcd_barrier(q, group, bar);
            if constexpr (!ITE) {
                if (!half) {
                    xcd_z<T, NZ, SHAPE_IF, LOAD_PLAIN, MID_VSTEP2, false>(g, S, B, A, 0, idx, group);
                } else if (!last) {
                    xcd_z<T, NZ, SHAPE_IF, LOAD_PLAIN, MID_VSTEP3, false>(g, S, A, B, F_NEXT_VSTEP1, idx, group);
                } else {
                    xcd_z<T, NZ, SHAPE_I, LOAD_PLAIN, MID_VSTEP3, false>(g, S, A, nullptr, 0, idx, group);
                }
            } else {
                if (!half) xcd_z<T, NZ, SHAPE_I, LOAD_PLAIN, MID_PART1, true>(g, S, B, B, 0, idx, group);
                else xcd_z<T, NZ, SHAPE_I, LOAD_PLAIN, MID_VSTEP3, true>(g, S, A, nullptr, F_RED_NORM, idx, group);
                xcd_barrier(q, group, bar);
                xcd_norm<T, NZ>(g, S);
                if (!half) {
                    xcd_z<T, NZ, SHAPE_F, LOAD_PART2, MID_NONE, false>(g, S, B, A, F_SCALE, idx, group);
                } else if (!last) {
                    xcd_z<T, NZ, SHAPE_F, LOAD_PSI0, MID_NONE, false>(g, S, nullptr, B, F_SCALE | F_VSTEP1, idx, group);
                } else {
                    const T f = (T)S.scal[1];
                    for (unsigned i = idx * kThreads + threadIdx.x; i < g.a.n1; i += group * kThreads)
                        A[i] = cscale(ld_l2(A + i), f);
                    if (idx == 0 && threadIdx.x == 0) {
                        double* sc = const_cast<double*>(g.a.scal);
                        sc[0] = S.scal[0];
                        sc[1] = S.scal[1];
                        sc[2] = -.5 * log(S.scal[0] / g.a.ph.npart) / g.a.ph.dt;
                    }
                }
            }
        }
    }
}

// The same for real time on planes of ny = nz = L points (gpe_plane.hpp): a
// workgroup takes planes idx, idx + group, ..., and a step has four barriers
// instead of six.
template <typename T, int L>
__global__ __launch_bounds__(kThreads) void xcd_plane_kernel(const XcdArgs<T> g) {
    static_assert(plane_threads<L>() == kThreads, "plane workgroup");
    __shared__ PlaneLds<T, L> S;
    __shared__ TwE<T> twx[kXcdMaxLen];
    __shared__ cplx<T> xt[2048];
    __shared__ unsigned sidx, sgroup;
    unsigned* q = g.q;
    xcd_join<T>(g, sidx, sgroup);
    const unsigned idx = __builtin_amdgcn_readfirstlane(sidx), group = __builtin_amdgcn_readfirstlane(sgroup);
    if (idx == ~0u) return;
    PassArgs<T> a = g.a;
    a.tw = g.twz;
    a.twlo = g.twloz;
    plane_tables<T, L>(a, S);
    xcd_table<T>(twx, g.twx, g.twlox, a.ph.nx);
    __syncthreads();
    cplx<T>*A = a.psiA, *B = g.B;
    const unsigned planes = (unsigned)a.ph.nx;
    unsigned bar = 0;
    a.dst = B;
    for (unsigned p = idx; p < planes; p += group) {
        plane_tile<T, L, PL_OPEN, false, true>(a, S, p, xcd_tid());
        __syncthreads();
    }
    for (int s = 0; s < g.nt; s++) {
        xcd_barrier(q, group, bar);
        xcd_turn<T, 0>(g, B, xt, twx, idx, group);
        xcd_barrier(q, group, bar);
        a.src = B;
        a.dst = A;
        for (unsigned p = idx; p < planes; p += group) {
            plane_tile<T, L, PL_VSTEP2, false, true>(a, S, p, xcd_tid());
            __syncthreads();
        }
        xcd_barrier(q, group, bar);
        xcd_turn<T, 0>(g, A, xt, twx, idx, group);
        xcd_barrier(q, group, bar);
        a.src = A;
        a.dst = B;
        for (unsigned p = idx; p < planes; p += group) {
            if (s < g.nt - 1) plane_tile<T, L, PL_VSTEP3_NEXT, false, true>(a, S, p, xcd_tid());
            else plane_tile<T, L, PL_VSTEP3_LAST, false, true>(a, S, p, xcd_tid());
            __syncthreads();
        }
    }
}

// false: no kernel for the lattice
template <typename T, int NZ>
bool launch_xcd_len(const XcdArgs<T>& g, bool ite, unsigned blocks, hipStream_t s) {
    if constexpr (!xcd_length(NZ)) {
        return false;
    } else {
        if (ite) hipLaunchKernelGGL((xcd_steps_kernel<T, NZ, true>), dim3(blocks), dim3(kThreads), 0, s, g);
        else hipLaunchKernelGGL((xcd_steps_kernel<T, NZ, false>), dim3(blocks), dim3(kThreads), 0, s, g);
        return true;
    }
}

}  // namespace gpe
