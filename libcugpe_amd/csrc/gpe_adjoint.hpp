// One backward step of the discrete adjoint of the real-time split step.
//
// The objective is L = 1 - |<psi_t|psi(T)>|^2 / (|psi_t|^2 |psi(0)|^2) and the
// gradient is taken with respect to V_ext at every lattice point.  With
// dL = 2 Re sum conj(lambda) dpsi, one step backwards from the step's input
// psi0 and its output psi1 (stored by the recomputed forward steps) is, with
// V0 = Vext + g(rho(psi0)), E0 = exp(c V0), phi3 = phi E0,
// V1 = (V0 + Vext + g(rho(phi3)))/2 and W = exp(c V1),
//
//   P1  phi = K psi0 E0                     (kinetic factors)
//   P2  vb = 2 Re(conj(lam) psi1 c), lam <- conj(W) lam
//       lam <- K^+ lam                      (conj kinetic factors)
//   P3  chi = psi0 W, lam0 = conj(W) lam, Vb1 = vb + 2 Re(conj(lam) chi c)
//       grad += Vb1/2, lp3 = (Vb1/2) g'(rho3) gamma phi3,
//       vb <- Vb1/2 + 2 Re(conj(lp3) phi3 c), lam <- conj(E0) lp3
//       lam <- K^+ lam
//   P4  lam <- lam0 + conj(E0) lam + gamma g'(rho0) Vb0 psi0,
//       Vb0 = vb + 2 Re(conj(lam) psi0 E0 c), grad += Vb0
//
// Every pointwise quantity is formed in FP64 from the stored states (complex64
// or complex128), so the factors exp(c V) are exact rotations and the gradient
// accumulates in FP64; phi is the predictor before its last factor, so that
// phi3 too is formed in FP64 by each part that needs it.  (The forward kernels'
// own predictor ends, kept while the steps are recomputed, would save P1's four
// passes, but in complex64 they are FP32 phases and products.)  V_ext is read
// from a precomputed FP64 array holding the forward kernels' own values.
//
// The parts run on the registers of the z passes around them
// (adj_zwave_kernel): P1 and P2 before a forward z, P3 between an inverse and a
// forward z, P4 after an inverse z and, within a segment, followed by the
// previous step's P2 and its forward z.  P1 needs the states alone, so its
// passes run once over all steps of a segment.  A backward step is then two z
// passes and four turn-arounds; every pointwise part and every z transform as a
// pass of its own were four kernels and fifteen passes (64^3 complex64, a
// gradient of 32 steps: 6.1 -> 4.45 ms, about 0.7 of it by pow23; with the
// forward kernels' predictor ends 4.17).
// z lengths without a wave split run the parts as pointwise kernels between
// plain passes.
#pragma once

#include "gpe_zwave.hpp"

namespace gpe {

struct AdjPhys {
    int interactions;
    double gamma;
    double a;       // scattering length
    double cx, cy;  // step coefficient c
};

// The arrays of one backward step (complex arrays in the working precision).
// psi1 is read by P2 on its own; after P4 the previous step's psi1 is psi0.
template <typename T>
struct AdjArgs {
    AdjPhys p;
    size_t n;
    const double* vx;                          // V_ext per point
    const cplx<T>*psi0, *psi1, *phi;           // the step's input, output and predictor
    const cplx<T>*psi0p, *phip;                // the previous step's, for its P2
    cplx<T>* out;                              // P1: the predictors, of as many states as there are at psi0
    cplx<T>*lam, *lam0;                        // adjoint state; the part of it that P3 leaves to P4
    double *vb, *grad;                         // potential sensitivity, dL/dV_ext
    const cplx<T>*tw, *twlo;                   // z twiddles (z passes)
    unsigned M, M1;                            // z pencils of the pass, and of one lattice
};

// z passes of a backward step
enum AdjPass { ADJ_P1 = 0, ADJ_P2 = 1, ADJ_P3 = 2, ADJ_P4 = 3, ADJ_P4P2 = 4 };

__device__ __forceinline__ double adj_g(const AdjPhys& p, double rho) {
    const double PI = 3.14159265358979323846;
    switch (p.interactions) {
    case INT_UFG: return 0.37 * pow23(3.0 * PI * PI * rho) / 2.0;
    case INT_CONTACT: return 4 * PI * p.a * rho;
    default: return 0.0;
    }
}
// derivative of dEDF/drho in rho, from g(rho) (UFG: (2/3) g / rho, 0 at rho = 0)
__device__ __forceinline__ double adj_dg(const AdjPhys& p, double rho, double g) {
    const double PI = 3.14159265358979323846;
    switch (p.interactions) {
    case INT_UFG: return rho > 0.0 ? (2.0 / 3.0) * g / rho : 0.0;
    case INT_CONTACT: return 4 * PI * p.a;
    default: return 0.0;
    }
}

template <typename T>
__device__ __forceinline__ cplx<double> to64(cplx<T> v) { return mk((double)v.x, (double)v.y); }
template <typename T>
__device__ __forceinline__ cplx<T> from64(cplx<double> v) { return mk((T)v.x, (T)v.y); }
__device__ __forceinline__ cplx<double> conj_(cplx<double> a) { return mk(a.x, -a.y); }
// exp(c V) (c is imaginary in real time)
__device__ __forceinline__ cplx<double> ecv(const AdjPhys& p, double V) {
    const double x = p.cy * V;
    double s, c;
    if (fabs(x) <= 0.25) sincos_taylor(x, &s, &c);
    else sincos(x, &s, &c);
    if (p.cx != 0.0) {
        const double t = exp(p.cx * V);
        return mk(t * c, t * s);
    }
    return mk(c, s);
}
// 2 Re(conj(l) y c)
__device__ __forceinline__ double sens(const AdjPhys& p, cplx<double> l, cplx<double> y) {
    const cplx<double> t = cmulc(y, l);  // y conj(l)
    return 2.0 * (t.x * p.cx - t.y * p.cy);
}
__device__ __forceinline__ double rho_of(const AdjPhys& p, cplx<double> v) { return p.gamma * (v.x * v.x + v.y * v.y); }

__device__ __forceinline__ cplx<double> adj_part1(const AdjPhys& p, double vx, cplx<double> psi0) {
    return cmul(psi0, ecv(p, vx + adj_g(p, rho_of(p, psi0))));
}

__device__ __forceinline__ cplx<double> adj_part2(const AdjPhys& p, double vx, cplx<double> psi0, cplx<double> psi1,
                                                  cplx<double> phi, cplx<double> l, double& vb) {
    const double V0 = vx + adj_g(p, rho_of(p, psi0));
    const cplx<double> phi3 = cmul(phi, ecv(p, V0));
    const double V1 = 0.5 * (V0 + vx + adj_g(p, rho_of(p, phi3)));
    vb = sens(p, l, psi1);
    return cmul(conj_(ecv(p, V1)), l);
}

__device__ __forceinline__ cplx<double> adj_part3(const AdjPhys& p, double vx, cplx<double> psi0, cplx<double> phi,
                                                  cplx<double> l, double& vb, cplx<double>& lam0, double& dgrad) {
    const double V0 = vx + adj_g(p, rho_of(p, psi0));
    const cplx<double> E0 = ecv(p, V0), phi3 = cmul(phi, E0);
    const double r3 = rho_of(p, phi3), g3 = adj_g(p, r3);
    const cplx<double> W = ecv(p, 0.5 * (V0 + vx + g3));
    lam0 = cmul(conj_(W), l);
    const double V1b = vb + sens(p, l, cmul(psi0, W));
    dgrad = 0.5 * V1b;
    const double f = 0.5 * V1b * adj_dg(p, r3, g3) * p.gamma;
    const cplx<double> lp3 = mk(f * phi3.x, f * phi3.y);
    vb = 0.5 * V1b + sens(p, lp3, phi3);
    return cmul(conj_(E0), lp3);
}

__device__ __forceinline__ cplx<double> adj_part4(const AdjPhys& p, double vx, cplx<double> psi0, cplx<double> lam0,
                                                  cplx<double> l, double vb, double& dgrad) {
    const double r0 = rho_of(p, psi0), g0 = adj_g(p, r0);
    const cplx<double> E0 = ecv(p, vx + g0);
    const double V0b = vb + sens(p, l, cmul(psi0, E0));
    dgrad = V0b;
    const double f = p.gamma * adj_dg(p, r0, g0) * V0b;
    const cplx<double> r = cadd(lam0, cmul(conj_(E0), l));
    return mk(r.x + f * psi0.x, r.y + f * psi0.y);
}

// One z pass of a backward step, on the adjoint state in place (P1: from the
// states to the predictors): the layout and transforms of zwave_kernel.  What bounds it: the 7-9 side arrays of a
// part (P3 reads and writes about 11 doubles per point), so the parts run
// chunk by chunk with the chunk's loads in flight together and no state but
// the pencil's own registers kept between chunks.
template <typename T, int N, int PASS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void adj_zwave_kernel(const AdjArgs<T> a) {
    using Z = ZW<T, N>;
    constexpr int A = Z::A, B = Z::B;
    __shared__ ZwLds<T, N> L;
    for (int i = threadIdx.x; i < N; i += kThreads) {
        const int m = (i / A) * (i % A);
        if constexpr (sizeof(T) == 4) {
            const cplx<float> h = a.tw[m], lo = a.twlo[m];
            L.tw[i].t = make_float4(h.x, h.y, lo.x, lo.y);
        } else {
            L.tw[i].t = a.tw[m];
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int g = lane / A, l = lane % A;
    cplx<T>* X = L.x + wv * Z::WAVE + g * Z::GS;
    const unsigned p = (blockIdx.x * Z::WAVES + (unsigned)wv) * Z::PW + (unsigned)g;
    const bool ok = p < a.M;
    const size_t base = (size_t)(ok ? p : 0u) * N + (size_t)l;
    const AdjPhys ph = a.p;
    cplx<T> v[B];
#pragma unroll
    for (int b = 0; b < B; b++) v[b] = (PASS == ADJ_P1 ? a.psi0 : a.lam)[base + (size_t)(A * b)];
    // V_ext is one lattice's
    const size_t vbase = PASS == ADJ_P1 ? (size_t)(ok ? p % a.M1 : 0u) * N + (size_t)l : base;
    if constexpr (PASS != ADJ_P1 && PASS != ADJ_P2) zw_fft<T, N, +1, B>(v, X, L.tw, l);
    constexpr int CH = zw_chunk(B, sizeof(T) == 4 ? 4 : 2);
    static_for<0, B / CH>([&](auto qc) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
        double vx[CH], vb[CH], gr[CH];
        cplx<T> p0[CH], p3[CH], x[CH], p0p[CH];
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const size_t o = base + (size_t)(A * (q * CH + j));
            vx[j] = a.vx[vbase + (size_t)(A * (q * CH + j))];
            if constexpr (PASS != ADJ_P1) p0[j] = a.psi0[o];
            if constexpr (PASS == ADJ_P2) x[j] = a.psi1[o];
            if constexpr (PASS == ADJ_P4 || PASS == ADJ_P4P2) x[j] = a.lam0[o];
            if constexpr (PASS == ADJ_P2 || PASS == ADJ_P3) p3[j] = a.phi[o];
            if constexpr (PASS == ADJ_P4P2) {
                p3[j] = a.phip[o];
                p0p[j] = a.psi0p[o];
            }
            if constexpr (PASS != ADJ_P1 && PASS != ADJ_P2) {
                vb[j] = a.vb[o];
                gr[j] = a.grad[o];
            }
        }
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const size_t o = base + (size_t)(A * (q * CH + j));
            cplx<double> u = to64(v[q * CH + j]);
            double dg = 0.0;
            if constexpr (PASS == ADJ_P1) u = adj_part1(ph, vx[j], u);
            if constexpr (PASS == ADJ_P3) {
                cplx<double> l0;
                u = adj_part3(ph, vx[j], to64(p0[j]), to64(p3[j]), u, vb[j], l0, dg);
                if (ok) a.lam0[o] = from64<T>(l0);
            }
            if constexpr (PASS == ADJ_P4 || PASS == ADJ_P4P2)
                u = adj_part4(ph, vx[j], to64(p0[j]), to64(x[j]), u, vb[j], dg);
            // the adjoint state of a step boundary is kept in the working precision
            if constexpr (PASS == ADJ_P4P2) {
                u = to64(from64<T>(u));
                u = adj_part2(ph, vx[j], to64(p0p[j]), to64(p0[j]), to64(p3[j]), u, vb[j]);
            }
            if constexpr (PASS == ADJ_P2) u = adj_part2(ph, vx[j], to64(p0[j]), to64(x[j]), to64(p3[j]), u, vb[j]);
            if (ok && PASS != ADJ_P1) {
                if constexpr (PASS != ADJ_P2) a.grad[o] = gr[j] + dg;
                if constexpr (PASS != ADJ_P4) a.vb[o] = vb[j];
            }
            // P4 ends here: stored at once, or the compiler interleaves the
            // chunks and spills (412 bytes per lane at 128 points in complex128)
            if constexpr (PASS == ADJ_P4) {
                if (ok) a.lam[o] = from64<T>(u);
            } else {
                v[q * CH + j] = from64<T>(u);
            }
        }
    });
    if constexpr (PASS == ADJ_P4) return;
    if constexpr (PASS != ADJ_P4) zw_fft<T, N, -1, B>(v, X, L.tw, l);
    if (ok) {
#pragma unroll
        for (int b = 0; b < B; b++) (PASS == ADJ_P1 ? a.out : a.lam)[base + (size_t)(A * b)] = v[b];
    }
}

// false: the z length has no wave split, or one of more than 16 points per lane:
// the parts then leave too few registers and spill, and the pointwise kernels
// are faster (us a step of a complex64 gradient in waves / pointwise: 8x12x96
// 195 / 156, 32x64x192 280 / 229, 64x64x512 1089 / 970).  None of these
// kernels needs scratch memory, which the runtime would allocate at a first
// launch on a queue, aborting where none is left.
template <typename T, int N>
bool launch_adj_zwave(const AdjArgs<T>& a, int pass, hipStream_t s) {
    if constexpr (zw_lanes<T>(N) == 0 || N > 16 * zw_lanes<T>(N)) {
        return false;
    } else {
        const dim3 g((a.M + ZW<T, N>::PENCILS - 1) / ZW<T, N>::PENCILS), b(kThreads);
        switch (pass) {
        case ADJ_P1: hipLaunchKernelGGL((adj_zwave_kernel<T, N, ADJ_P1>), g, b, 0, s, a); break;
        case ADJ_P2: hipLaunchKernelGGL((adj_zwave_kernel<T, N, ADJ_P2>), g, b, 0, s, a); break;
        case ADJ_P3: hipLaunchKernelGGL((adj_zwave_kernel<T, N, ADJ_P3>), g, b, 0, s, a); break;
        case ADJ_P4: hipLaunchKernelGGL((adj_zwave_kernel<T, N, ADJ_P4>), g, b, 0, s, a); break;
        default: hipLaunchKernelGGL((adj_zwave_kernel<T, N, ADJ_P4P2>), g, b, 0, s, a); break;
        }
        return true;
    }
}

}  // namespace gpe
