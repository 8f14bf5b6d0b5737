// Pointwise kernels of the discrete adjoint (gpe_adjoint.hpp): the parts of a
// backward step for z lengths without a wave split, V_ext as the forward
// kernels see it, the overlap sums and the first adjoint state.
#include "gpe_kernels.hpp"

namespace gpe {

namespace {

// part PASS (ADJ_P2, ADJ_P3, ADJ_P4) on the adjoint state, ADJ_P1 on the states
template <typename T, int PASS>
__global__ __launch_bounds__(kThreads) void adj_point_kernel(const AdjArgs<T> a, size_t n) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const cplx<double> p0 = to64(a.psi0[i]);
    if constexpr (PASS == ADJ_P1) {
        a.out[i] = from64<T>(adj_part1(a.p, a.vx[i % a.n], p0));
        return;
    }
    const cplx<double> l = to64(a.lam[i]);
    double dg = 0.0;
    if constexpr (PASS == ADJ_P2) {
        double vb;
        a.lam[i] = from64<T>(adj_part2(a.p, a.vx[i], p0, to64(a.psi1[i]), to64(a.phi[i]), l, vb));
        a.vb[i] = vb;
    } else if constexpr (PASS == ADJ_P3) {
        double vb = a.vb[i];
        cplx<double> l0;
        a.lam[i] = from64<T>(adj_part3(a.p, a.vx[i], p0, to64(a.phi[i]), l, vb, l0, dg));
        a.lam0[i] = from64<T>(l0);
        a.vb[i] = vb;
        a.grad[i] += dg;
    } else {
        a.lam[i] = from64<T>(adj_part4(a.p, a.vx[i], p0, to64(a.lam0[i]), l, a.vb[i], dg));
        a.grad[i] += dg;
    }
}

// V_ext at every point exactly as the forward kernels evaluate it
template <typename T>
__global__ __launch_bounds__(kThreads) void adj_vfill(Phys<T> ph, double* __restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const unsigned nyz = (unsigned)(ph.ny * ph.nz);
    const unsigned ix = (unsigned)(i / nyz), r = (unsigned)(i % nyz);
    const unsigned iy = r / (unsigned)ph.nz, iz = r % (unsigned)ph.nz;
    out[i] = (double)vext(ph, ix, iy, iz, (unsigned)i, ph.it);
}

// per workgroup: Re and Im of sum conj(t) psi, sum |a|^2, sum |t|^2
template <typename T>
__global__ __launch_bounds__(kThreads) void adj_overlap(const cplx<T>* __restrict__ psi, const cplx<T>* __restrict__ tgt,
                                                        const cplx<T>* __restrict__ a0, size_t n,
                                                        double* __restrict__ partials) {
    __shared__ double red[kThreads / 64];
    double s[4] = {0, 0, 0, 0};
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads) {
        const cplx<double> p = to64(psi[i]), t = to64(tgt[i]), q = to64(a0[i]);
        s[0] += t.x * p.x + t.y * p.y;
        s[1] += t.x * p.y - t.y * p.x;
        s[2] += q.x * q.x + q.y * q.y;
        s[3] += t.x * t.x + t.y * t.y;
    }
    for (int k = 0; k < 4; k++) {
        const double b = block_sum(s[k], red);
        if (threadIdx.x == 0) partials[(size_t)k * gridDim.x + blockIdx.x] = b;
    }
}

// lam = (fr + i fi) tgt
template <typename T>
__global__ __launch_bounds__(kThreads) void adj_lam_init(cplx<T>* __restrict__ lam, const cplx<T>* __restrict__ tgt,
                                                         double fr, double fi, size_t n) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    lam[i] = from64<T>(cmul(to64(tgt[i]), mk(fr, fi)));
}

inline dim3 grid_of(size_t n) { return dim3((unsigned)((n + kThreads - 1) / kThreads)); }

}  // namespace

template <typename T>
void launch_adjoint_point(const AdjArgs<T>& a, int part, size_t n, hipStream_t s) {
    const dim3 g = grid_of(n), b(kThreads);
    switch (part) {
    case ADJ_P1: hipLaunchKernelGGL((adj_point_kernel<T, ADJ_P1>), g, b, 0, s, a, n); break;
    case ADJ_P2: hipLaunchKernelGGL((adj_point_kernel<T, ADJ_P2>), g, b, 0, s, a, n); break;
    case ADJ_P3: hipLaunchKernelGGL((adj_point_kernel<T, ADJ_P3>), g, b, 0, s, a, n); break;
    default: hipLaunchKernelGGL((adj_point_kernel<T, ADJ_P4>), g, b, 0, s, a, n); break;
    }
}

template <typename T>
void launch_adjoint_vfill(const Phys<T>& ph, double* out, size_t n, hipStream_t s) {
    hipLaunchKernelGGL((adj_vfill<T>), grid_of(n), dim3(kThreads), 0, s, ph, out, n);
}

template <typename T>
int launch_adjoint_overlap(const void* psi, const void* tgt, const void* a0, size_t n, double* partials,
                           hipStream_t s) {
    size_t b = (n + kThreads - 1) / kThreads;
    if (b > (size_t)kMaxReduceBlocks / 2) b = kMaxReduceBlocks / 2;  // 4 sums fit the engine's partials
    hipLaunchKernelGGL((adj_overlap<T>), dim3((unsigned)b), dim3(kThreads), 0, s, (const cplx<T>*)psi,
                       (const cplx<T>*)tgt, (const cplx<T>*)a0, n, partials);
    return (int)b;
}

template <typename T>
void launch_adjoint_lam_init(void* lam, const void* tgt, double fr, double fi, size_t n, hipStream_t s) {
    hipLaunchKernelGGL((adj_lam_init<T>), grid_of(n), dim3(kThreads), 0, s, (cplx<T>*)lam, (const cplx<T>*)tgt, fr,
                       fi, n);
}

#define GPE_ADJ_INST(T)                                                                                      \
    template void launch_adjoint_point<T>(const AdjArgs<T>&, int, size_t, hipStream_t);                       \
    template void launch_adjoint_vfill<T>(const Phys<T>&, double*, size_t, hipStream_t);                     \
    template int launch_adjoint_overlap<T>(const void*, const void*, const void*, size_t, double*, hipStream_t); \
    template void launch_adjoint_lam_init<T>(void*, const void*, double, double, size_t, hipStream_t);
GPE_ADJ_INST(float)
GPE_ADJ_INST(double)
#undef GPE_ADJ_INST

}  // namespace gpe
