// Kernel bodies and launchers, instantiated once per precision by
// gpe_kernels_f32.hip / gpe_kernels_f64.hip.
#pragma once

#include "gpe_kernels.hpp"

namespace gpe {

template <typename T>
unsigned launch_fft_pass_impl(int N, const PassArgs<T>& a, hipStream_t s) {
#define GPE_CASE(NN) \
    case NN: return launch_fft_pass_n<T, NN>(a, s);
    switch (N) {
        GPE_FFT_LENGTHS(GPE_CASE)
    default:
        return 0;
    }
#undef GPE_CASE
}

template <typename T>
bool launch_xcd_impl(int N, const XcdArgs<T>& g, bool ite, unsigned blocks, hipStream_t s) {
#define GPE_CASE(NN) \
    case NN: return launch_xcd_n<T, NN>(g, ite, blocks, s);
    switch (N) {
        GPE_FFT_LENGTHS(GPE_CASE)
    default:
        return false;
    }
#undef GPE_CASE
}

template <typename T>
bool launch_adjoint_z_impl(int N, const AdjArgs<T>& a, int pass, hipStream_t s) {
#define GPE_CASE(NN) \
    case NN: return launch_adjoint_z_n<T, NN>(a, pass, s);
    switch (N) {
        GPE_FFT_LENGTHS(GPE_CASE)
    default:
        return false;
    }
#undef GPE_CASE
}

template <typename T, int NN>
constexpr int min_tile() {
    constexpr int w = full_tile_w<T, NN, true>();
    if constexpr (zw_lanes<T>(NN) != 0) return ZW<T, NN>::PENCILS < w ? ZW<T, NN>::PENCILS : w;
    return w;
}

template <typename T>
int fft_tile_width_impl(int N) {
#define GPE_CASE(NN) \
    case NN: return min_tile<T, NN>();  /* the narrowest tile of any pass */
    switch (N) {
        GPE_FFT_LENGTHS(GPE_CASE)
    default:
        return 0;
    }
#undef GPE_CASE
}

template <typename T>
int fft_lean_width_impl(int N) {
#define GPE_CASE(NN) \
    case NN: return lean_w<T, NN, 1>();
    switch (N) {
        GPE_FFT_LENGTHS(GPE_CASE)
    default:
        return 0;
    }
#undef GPE_CASE
}

// ---------------------------------------------------------- reductions

template <typename T>
__global__ __launch_bounds__(kThreads) void norm_partials_kernel(const cplx<T>* __restrict__ A, unsigned n,
                                                                 double gamma, double* __restrict__ partials) {
    __shared__ double red[kThreads / 64];
    double acc = 0.0;
    const unsigned stride = gridDim.x * kThreads;
    for (unsigned i = blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
        const cplx<T> v = A[i];
        acc += gamma * ((double)v.x * (double)v.x + (double)v.y * (double)v.y);
    }
    const double s = block_sum(acc, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void scale_kernel(cplx<T>* __restrict__ A, unsigned n,
                                                         const double* __restrict__ scal) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) A[i] = cscale(A[i], (T)scal[1]);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void density_kernel(const cplx<T>* __restrict__ A, unsigned n, double gamma,
                                                           double* __restrict__ out) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) {
        const cplx<T> v = A[i];
        out[i] = gamma * ((double)v.x * (double)v.x + (double)v.y * (double)v.y);
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void mean_density_kernel(const cplx<T>* __restrict__ A, unsigned n,
                                                                unsigned batch, double gamma,
                                                                double* __restrict__ out) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) {
        double acc = 0.0;
        for (unsigned b = 0; b < batch; b++) {
            const cplx<T> v = A[(size_t)b * n + i];
            acc += (double)v.x * (double)v.x + (double)v.y * (double)v.y;
        }
        out[i] = gamma * acc / (double)batch;
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void phase_kernel(const cplx<T>* __restrict__ A, unsigned n,
                                                         double* __restrict__ out) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) {
        const cplx<T> v = A[i];
        out[i] = atan2((double)v.y, (double)v.x);
    }
}

// dev/gpe_engine.cu:584-591: psi = |psi| exp(i phase)
template <typename T>
__global__ __launch_bounds__(kThreads) void enforce_phase_kernel(cplx<T>* __restrict__ A, unsigned n,
                                                                 const double* __restrict__ phase) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) {
        const cplx<T> v = A[i];
        const T a = g_sqrt(v.x * v.x + v.y * v.y);
        T s, c;
        g_sincos((T)phase[i], &s, &c);
        A[i] = mk(a * c, a * s);
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void from_c128_kernel(const cplx<double>* __restrict__ in,
                                                             cplx<T>* __restrict__ out, unsigned n) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) out[i] = mk((T)in[i].x, (T)in[i].y);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void to_c128_kernel(const cplx<T>* __restrict__ in,
                                                           cplx<double>* __restrict__ out, unsigned n) {
    const unsigned i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) out[i] = mk((double)in[i].x, (double)in[i].y);
}

// -------------------------------------------------- plaquette windings
//
// Winding of the phase of psi around each elementary plaquette, counted in
// quarter turns: the quadrant of every corner is compared with the next
// corner's; opposite quadrants are resolved by the sign of the cross product.
// All arithmetic is on FP64 values with separately rounded products (no fused
// multiply-add), so the result is bit-identical to the CPU oracle's on the same
// input, in either precision.

__device__ __forceinline__ int quadrant(double x, double y) {
    if (y >= 0.0 && x > 0.0) return 0;
    if (x <= 0.0 && y > 0.0) return 1;
    if (y <= 0.0 && x < 0.0) return 2;
    return 3;
}

// a corner of a plaquette: its value, quadrant, and whether it is dense enough to count
struct Corner {
    double x, y;
    int q;
    bool ok;
};
template <typename T>
__device__ __forceinline__ Corner corner(cplx<T> v, double rho_min) {
    Corner c;
    c.x = (double)v.x;
    c.y = (double)v.y;
    c.q = quadrant(c.x, c.y);
    c.ok = __dadd_rn(__dmul_rn(c.x, c.x), __dmul_rn(c.y, c.y)) >= rho_min;
    return c;
}

__device__ __forceinline__ int quarter_turns(const Corner& a, const Corner& b) {
    const int d = (b.q - a.q) & 3;
    if (d == 1) return 1;
    if (d == 3) return -1;
    if (d == 0) return 0;
    const double cr = __dsub_rn(__dmul_rn(a.x, b.y), __dmul_rn(a.y, b.x));
    return (cr < 0.0) ? -2 : 2;
}
__device__ __forceinline__ int plaquette(const Corner& a, const Corner& b, const Corner& c, const Corner& d) {
    if (!(a.ok && b.ok && c.ok && d.ok)) return 0;
    return (quarter_turns(a, b) + quarter_turns(b, c) + quarter_turns(c, d) + quarter_turns(d, a)) / 4;
}

// A thread walks RUN points along x, so every corner is loaded, classified
// and located once and serves the planes on both sides of it.  w may be null:
// the count alone.  A run is a serial chain of loads, so it pays once its threads
// fill the chip (256 CUs of 1024): us of a count at a run of 1 / of 8, complex128:
// 32^3 26.1 / 36.9, 64^3 27.8 / 37.0, 128x128x64 (131072 threads of 8) 36.2 /
// 38.2, 128^3 (262144) 52.6 / 45.8, 256^3 257 / 199 (26.4, 29.0, 39.9, 56.0 and 284
// with 12 loads, 12 classifications and two integer divisions per point).
constexpr unsigned kWindRun = 8, kWindThreads = 196608;
template <typename T, unsigned RUN>
__global__ __launch_bounds__(kThreads) void windings_kernel(const cplx<T>* __restrict__ A, int nx, int ny, int nz,
                                                            double rho_min, int8_t* __restrict__ w,
                                                            double* __restrict__ partials) {
    __shared__ double red[kThreads / 64];
    const unsigned ux = (unsigned)nx, uy = (unsigned)ny, uz = (unsigned)nz, plane = uy * uz;
    const unsigned n = ux * plane;
    const unsigned runs = (ux + RUN - 1) / RUN;
    double cnt = 0.0;
    const unsigned stride = gridDim.x * kThreads;
    // plane runs <= n / 8 + plane < 2^31, so the index does not wrap within one stride past it
    for (unsigned i = blockIdx.x * kThreads + threadIdx.x; i < plane * runs; i += stride) {
        const unsigned run = i / plane, r = i - run * plane;
        const unsigned iy = r / uz, iz = r - iy * uz;
        const unsigned jy = (iy + 1 == uy) ? 0 : iy + 1, jz = (iz + 1 == uz) ? 0 : iz + 1;
        const unsigned o10 = jy * uz + iz, o01 = iy * uz + jz, o11 = jy * uz + jz;
        const unsigned x0 = run * RUN, x1 = x0 + RUN < ux ? x0 + RUN : ux;
        const cplx<T>* p = A + (size_t)x0 * plane;
        Corner a00 = corner(p[r], rho_min), a10 = corner(p[o10], rho_min), a01 = corner(p[o01], rho_min),
               a11 = corner(p[o11], rho_min);
        for (unsigned ix = x0; ix < x1; ix++) {
            p = A + (size_t)(ix + 1 == ux ? 0 : ix + 1) * plane;
            const Corner b00 = corner(p[r], rho_min), b10 = corner(p[o10], rho_min), b01 = corner(p[o01], rho_min),
                         b11 = corner(p[o11], rho_min);
            const int w0 = plaquette(a00, b00, b10, a10), w1 = plaquette(a00, a10, a11, a01),
                      w2 = plaquette(a00, a01, b01, b00);
            if (w) {
                const size_t at = (size_t)ix * plane + r;
                w[at] = (int8_t)w0;
                w[(size_t)n + at] = (int8_t)w1;
                w[2 * (size_t)n + at] = (int8_t)w2;
            }
            cnt += (double)((w0 != 0) + (w1 != 0) + (w2 != 0));
            a00 = b00;
            a10 = b10;
            a01 = b01;
            a11 = b11;
        }
    }
    const double s = block_sum(cnt, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

static inline int reduce_grid(unsigned n) {
    unsigned b = (n + kThreads - 1) / kThreads;
    if (b > (unsigned)kMaxReduceBlocks) b = kMaxReduceBlocks;
    if (b < 1) b = 1;
    return (int)b;
}

// Cloud parameters (dev/gpe_cloud_params.h:60-119) on the device: the
// largest gamma |psi|^2 of each workgroup into partials[blockIdx], and from
// workgroup 0 the densities along the three lines through the lattice centre
// (nx/2, ny/2, nz/2) into lines[nx | ny | nz].
template <typename T>
__global__ __launch_bounds__(kThreads) void cloud_kernel(const cplx<T>* __restrict__ A, unsigned n, int nx, int ny,
                                                         int nz, double gamma, double* __restrict__ partials,
                                                         double* __restrict__ lines) {
    __shared__ double red[kThreads / 64];
    double m = 0.0;
    const unsigned stride = gridDim.x * kThreads;
    for (unsigned i = blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
        const cplx<T> v = A[i];
        m = fmax(m, gamma * ((double)v.x * (double)v.x + (double)v.y * (double)v.y));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; w++) m = fmax(m, red[w]);
        partials[blockIdx.x] = m;
    }
    if (blockIdx.x == 0) {
        const unsigned cx = (unsigned)(nx / 2), cy = (unsigned)(ny / 2), cz = (unsigned)(nz / 2);
        const unsigned nl = (unsigned)(nx + ny + nz);
        for (unsigned i = threadIdx.x; i < nl; i += kThreads) {
            unsigned ix = cx, iy = cy, iz = cz;
            if (i < (unsigned)nx) ix = i;
            else if (i < (unsigned)(nx + ny)) iy = i - (unsigned)nx;
            else iz = i - (unsigned)(nx + ny);
            const cplx<T> v = A[((size_t)ix * (unsigned)ny + iy) * (unsigned)nz + iz];
            lines[i] = gamma * ((double)v.x * (double)v.x + (double)v.y * (double)v.y);
        }
    }
}

template <typename T>
int launch_norm_partials_impl(const cplx<T>* A, unsigned n, double gamma, double* partials, hipStream_t s) {
    const int nb = reduce_grid(n);
    hipLaunchKernelGGL((norm_partials_kernel<T>), dim3(nb), dim3(kThreads), 0, s, A, n, gamma, partials);
    return nb;
}

template <typename T>
int launch_windings_impl(const cplx<T>* A, int nx, int ny, int nz, double rho_min, int8_t* w, double* partials,
                         hipStream_t s) {
    const unsigned plane = (unsigned)ny * nz, runs = ((unsigned)nx + kWindRun - 1) / kWindRun;
    if (plane * runs >= kWindThreads) {
        const int nb = reduce_grid(plane * runs);
        hipLaunchKernelGGL((windings_kernel<T, kWindRun>), dim3(nb), dim3(kThreads), 0, s, A, nx, ny, nz, rho_min, w, partials);
        return nb;
    }
    const int nb = reduce_grid(plane * (unsigned)nx);
    hipLaunchKernelGGL((windings_kernel<T, 1>), dim3(nb), dim3(kThreads), 0, s, A, nx, ny, nz, rho_min, w, partials);
    return nb;
}

static inline dim3 ew_grid(unsigned n) { return dim3((n + kThreads - 1) / kThreads); }

#define GPE_INSTANTIATE(T)                                                                                        \
    template <>                                                                                                   \
    unsigned launch_fft_pass<T>(int N, const PassArgs<T>& a, hipStream_t s) {                                     \
        return launch_fft_pass_impl<T>(N, a, s);                                                                  \
    }                                                                                                             \
    template <>                                                                                                   \
    bool launch_xcd<T>(int N, const XcdArgs<T>& g, bool ite, unsigned blocks, hipStream_t s) {                    \
        return launch_xcd_impl<T>(N, g, ite, blocks, s);                                                          \
    }                                                                                                             \
    template <>                                                                                                   \
    bool launch_adjoint_z<T>(int N, const AdjArgs<T>& a, int pass, hipStream_t s) {                               \
        return launch_adjoint_z_impl<T>(N, a, pass, s);                                                           \
    }                                                                                                             \
    template <>                                                                                                   \
    int fft_tile_width<T>(int N) {                                                                                \
        return fft_tile_width_impl<T>(N);                                                                         \
    }                                                                                                             \
    template <>                                                                                                   \
    int fft_lean_width<T>(int N) {                                                                                \
        return fft_lean_width_impl<T>(N);                                                                         \
    }                                                                                                             \
    template <>                                                                                                   \
    int launch_norm_partials<T>(const cplx<T>* A, unsigned n, double gamma, double* partials, hipStream_t s) {    \
        return launch_norm_partials_impl<T>(A, n, gamma, partials, s);                                            \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_scale<T>(cplx<T> * A, unsigned n, const double* scal, hipStream_t s) {                            \
        hipLaunchKernelGGL((scale_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, A, n, scal);                      \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_density<T>(const cplx<T>* A, unsigned n, double gamma, double* out, hipStream_t s) {              \
        hipLaunchKernelGGL((density_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, A, n, gamma, out);              \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_mean_density<T>(const cplx<T>* A, unsigned n, unsigned batch, double gamma, double* out,          \
                                hipStream_t s) {                                                                  \
        hipLaunchKernelGGL((mean_density_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, A, n, batch, gamma, out);  \
    }                                                                                                             \
    template <>                                                                                                   \
    int launch_windings<T>(const cplx<T>* A, int nx, int ny, int nz, double rho_min, int8_t* w, double* partials, \
                           hipStream_t s) {                                                                       \
        return launch_windings_impl<T>(A, nx, ny, nz, rho_min, w, partials, s);                                   \
    }                                                                                                             \
    template <>                                                                                                   \
    int launch_cloud<T>(const cplx<T>* A, int nx, int ny, int nz, double gamma, double* partials, double* lines,  \
                        hipStream_t s) {                                                                          \
        const unsigned n = (unsigned)nx * (unsigned)ny * (unsigned)nz;                                            \
        unsigned nb = (n + kThreads - 1) / kThreads;                                                              \
        if (nb > (unsigned)kMaxReduceBlocks) nb = kMaxReduceBlocks;                                               \
        hipLaunchKernelGGL((cloud_kernel<T>), dim3(nb), dim3(kThreads), 0, s, A, n, nx, ny, nz, gamma, partials,  \
                           lines);                                                                                \
        return (int)nb;                                                                                           \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_phase<T>(const cplx<T>* A, unsigned n, double* out, hipStream_t s) {                              \
        hipLaunchKernelGGL((phase_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, A, n, out);                       \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_enforce_phase<T>(cplx<T> * A, unsigned n, const double* phase, hipStream_t s) {                   \
        hipLaunchKernelGGL((enforce_phase_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, A, n, phase);             \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_from_c128<T>(const cplx<double>* in, cplx<T>* out, unsigned n, hipStream_t s) {                   \
        hipLaunchKernelGGL((from_c128_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, in, out, n);                  \
    }                                                                                                             \
    template <>                                                                                                   \
    void launch_to_c128<T>(const cplx<T>* in, cplx<double>* out, unsigned n, hipStream_t s) {                     \
        hipLaunchKernelGGL((to_c128_kernel<T>), ew_grid(n), dim3(kThreads), 0, s, in, out, n);                    \
    }

}  // namespace gpe
