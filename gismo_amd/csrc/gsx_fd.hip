// Fast diagonalization preconditioner on the device
// (gsPatchPreconditionersCreator::fastDiagonalizationOp,
// src/gsSolver/gsPatchPreconditionersCreator.hpp:258-348):
//   z = (Q_{d-1} x ... x Q_0) diag(1 / (alpha + sum_k lambda_k)) (Q_{d-1} x ... x Q_0)^T r
// over the free box of a single patch (direction 0 fastest).  Each factor is
// a mode product along one direction: y_a = sum_i M[i*m + a] x_i with
// M = Q_k (to apply Q_k^T) or M = Q_k^T (to apply Q_k).
#include "gsx_common.h"
#include "gsx_kernels.h"

namespace gsx {

// One mode product, one thread per output (boxes whose strips exceed the LDS
// of the fused kernels below): along direction 0 the lanes share the input
// line (broadcast) and read consecutive columns of M; along directions 1, 2
// they read consecutive inputs and share the row of M.
template <typename T>
__global__ __launch_bounds__(256) void k_fd_mode(int m0, int m1, int m2, int dir, const T *__restrict__ M,
                                                 const T *__restrict__ x, int64_t xo, int64_t xs1, int64_t xs2,
                                                 T *__restrict__ y, int64_t yo, int64_t ys1, int64_t ys2,
                                                 const double *__restrict__ l0, const double *__restrict__ l1,
                                                 const double *__restrict__ l2, double alpha,
                                                 const CGState *__restrict__ st)
{
    if (st && st->done) return;
    const int64_t n = (int64_t)m0 * m1 * m2;
    const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (o >= n) return;
    const int a = (int)(o % m0), b = (int)((o / m0) % m1), c = (int)(o / ((int64_t)m0 * m1));
    int m, j;
    int64_t stride, base;
    if (dir == 0) {
        m = m0; j = a; stride = 1; base = xo + b * xs1 + c * xs2;
    } else if (dir == 1) {
        m = m1; j = b; stride = xs1; base = xo + a + c * xs2;
    } else {
        m = m2; j = c; stride = xs2; base = xo + a + b * xs1;
    }
    T acc = 0;
    for (int i = 0; i < m; ++i) acc += M[(int64_t)i * m + j] * x[base + i * stride];
    if (l0) {
        const double den = alpha + l0[a] + l1[b] + (l2 ? l2[c] : 0.0);
        acc = (T)((double)acc / den);
    }
    y[yo + a + b * ys1 + c * ys2] = acc;
}

// Slab form (thin boxes, see fd_fused): the block stages the 2D slab of its fixed
// third index (c for directions 0 and 1, b for direction 2; rows x m0 values) in
// LDS and each thread computes one output of that slab from it: along direction
// 0 y[c][b][j] = sum_i M[i][j] x[c][b][i] (the lanes share the slab row and read
// consecutive columns of M), along directions 1 and 2 y[..][j][a] =
// sum_i M[i][j] x[..][i][a] (the lanes read consecutive slab entries and share
// the column of M).
template <typename T, int DIR>
__global__ __launch_bounds__(256) void k_fd_slab(int m0, int m1, int m2, const T *__restrict__ M,
                                                 const T *__restrict__ x, int64_t xo, int64_t xs1, int64_t xs2,
                                                 T *__restrict__ y, int64_t yo, int64_t ys1, int64_t ys2,
                                                 const double *__restrict__ l0, const double *__restrict__ l1,
                                                 const double *__restrict__ l2, double alpha,
                                                 const CGState *__restrict__ st)
{
    extern __shared__ double fd_smem[];
    T *sX = reinterpret_cast<T *>(fd_smem);
    if (st && st->done) return;
    const int fixed = blockIdx.y;
    const int rows = DIR == 2 ? m2 : m1;
    const int64_t base = xo + (DIR == 2 ? (int64_t)fixed * xs1 : (int64_t)fixed * xs2);
    const int64_t rstride = DIR == 2 ? xs2 : xs1;
    const int n = rows * m0;
    for (int idx = threadIdx.x; idx < n; idx += 256) {
        const int r = idx / m0, a = idx % m0;
        sX[idx] = x[base + a + r * rstride];
    }
    __syncthreads();
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= n) return;
    const int r = idx / m0, q = idx % m0;
    T acc = 0;
    if (DIR == 0) {
        const T *xr = sX + r * m0;
        for (int i = 0; i < m0; ++i) acc += M[(int64_t)i * m0 + q] * xr[i];
    } else {
        for (int i = 0; i < rows; ++i) acc += M[(int64_t)i * rows + r] * sX[i * m0 + q];
    }
    const int a = q, b = DIR == 2 ? fixed : r, c = DIR == 2 ? r : fixed;
    if (l0) acc = (T)((double)acc / (alpha + l0[a] + l1[b] + (l2 ? l2[c] : 0.0)));
    y[yo + a + (int64_t)b * ys1 + (int64_t)c * ys2] = acc;
}

// ---------------------------------------------------------------------------
// Two mode products per launch on the matrix cores.  The products are small
// GEMMs (65-deep at 64^3 p = 3) whose operands sit in the L2, so the apply is
// bound by latency and launches, not by arithmetic or bandwidth: a strip of 16
// outputs keeps the intermediate in LDS, every global operand is read along
// its contiguous direction (16 lanes, 128 bytes in FP64), and the 3D apply
// takes three launches instead of six:
//   k_fd_pair     directions 1 and 0 of a plane (forward), 16 rows j1 a block
//   k_fd_column   direction 2 forward, the division, direction 2 backward,
//                 16 columns (a, b) a block
//   k_fd_pair     directions 1 and 0 backward
// In 2D two k_fd_pair launches, the division in the first.  At 65^3 (64^3
// elements, p = 3) one FP32 apply takes 7.4 + 8.3 + 7.4 us; one thread per
// output, one product a launch, took six times 13.2 us.
// MFMA 16x16x4 operands: A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k;
// result [i][j]: FP64 lane j + 16 (i % 4), element i / 4; FP32 lane
// j + 16 (i / 4), element i % 4.
// ---------------------------------------------------------------------------
typedef double fd_d4 __attribute__((ext_vector_type(4)));
typedef float fd_f4 __attribute__((ext_vector_type(4)));

template <typename T> struct FdMfma;
template <> struct FdMfma<double> {
    using V = fd_d4;
    static __device__ inline V mul(double a, double b, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ inline int row(int q, int lk) { return 4 * q + lk; }
};
template <> struct FdMfma<float> {
    using V = fd_f4;
    static __device__ inline V mul(float a, float b, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ inline int row(int q, int lk) { return 4 * lk + q; }
};

// acc[i][j] = sum_k A(k) B(k) over k < m, A and B loaders of (k, lane li);
// two accumulators shorten the dependent MFMA chain
template <typename T, typename LA, typename LB>
__device__ inline typename FdMfma<T>::V fd_tile(int m, int lk, LA la, LB lb)
{
    using M = FdMfma<T>;
    typename M::V c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
    const int full = m / 4;
    int ks = 0;
    for (; ks + 4 <= full; ks += 4) {
        T a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            a[u] = la(4 * (ks + u) + lk);
            b[u] = lb(4 * (ks + u) + lk);
        }
#pragma unroll
        for (int u = 0; u < 4; u += 2) {
            c0 = M::mul(a[u], b[u], c0);
            c1 = M::mul(a[u + 1], b[u + 1], c1);
        }
    }
    for (; 4 * ks < m; ++ks) {
        const int k = 4 * ks + lk;
        const T a = k < m ? la(k) : (T)0, b = k < m ? lb(k) : (T)0;
        c0 = M::mul(a, b, c0);
    }
    return c0 + c1;
}

// row stride of k_fd_pair's strip: the A operand is read across 16 rows, and a
// stride of 4 (mod 16) entries puts the 64 lanes on distinct banks
__host__ __device__ inline int fd_strip(int m0) { return (m0 + 15) / 16 * 16 + 4; }

// Plane c: y[j1][j0] = sum_{b, a} M1[b][j1] M0[a][j0] x[b][a]; optionally
// divided by alpha + l0[j0] + l1[j1] (2D).
template <typename T>
__global__ __launch_bounds__(1024) void k_fd_pair(int m0, int m1, const T *__restrict__ M0,
                                                  const T *__restrict__ M1, const T *__restrict__ x, int64_t xo,
                                                  int64_t xs1, int64_t xs2, T *__restrict__ y, int64_t yo,
                                                  int64_t ys1, int64_t ys2, const double *__restrict__ l0,
                                                  const double *__restrict__ l1, double alpha,
                                                  const CGState *__restrict__ st)
{
    extern __shared__ double fd_smem[];
    T *sT = reinterpret_cast<T *>(fd_smem);   // [16][LD]
    if (st && st->done) return;
    using M = FdMfma<T>;
    const int LD = fd_strip(m0), NT = (m0 + 15) / 16;
    const int nw = blockDim.x / 64, w = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 16, lk = l / 16;
    const int j1 = blockIdx.x * 16 + li;   // this lane's row of M1^T
    const bool ok1 = j1 < m1;
    const T *m1p = M1 + (ok1 ? j1 : 0);
    const T *xp = x + xo + (int64_t)blockIdx.y * xs2;
    for (int ct = w; ct < NT; ct += nw) {
        const int a = ct * 16 + li;
        const bool oka = a < m0;
        const T *xa = xp + (oka ? a : 0);
        const typename M::V c = fd_tile<T>(
            m1, lk, [&](int k) { return ok1 ? m1p[(int64_t)k * m1] : (T)0; },
            [&](int k) { return oka ? xa[k * xs1] : (T)0; });
#pragma unroll
        for (int q = 0; q < 4; ++q) sT[M::row(q, lk) * LD + a] = c[q];
    }
    __syncthreads();
    for (int ct = w; ct < NT; ct += nw) {
        const int j0 = ct * 16 + li;
        const bool ok0 = j0 < m0;
        const T *m0p = M0 + (ok0 ? j0 : 0);
        const typename M::V c = fd_tile<T>(
            m0, lk, [&](int k) { return sT[li * LD + k]; },
            [&](int k) { return ok0 ? m0p[(int64_t)k * m0] : (T)0; });
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = blockIdx.x * 16 + M::row(q, lk);
            if (!ok0 || r >= m1) continue;
            T v = c[q];
            if (l0) v = (T)((double)v / (alpha + l0[j0] + l1[r]));
            y[yo + j0 + r * ys1 + (int64_t)blockIdx.y * ys2] = v;
        }
    }
}

// Columns (a, b) of compact tensors: y[i] = sum_j QT[j][i] (sum_k Q[k][j] x[k]) /
// (alpha + l0[a] + l1[b] + l2[j]).
template <typename T>
__global__ __launch_bounds__(512) void k_fd_column(int m0, int m1, int m2, const T *__restrict__ Q,
                                                   const T *__restrict__ QT, const T *__restrict__ x,
                                                   T *__restrict__ y, const double *__restrict__ l0,
                                                   const double *__restrict__ l1, const double *__restrict__ l2,
                                                   double alpha, const CGState *__restrict__ st)
{
    extern __shared__ double fd_smem[];
    T *sT = reinterpret_cast<T *>(fd_smem);   // [m2 rounded up to 16][16]
    if (st && st->done) return;
    using M = FdMfma<T>;
    const int NT = (m2 + 15) / 16;
    const int nw = blockDim.x / 64, w = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 16, lk = l / 16;
    const int64_t n01 = (int64_t)m0 * m1, col = (int64_t)blockIdx.x * 16 + li;
    const bool okc = col < n01;
    const T *xc = x + (okc ? col : 0);
    const double l01 = okc ? alpha + l0[col % m0] + l1[col / m0] : 1.0;
    for (int rt = w; rt < NT; rt += nw) {
        const int j = rt * 16 + li;
        const bool okj = j < m2;
        const T *qp = Q + (okj ? j : 0);
        const typename M::V c = fd_tile<T>(
            m2, lk, [&](int k) { return okj ? qp[(int64_t)k * m2] : (T)0; },
            [&](int k) { return okc ? xc[k * n01] : (T)0; });
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = rt * 16 + M::row(q, lk);
            sT[r * 16 + li] = r < m2 ? (T)((double)c[q] / (l01 + l2[r])) : (T)0;
        }
    }
    __syncthreads();
    for (int rt = w; rt < NT; rt += nw) {
        const int i = rt * 16 + li;
        const bool oki = i < m2;
        const T *qp = QT + (oki ? i : 0);
        const typename M::V c = fd_tile<T>(
            m2, lk, [&](int k) { return oki ? qp[(int64_t)k * m2] : (T)0; },
            [&](int k) { return sT[k * 16 + li]; });
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = rt * 16 + M::row(q, lk);
            if (okc && r < m2) y[col + r * n01] = c[q];
        }
    }
}

constexpr size_t kFdLds = 64 * 1024;       // dynamic LDS a launch takes without opting in
constexpr size_t kFdSlabLds = 60 * 1024;   // of a slab

bool fd_fused(int d, int m0, int m1, int m2, size_t esz)
{
    // strips of 16 outputs in LDS; larger boxes take one mode product per launch
    if (16 * (size_t)fd_strip(m0) * esz > kFdLds || (d == 3 && 16 * (size_t)((m2 + 15) / 16 * 16) * esz > kFdLds))
        return false;
    // so do thin boxes, whose long sums fall to a few blocks of the fused kernels
    // and to many of the slab form.  FP64 apply, fused / slabs: 4 x 4 x 128 21 / 32
    // us, x 200 38 / 35, x 300 69 / 40; 12 x 12 x 300 71 / 50, 16 x 16 x 300 70 / 69;
    // 200 x 4 x 4 29 / 37, 300 x 4 x 4 54 / 46, 300 x 8 x 8 56 / 57; 2D 200 x 4 25 /
    // 28, 300 x 4 50 / 36, 300 x 16 53 / 54, 450 x 12 87 / 67
    const bool slabs = (size_t)(m1 > m2 ? m1 : m2) * m0 * esz <= kFdSlabLds;
    const int64_t pair_blocks = (int64_t)((m1 + 15) / 16) * m2, column_blocks = ((int64_t)m0 * m1 + 15) / 16;
    return !(slabs && ((m2 >= 192 && column_blocks <= 16) || (m0 >= 256 && pair_blocks < (d == 3 ? 8 : 2))));
}

// waves of a block over nt tiles of 16: as many as share the tiles evenly
static unsigned fd_waves(int nt, int cap)
{
    const int rounds = (nt + cap - 1) / cap;
    return (unsigned)((nt + rounds - 1) / rounds);
}

template <typename T>
hipError_t launch_fd_pair_t(int m0, int m1, int m2, const T *M0, const T *M1, const T *x, int64_t xo, int64_t xs1,
                            int64_t xs2, T *y, int64_t yo, int64_t ys1, int64_t ys2, const double *l0,
                            const double *l1, double alpha, const CGState *st, hipStream_t s)
{
    if ((int64_t)m0 * m1 * m2 <= 0) return hipSuccess;
    if (m2 > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((m1 + 15) / 16), (unsigned)m2);
    hipLaunchKernelGGL((k_fd_pair<T>), grid, dim3(64 * fd_waves((m0 + 15) / 16, 16)),
                       16 * (size_t)fd_strip(m0) * sizeof(T), s, m0, m1, M0, M1, x, xo, xs1, xs2, y, yo, ys1, ys2,
                       l0, l1, alpha, st);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_fd_column_t(int m0, int m1, int m2, const T *Q, const T *QT, const T *x, T *y, const double *l0,
                              const double *l1, const double *l2, double alpha, const CGState *st, hipStream_t s)
{
    const int64_t n01 = (int64_t)m0 * m1;
    if (n01 * m2 <= 0) return hipSuccess;
    const int nt = (m2 + 15) / 16;
    hipLaunchKernelGGL((k_fd_column<T>), dim3((unsigned)((n01 + 15) / 16)), dim3(64 * fd_waves(nt, 8)),
                       16 * (size_t)nt * 16 * sizeof(T), s, m0, m1, m2, Q, QT, x, y, l0, l1, l2, alpha, st);
    return hipGetLastError();
}

#define GSX_FD_T(SUF, T)                                                                                          \
    hipError_t launch_fd_pair_##SUF(int m0, int m1, int m2, const T *M0, const T *M1, const T *x, int64_t xo,     \
                                    int64_t xs1, int64_t xs2, T *y, int64_t yo, int64_t ys1, int64_t ys2,         \
                                    const double *l0, const double *l1, double alpha, const CGState *st,          \
                                    hipStream_t s)                                                                \
    {                                                                                                             \
        return launch_fd_pair_t<T>(m0, m1, m2, M0, M1, x, xo, xs1, xs2, y, yo, ys1, ys2, l0, l1, alpha, st, s);   \
    }                                                                                                             \
    hipError_t launch_fd_column_##SUF(int m0, int m1, int m2, const T *Q, const T *QT, const T *x, T *y,          \
                                      const double *l0, const double *l1, const double *l2, double alpha,         \
                                      const CGState *st, hipStream_t s)                                           \
    {                                                                                                             \
        return launch_fd_column_t<T>(m0, m1, m2, Q, QT, x, y, l0, l1, l2, alpha, st, s);                          \
    }
GSX_FD_T(f64, double)
GSX_FD_T(f32, float)
#undef GSX_FD_T

template <typename T>
hipError_t launch_fd_mode_t(int m0, int m1, int m2, int dir, const T *M, const T *x, int64_t xo, int64_t xs1,
                            int64_t xs2, T *y, int64_t yo, int64_t ys1, int64_t ys2, const double *l0,
                            const double *l1, const double *l2, double alpha, const CGState *st, hipStream_t s)
{
    const int64_t n = (int64_t)m0 * m1 * m2;
    if (n <= 0) return hipSuccess;
    if (dir < 0 || dir > 2) return hipErrorInvalidValue;
    const int rows = dir == 2 ? m2 : m1;
    const size_t lds = sizeof(T) * (size_t)rows * m0;
    if (lds <= kFdSlabLds && (dir == 2 ? m1 : m2) <= 65535) {
        const dim3 grid((unsigned)((rows * m0 + 255) / 256), (unsigned)(dir == 2 ? m1 : m2));
#define GSX_SLAB(DIR)                                                                                                  \
    if (dir == DIR)                                                                                                    \
        hipLaunchKernelGGL((k_fd_slab<T, DIR>), grid, dim3(256), lds, s, m0, m1, m2, M, x, xo, xs1, xs2, y, yo, ys1,   \
                           ys2, l0, l1, l2, alpha, st);
        GSX_SLAB(0) GSX_SLAB(1) GSX_SLAB(2)
#undef GSX_SLAB
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_fd_mode<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m0, m1, m2, dir, M, x,
                       xo, xs1, xs2, y, yo, ys1, ys2, l0, l1, l2, alpha, st);
    return hipGetLastError();
}

hipError_t launch_fd_mode_f64(int m0, int m1, int m2, int dir, const double *M, const double *x, int64_t xo,
                              int64_t xs1, int64_t xs2, double *y, int64_t yo, int64_t ys1, int64_t ys2,
                              const double *l0, const double *l1, const double *l2, double alpha,
                              const CGState *st, hipStream_t s)
{
    return launch_fd_mode_t<double>(m0, m1, m2, dir, M, x, xo, xs1, xs2, y, yo, ys1, ys2, l0, l1, l2, alpha, st, s);
}

hipError_t launch_fd_mode_f32(int m0, int m1, int m2, int dir, const float *M, const float *x, int64_t xo,
                              int64_t xs1, int64_t xs2, float *y, int64_t yo, int64_t ys1, int64_t ys2,
                              const double *l0, const double *l1, const double *l2, double alpha,
                              const CGState *st, hipStream_t s)
{
    return launch_fd_mode_t<float>(m0, m1, m2, dir, M, x, xo, xs1, xs2, y, yo, ys1, ys2, l0, l1, l2, alpha, st, s);
}

// Rectangular mode product of the subspace corrected mass smoother: output
// box o0 x o1 x o2, along direction dir the input has m_in entries and
// y_a = sum_{i < m_in} M[i*o_dir + a] x_i; optionally divided by
// alpha + l0[a] + l1[b] + l2[c] (null arrays count 0) and added to y.
template <typename T>
__global__ __launch_bounds__(256) void k_tensor_mode(int o0, int o1, int o2, int dir, int m_in,
                                                     const T *__restrict__ M, const T *__restrict__ x, int64_t xo,
                                                     int64_t xs1, int64_t xs2, T *__restrict__ y, int64_t yo,
                                                     int64_t ys1, int64_t ys2, int scale, double alpha,
                                                     const double *__restrict__ l0, const double *__restrict__ l1,
                                                     const double *__restrict__ l2, int accumulate,
                                                     const CGState *__restrict__ st)
{
    if (st && st->done) return;
    const int64_t n = (int64_t)o0 * o1 * o2;
    const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (o >= n) return;
    const int a = (int)(o % o0), b = (int)((o / o0) % o1), c = (int)(o / ((int64_t)o0 * o1));
    const int od = dir == 0 ? o0 : (dir == 1 ? o1 : o2);
    const int j = dir == 0 ? a : (dir == 1 ? b : c);
    const int64_t stride = dir == 0 ? 1 : (dir == 1 ? xs1 : xs2);
    const int64_t base = xo + (dir == 0 ? 0 : a) + (dir == 1 ? 0 : b * xs1) + (dir == 2 ? 0 : c * xs2);
    double acc = 0.0;
    for (int i = 0; i < m_in; ++i) acc += (double)M[(int64_t)i * od + j] * (double)x[base + i * stride];
    if (scale) acc /= alpha + (l0 ? l0[a] : 0.0) + (l1 ? l1[b] : 0.0) + (l2 ? l2[c] : 0.0);
    const int64_t at = yo + a + b * ys1 + c * ys2;
    y[at] = accumulate ? (T)((double)y[at] + acc) : (T)acc;
}

template <typename T>
hipError_t launch_tensor_mode_t(int o0, int o1, int o2, int dir, int m_in, const T *M, const T *x, int64_t xo,
                                int64_t xs1, int64_t xs2, T *y, int64_t yo, int64_t ys1, int64_t ys2, int scale,
                                double alpha, const double *l0, const double *l1, const double *l2, int accumulate,
                                const CGState *st, hipStream_t s)
{
    const int64_t n = (int64_t)o0 * o1 * o2;
    if (n <= 0) return hipSuccess;
    if (dir < 0 || dir > 2 || m_in <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_tensor_mode<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, o0, o1, o2, dir, m_in,
                       M, x, xo, xs1, xs2, y, yo, ys1, ys2, scale, alpha, l0, l1, l2, accumulate, st);
    return hipGetLastError();
}

hipError_t launch_tensor_mode_f64(int o0, int o1, int o2, int dir, int m_in, const double *M, const double *x,
                                  int64_t xo, int64_t xs1, int64_t xs2, double *y, int64_t yo, int64_t ys1,
                                  int64_t ys2, int scale, double alpha, const double *l0, const double *l1,
                                  const double *l2, int accumulate, const CGState *st, hipStream_t s)
{
    return launch_tensor_mode_t<double>(o0, o1, o2, dir, m_in, M, x, xo, xs1, xs2, y, yo, ys1, ys2, scale, alpha, l0,
                                        l1, l2, accumulate, st, s);
}

hipError_t launch_tensor_mode_f32(int o0, int o1, int o2, int dir, int m_in, const float *M, const float *x,
                                  int64_t xo, int64_t xs1, int64_t xs2, float *y, int64_t yo, int64_t ys1,
                                  int64_t ys2, int scale, double alpha, const double *l0, const double *l1,
                                  const double *l2, int accumulate, const CGState *st, hipStream_t s)
{
    return launch_tensor_mode_t<float>(o0, o1, o2, dir, m_in, M, x, xo, xs1, xs2, y, yo, ys1, ys2, scale, alpha, l0,
                                       l1, l2, accumulate, st, s);
}

}  // namespace gsx
