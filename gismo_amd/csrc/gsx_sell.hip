// Sliced ELL operators of the multigrid levels (libgsx, gfx950).
//
// The CSR kernels (gsx_csr.h) gather the input entry by entry: 64 lanes read
// two rows' worth of columns, scattered over some 18 runs, which bounds them
// near 3 TB/s of FP32 matrix bytes.  A level operator is applied hundreds of
// times per solve, so it is stored a second time in slices of 64 rows,
// [slice][k][row]: lane = row, the values of entry k are contiguous, and the
// columns of consecutive rows are (nearly) consecutive, so the gather coalesces
// too.  In a slice whose 64 rows have the same column offsets (col - row), as
// rows inside a patch do, the offsets are stored once and no columns are read:
// 4 bytes per FP32 entry instead of 8.  Rows shorter than the slice's widest
// are padded with zero entries in the row's own column.  Bound by the matrix
// bytes.  1.06 M rows of 49 entries (16 patches of 256^2 elements, p = 3), CSR
// kernels against slices: Jacobi step on FP32 values with FP64 vectors 142 / 69
// us, residual 133 / 64 us, FP64 SpMV 157 / 109 us; the slices of that level
// take 0.78 ms to fill, 19 iterations of V(2,2) apply them 95 times.
#include "gsx_common.h"
#include "gsx_kernels.h"

namespace gsx {

// width of every slice: the longest of its rows
__global__ __launch_bounds__(256) void k_sell_width(int n, const int *__restrict__ rowptr, int *__restrict__ width)
{
    const int sl = (int)(((int64_t)blockIdx.x * 256 + threadIdx.x) / 64), r = sl * 64 + (threadIdx.x & 63);
    if (sl * 64 >= n) return;   // the whole wave leaves
    int w = r < n ? rowptr[r + 1] - rowptr[r] : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) w = max(w, __shfl_xor(w, off, 64));
    if ((threadIdx.x & 63) == 0) width[sl] = w;
}

// A block per slice: columns (or, uniform slices, offsets) and values.  The
// values go through LDS, as many rows at a time as fit (all 64 up to 64 entries
// each), so the CSR array is read and the slice written coalesced; longer rows
// are copied entry by entry.  Whether a slice is uniform is tested over its
// entries as one range, all loads independent; only other slices read their
// columns again.  Bound by the bytes: 1.06 M rows of
// 49 entries 374 us (16 rows at a time with their columns, row by row tests: 780).
constexpr int kSellLds = 4096;
template <typename VO>
__global__ __launch_bounds__(256) void k_sell_fill(int n, const int *__restrict__ rowptr, const int *__restrict__ col,
                                                   const double *__restrict__ val, const int *__restrict__ sptr,
                                                   int *__restrict__ uniform, int *__restrict__ scol,
                                                   VO *__restrict__ sval, double *__restrict__ sval64)
{
    __shared__ double sv[kSellLds];
    __shared__ int srp[65];
    const int sl = blockIdx.x, t = threadIdx.x, r0 = sl * 64, nr = min(64, n - r0);
    const int K = sptr[sl + 1] - sptr[sl];
    const int64_t base = (int64_t)sptr[sl] * 64;
    if (t < 65) srp[t] = rowptr[r0 + min(t, nr)];
    __syncthreads();
    // uniform: every row has K entries at the first row's offsets
    const int a0 = srp[0];
    int bad = nr < 64 || (t < 64 && srp[t + 1] - srp[t] != K);
    bad = __syncthreads_count(bad);
    if (!bad) {
        int off = 0;
#pragma unroll 4
        for (int e = t; e < 64 * K; e += 256) {
            const int i = e / K;
            off |= col[a0 + e] - i - col[a0 + e - i * K];
        }
        bad = __syncthreads_count(off != 0);
    }
    const int uni = !bad;
    if (t == 0) uniform[sl] = uni;
    if (uni)
        for (int k = t; k < K; k += 256) scol[base + k] = col[a0 + k] - r0;
    const int sh = 64 * K <= kSellLds ? 6 : 32 * K <= kSellLds ? 5 : 4, R = 1 << sh;   // rows at a time
    const bool lds = R * K <= kSellLds;
    for (int q = 0; q < 64; q += R) {
        const int b0 = srp[q], b1 = srp[q + R];
        if (lds) {
            __syncthreads();
            for (int k = b0 + t; k < b1; k += 256) sv[k - b0] = val[k];
            __syncthreads();
        }
        const int i = q + (t & (R - 1));
        const int ra = srp[i], len = srp[i + 1] - ra;   // 0 beyond the last row
        for (int k = t >> sh; k < K; k += 256 >> sh) {
            const int64_t at = base + (int64_t)k * 64 + i;
            const double v = k < len ? (lds ? sv[ra + k - b0] : val[ra + k]) : 0.0;
            sval[at] = (VO)v;
            if (sval64) sval64[at] = v;
            if (!uni) scol[at] = k < len ? col[ra + k] : min(r0 + i, n - 1);
        }
    }
}

// acc = row sum of this lane's row over the entries part, part + step, ...
template <typename V, typename T>
__device__ inline double sell_sum(const SellOp &S, const V *__restrict__ sval, const T *__restrict__ x, int sl, int r,
                                  int part, int step)
{
    const int lane = threadIdx.x & 63;
    const int p0 = S.sptr[sl], K = S.sptr[sl + 1] - p0;
    const V *v = sval + (int64_t)p0 * 64 + lane;
    const int *c = S.col + (int64_t)p0 * 64;
    double acc = 0.0;
    constexpr int U = 8;
    // eight products in a tree: a row's sum rounds through a chain of K / 8
    // chunks, not of K products
    auto chunk = [](const V *a, const double *q) {
        double h[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) h[u] = (double)a[u] * q[u] + (double)a[u + 4] * q[u + 4];
        return (h[0] + h[1]) + (h[2] + h[3]);
    };
    double q[U];
    int k = part;
    if (S.uniform[sl]) {
        const T *xr = x + r;
        for (; k + (U - 1) * step < K; k += U * step) {
            V a[U];
            T b[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                a[u] = v[(int64_t)(k + u * step) * 64];
                b[u] = xr[c[k + u * step]];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) q[u] = (double)b[u];
            acc += chunk(a, q);
        }
        for (; k < K; k += step) acc += (double)v[(int64_t)k * 64] * (double)xr[c[k]];
    } else {
        c += lane;
        for (; k + (U - 1) * step < K; k += U * step) {
            V a[U];
            int j[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                a[u] = v[(int64_t)(k + u * step) * 64];
                j[u] = c[(int64_t)(k + u * step) * 64];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) q[u] = (double)x[j[u]];
            acc += chunk(a, q);
        }
        for (; k < K; k += step) acc += (double)v[(int64_t)k * 64] * (double)x[c[(int64_t)k * 64]];
    }
    return acc;
}

// WPS waves share a slice (small levels, where one wave per slice leaves the
// chip idle); the row sum then sits in the first wave.  Returns whether this
// thread finishes row r.
template <int WPS, typename V, typename T>
__device__ inline bool sell_row(const SellOp &S, const V *__restrict__ sval, const T *__restrict__ x, int &r,
                                double &acc)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nsl = (S.n + 63) / 64;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int sl = __builtin_amdgcn_readfirstlane(WPS == 1 ? blk * 4 + w : blk);
    r = sl * 64 + lane;
    acc = 0.0;
    // padded rows of the last slice hold zero entries; their reads stay on row n - 1
    if (sl < nsl) acc = sell_sum(S, sval, x, sl, min(r, S.n - 1), WPS == 1 ? 0 : w, WPS);
    if (WPS > 1) {
        __shared__ double red[WPS][64];
        red[w][lane] = acc;
        __syncthreads();
        if (w > 0) return false;
        for (int q = 1; q < WPS; ++q) acc += red[q][lane];
    }
    return sl < nsl && r < S.n;
}

template <int WPS, typename V, typename T>
__global__ __launch_bounds__(256) void k_sell_jacobi(SellOp S, const V *__restrict__ sval, const T *__restrict__ diag,
                                                     const T *__restrict__ b, const T *__restrict__ xin,
                                                     T *__restrict__ xout, T tau)
{
    int r;
    double acc;
    if (sell_row<WPS>(S, sval, xin, r, acc))
        xout[r] = (T)((double)xin[r] + (double)tau * ((double)b[r] - acc) / (double)diag[r]);
}

template <int WPS, typename V, typename T>
__global__ __launch_bounds__(256) void k_sell_residual(SellOp S, const V *__restrict__ sval, const T *__restrict__ x,
                                                       const T *__restrict__ b, T *__restrict__ y)
{
    int r;
    double acc;
    if (sell_row<WPS>(S, sval, x, r, acc)) y[r] = (T)((double)b[r] - acc);
}

// y = A x, partial[block] = sum x_i y_i
template <int WPS>
__global__ __launch_bounds__(256) void k_sell_spmv(SellOp S, const double *__restrict__ sval,
                                                   const double *__restrict__ x, double *__restrict__ y,
                                                   double *__restrict__ partial, const CGState *__restrict__ state)
{
    __shared__ double s[4];
    if (state && state->done) return;
    int r;
    double acc, v = 0.0;
    if (sell_row<WPS>(S, sval, x, r, acc)) {
        y[r] = acc;
        v = x[r] * acc;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (WPS > 1) {
        if (threadIdx.x == 0) partial[blockIdx.x] = v;
    } else {
        if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) partial[blockIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
    }
}

// below this many rows (two waves per SIMD) a slice is shared by four waves
constexpr int kSellSplitRows = 131072;
static bool split(int n) { return n < kSellSplitRows; }
int sell_blocks(int n) { return split(n) ? (n + 63) / 64 : (n + 255) / 256; }

hipError_t launch_sell_width(int n, const int *rowptr, int *width, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sell_width, dim3((n + 255) / 256), dim3(256), 0, s, n, rowptr, width);
    return hipGetLastError();
}

hipError_t launch_sell_fill(int n, const int *rowptr, const int *col, const double *val, const int *sptr, int *uniform,
                            int *scol, float *sval32, double *sval64, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const dim3 grid((n + 63) / 64), blk(256);
    if (sval32)
        hipLaunchKernelGGL((k_sell_fill<float>), grid, blk, 0, s, n, rowptr, col, val, sptr, uniform, scol, sval32,
                           sval64);
    else
        hipLaunchKernelGGL((k_sell_fill<double>), grid, blk, 0, s, n, rowptr, col, val, sptr, uniform, scol, sval64,
                           (double *)nullptr);
    return hipGetLastError();
}

template <typename V, typename T>
static hipError_t sell_jacobi(const SellOp &S, const V *v, const T *diag, const T *b, const T *xin, T *xout, T tau,
                              hipStream_t s)
{
    const dim3 grid(sell_blocks(S.n)), blk(256);
    if (split(S.n)) hipLaunchKernelGGL((k_sell_jacobi<4, V, T>), grid, blk, 0, s, S, v, diag, b, xin, xout, tau);
    else hipLaunchKernelGGL((k_sell_jacobi<1, V, T>), grid, blk, 0, s, S, v, diag, b, xin, xout, tau);
    return hipGetLastError();
}

template <typename V, typename T>
static hipError_t sell_residual(const SellOp &S, const V *v, const T *x, const T *b, T *y, hipStream_t s)
{
    const dim3 grid(sell_blocks(S.n)), blk(256);
    if (split(S.n)) hipLaunchKernelGGL((k_sell_residual<4, V, T>), grid, blk, 0, s, S, v, x, b, y);
    else hipLaunchKernelGGL((k_sell_residual<1, V, T>), grid, blk, 0, s, S, v, x, b, y);
    return hipGetLastError();
}

hipError_t launch_sell_jacobi_f64(const SellOp &S, const double *v, const double *diag, const double *b,
                                  const double *xin, double *xout, double tau, hipStream_t s)
{
    return sell_jacobi(S, v, diag, b, xin, xout, tau, s);
}

hipError_t launch_sell_jacobi_v32(const SellOp &S, const float *v, const double *diag, const double *b,
                                  const double *xin, double *xout, double tau, hipStream_t s)
{
    return sell_jacobi(S, v, diag, b, xin, xout, tau, s);
}

hipError_t launch_sell_jacobi_f32(const SellOp &S, const float *v, const float *diag, const float *b,
                                  const float *xin, float *xout, float tau, hipStream_t s)
{
    return sell_jacobi(S, v, diag, b, xin, xout, tau, s);
}

hipError_t launch_sell_residual_f64(const SellOp &S, const double *v, const double *x, const double *b, double *y,
                                    hipStream_t s)
{
    return sell_residual(S, v, x, b, y, s);
}

hipError_t launch_sell_residual_v32(const SellOp &S, const float *v, const double *x, const double *b, double *y,
                                    hipStream_t s)
{
    return sell_residual(S, v, x, b, y, s);
}

hipError_t launch_sell_residual_f32(const SellOp &S, const float *v, const float *x, const float *b, float *y,
                                    hipStream_t s)
{
    return sell_residual(S, v, x, b, y, s);
}

hipError_t launch_sell_spmv(const SellOp &S, const double *v, const double *x, double *y, double *partial,
                            const CGState *st, hipStream_t s)
{
    const dim3 grid(sell_blocks(S.n)), blk(256);
    if (split(S.n)) hipLaunchKernelGGL((k_sell_spmv<4>), grid, blk, 0, s, S, v, x, y, partial, st);
    else hipLaunchKernelGGL((k_sell_spmv<1>), grid, blk, 0, s, S, v, x, y, partial, st);
    return hipGetLastError();
}

}  // namespace gsx
