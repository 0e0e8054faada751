// Row sums of CSR matrices (libgsx, gfx950), shared by the SpMV, the residual
// and the damped Jacobi step.
//
// A wavefront takes 64 / L consecutive rows at a time.  Their entries are one
// contiguous range of the value and column arrays: the lanes read it in pairs
// of entries (8 to 16 byte loads, coalesced whatever the row lengths are),
// form the products with the gathered input and put them into the wave's LDS
// buffer; then L lanes per row sum the row's part of the buffer.  Bound by the
// matrix bytes.  Waves work without block barriers, several loads in flight
// each.  The other way (DIRECT), L lanes reading their row, keeps two loads per
// lane in flight at 49 entries per row, idles a quarter of the lanes in the
// last one and spends five shuffles per row, but it is the shorter chain and
// needs no buffer: it is taken where all rows are on the chip at once, and for
// rows longer than the buffer serves well (csr_direct).
// 1.06 M rows of 49 entries (16 patches of 256^2 elements, p = 3): FP64 SpMV
// 157 us (4.0 TB/s of matrix bytes; direct rows 249 us), damped Jacobi step on
// FP32 values with FP64 vectors 142 us (225 us).  69 K rows: 11.7 us (14.9 us).
#pragma once

#include "gsx_common.h"

namespace gsx {

constexpr int kCsrCap = 512;         // products a wave buffers
constexpr int kCsrMaxBlocks = 2048;  // blocks of 4 waves; more rows: more groups per wave

// lpr: the class of the mean row length (spmv_lpr), kCsrLong for the longest.
// A wave's buffer sums a row with lpr / 4 lanes, direct rows take lpr (64 for
// long ones).
constexpr int kCsrLong = 128;

// Direct rows where a lane per lpr entries' worth of rows fits the chip (256
// CUs x 2048 lanes), or for long rows.  Direct / buffered, FP64 SpMV: 36 rows
// 3.3 / 4.2 us, 4096 rows of 25 3.4 / 4.2, 14 K rows of 81 5.8 / 6.4, 8 K rows
// of 125 4.6 / 4.3 (512 K lanes); beyond the line 66 K rows of 25 7.6 / 6.2.
// Long rows: 39 K rows of 729 69 / 81 us, 16 K of 280 12.6 / 13.2; 262 K of 330
// 262 / 258.
__host__ __device__ inline bool csr_direct(int n, int lpr)
{
    return lpr == kCsrLong || (int64_t)n * lpr <= 256 * 2048;
}

constexpr int csr_lanes(int lpr) { return lpr / 4; }

__host__ __device__ inline int csr_blocks(int n, int lpr)
{
    const bool direct = csr_direct(n, lpr);
    const int rows = direct ? 256 / (lpr > 64 ? 64 : lpr) : 4 * (64 / csr_lanes(lpr));
    const int nb = (n + rows - 1) / rows;
    return nb < 1 ? 1 : (nb > kCsrMaxBlocks && !direct ? kCsrMaxBlocks : nb);
}

template <typename V> struct CsrPair;
template <> struct CsrPair<double> { using type = double2; };
template <> struct CsrPair<float> { using type = float2; };

// epi(r, sum, pre(r)) once per row, in the row's first lane (pre's loads are
// issued with the row's entries); buf: kCsrCap entries of the calling wave.
// All blocks of 256 threads of the grid take part (csr_blocks).
template <int L, bool DIRECT, typename Acc, typename V, typename T, typename Pre, typename Epi>
__device__ inline void csr_rows(int n, const int *__restrict__ rowptr, const int *__restrict__ col,
                                const V *__restrict__ val, const T *__restrict__ x, Acc *buf, Pre pre, Epi epi)
{
    if constexpr (DIRECT) {
        const int r = blockIdx.x * (256 / L) + threadIdx.x / L;
        Acc acc = 0;
        if (r < n) {
            const int k1 = rowptr[r + 1];
            for (int k = rowptr[r] + threadIdx.x % L; k < k1; k += L) acc += (Acc)val[k] * (Acc)x[col[k]];
        }
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (r < n && threadIdx.x % L == 0) epi(r, acc, pre(r));
        return;
    }
    constexpr int RW = 64 / L, NU = kCsrCap / 128;
    using V2 = typename CsrPair<V>::type;
    const int lane = threadIdx.x & 63;
    const int64_t ngrp = (n + RW - 1) / RW, nwave = (int64_t)gridDim.x * 4;
    const int64_t wv = (int64_t)xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
    const int g0 = (int)(wv * ngrp / nwave), g1 = (int)((wv + 1) * ngrp / nwave);
    int r = g0 * RW + lane / L;
    int ka = rowptr[min(r, n)], kb = rowptr[min(r + 1, n)];
    for (int g = g0; g < g1; ++g) {
        const int k0 = __builtin_amdgcn_readfirstlane(ka);
        const int k1 = __builtin_amdgcn_readfirstlane(__shfl(kb, 63, 64));
        const bool head = r < n && lane % L == 0;
        const auto pv = pre(min(r, n - 1));
        // the next group's row bounds
        const int rn = r + RW;
        const int kan = rowptr[min(rn, n)], kbn = rowptr[min(rn + 1, n)];
        Acc acc = 0;
        for (int c0 = k0 & ~1; c0 < k1;) {
            const int m = min(kCsrCap, k1 - c0), m0 = k0 - c0;   // entries [max(m0, 0), m) of the chunk
            // branch-free, so that all loads of the chunk are in flight at
            // once: pairs beyond the chunk repeat its last one (the pair's
            // second entry lies inside the arrays' allocations, which are
            // rounded up to 256 bytes), entries outside it gather x[0]
            int2 cc[NU];
            V2 vv[NU];
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int o = min(128 * u + 2 * lane, (m - 1) & ~1);
                cc[u] = *reinterpret_cast<const int2 *>(col + c0 + o);
                vv[u] = *reinterpret_cast<const V2 *>(val + c0 + o);
            }
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int o = 128 * u + 2 * lane;
                const T xa = x[o >= m0 && o < m ? cc[u].x : 0], xb = x[o + 1 < m ? cc[u].y : 0];
                buf[o] = (Acc)vv[u].x * (Acc)xa;
                buf[o + 1] = (Acc)vv[u].y * (Acc)xb;
            }
            // one wave's LDS accesses run in order; keep the compiler from moving them
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int e = min(kb - c0, m);
            // two sums a lane: half the chain, and half its rounding
            Acc half = 0;
            int o = max(ka - c0, 0) + lane % L;
            for (; o + L < e; o += 2 * L) {
                acc += buf[o];
                half += buf[o + L];
            }
            if (o < e) acc += buf[o];
            acc += half;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (k1 - c0 <= kCsrCap) break;
            c0 += kCsrCap;
        }
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (head) epi(r, acc, pv);
        r = rn;
        ka = kan;
        kb = kbn;
    }
}

}  // namespace gsx
