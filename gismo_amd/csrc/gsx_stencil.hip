// Structured (stencil) operator of single-patch problems and the grid-layout
// CG kernels of libgsx (gfx950).
//
// On one tensor-product patch with open knots the row of free function i
// couples exactly the functions j with |j_k - i_k| <= p in every direction,
// so the row is a (2p+1)^d stencil.  The stencil operator stores, for every
// free row, all (2p+1)^d coefficients (zero where the neighbour is outside
// the patch or eliminated) in [stencil slot][row] order and no column
// indices.  Vectors live on the full tensor grid of basis functions with
// zeros at the eliminated functions, so neighbour indices are the row's grid
// index plus a constant offset.  Same products and summation order per row
// as the CSR SpMV (columns ascending = grid order).
//
// CG (gsConjugateGradient::step, src/gsSolver/gsConjugateGradient.hpp:55-93)
// in two launches per iteration: k_cg2_spmv tests the last residual, forms the
// direction p = z + beta p where it stages its input, applies the operator and
// writes partial (p, A p); k_cg2_update moves x and r, applies the Jacobi
// preconditioner and writes partial (r, r), (r, z).  Every block of a launch
// sums the previous launch's partials itself (bounded counts, fixed order) and
// derives alpha or beta, so there is no single-block reduction kernel in the
// loop; block 0 records the scalars.  The direction of iteration k lives in
// buffer k & 1 (neighbouring blocks still read the old one while the new one
// is written), its (r, z) in slot k & 1.
#include "gsx_common.h"
#include "gsx_kernels.h"

#include <algorithm>

namespace gsx {

constexpr int kMaxPartials = 2048;

constexpr int kVecThreads = 512;   // threads of the vector kernels' blocks

// block sum of NT threads: wavefront shuffles, then the wave sums in wave
// order (fixed order: bitwise reproducible)
template <int NT>
__device__ inline double bsum(double v, double *s)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) r += s[w];
    __syncthreads();
    return r;
}

// two sums with one pair of barriers (s: 2 NT / 64 doubles)
template <int NT>
__device__ inline void bsum2(double &a, double &b, double *s)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        b += __shfl_xor(b, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        s[threadIdx.x >> 6] = a;
        s[NT / 64 + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    a = b = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        a += s[w];
        b += s[NT / 64 + w];
    }
    __syncthreads();
}

template <int NT>
__device__ inline double sum_partials(const double *__restrict__ p, int np, double *s)
{
    double a = 0.0;
    for (int i = threadIdx.x; i < np; i += NT) a += p[i];
    return bsum<NT>(a, s);
}

template <typename T>
__global__ void k_fill(T *__restrict__ a, int64_t n, T v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// CSR (free numbering, sorted columns) -> stencil slots.  One thread per row.
template <int D, int P>
__global__ void k_csr_to_stencil(int nfree, const int *__restrict__ rowptr,
                                 const int *__restrict__ col, const double *__restrict__ val,
                                 const int *__restrict__ free2grid, int nbx, int nby,
                                 double *__restrict__ s64, float *__restrict__ s32)
{
    constexpr int W = 2 * P + 1;
    constexpr int NS = (D == 3) ? W * W * W : W * W;
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nfree) return;
    const int g = free2grid[r];
    const int gx = g % nbx, gy = (g / nbx) % nby, gz = g / (nbx * nby);
    for (int k = rowptr[r]; k < rowptr[r + 1]; ++k) {
        const int h = free2grid[col[k]];
        const int dx = h % nbx - gx, dy = (h / nbx) % nby - gy;
        const int dz = (D == 3) ? h / (nbx * nby) - gz : 0;
        const int slot = (D == 3) ? ((dz + P) * W + (dy + P)) * W + (dx + P) : (dy + P) * W + (dx + P);
        if (s64) s64[stencil_index(slot, r, NS)] = val[k];
        if (s32 && slot >= NS / 2) s32[stencil_index(slot - NS / 2, r, stencil_half(NS))] = (float)val[k];
    }
}

// diagonal (centre slot) of the structured operator onto the grid
__global__ void k_stencil_diag(int nfree, int ns, int centre, const int *__restrict__ free2grid,
                               const double *__restrict__ s64, double *__restrict__ dst)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nfree) dst[free2grid[r]] = s64[stencil_index(centre, r, ns)];
}

template <typename S, typename Dt>
__global__ void k_scatter_to_grid(int nfree, const int *__restrict__ free2grid,
                                  const S *__restrict__ src, Dt *__restrict__ dst)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nfree) dst[free2grid[r]] = (Dt)src[r];
}

template <typename S>
__global__ void k_gather_from_grid(int nfree, const int *__restrict__ free2grid,
                                   const S *__restrict__ src, double *__restrict__ dst)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nfree) dst[r] = (double)src[free2grid[r]];
}

// ---------------------------------------------------------------------------
// Stencil SpMV.  Vectors on the grid; rows = free functions, the free box
// m0 x m1 x m2 in lexicographic order.  MODE 1, iteration k of CG: stop test,
// pn = x + beta po (x is the preconditioned residual z), y = A pn, partial
// (pn, y).  MODE 2: y = b - A x, partial (y, y).
//
// KIND 0, the FP32 copy: only the upper slots are stored (stencil_half).
// KIND 1, 2, the FP64 operator: all slots are stored.  With KIND 0 and 1 an
// upper slot is read from the row itself and a lower one from the neighbour
// row at that offset, whose mirrored upper slot holds the same coefficient
// (the operator is bitwise symmetric): half the bytes of the operator move.
// Each upper x-line of the stencil, (dz, dy) > 0 lexicographically, is taken
// together with its mirror line (-dz, -dy): both read the same slot plane, the
// mirror one at the rows shifted by the offset, so a block reads the plane at
// the same point of its loop as the blocks that own those rows (up to p
// z-planes back, on the same XCD through xcd_block) and part of the second
// reads hit the L2 (64^3 elements p = 3: FP32 moves 1.40 times the upper half
// and the vectors, FP64 1.73 times).  Neighbours outside the free box contribute 0 (x is 0 there).
// KIND 2 reads every slot from the row itself, with fewer index operations.
//
// The input of a block's 256 rows is staged in LDS, in planes dz and -dz: it is
// read from memory once instead of once per coefficient, and in MODE 1 the
// direction is formed there, which saves its own launch.  Staged is the window
// of grid entries around the rows, lines -p .. p of them whole, or, where that
// is less (lines longer than about 150 entries), the 2 p + 1 stretches of lines
// that the rows reach (SpmvStage).  What does not fit (STAGED = 0) is read
// entry by entry.  With the whole windows alone 32 mixed CG iterations took 7.8
// ms at 1800^2 elements p = 2 (now 4.3) and 24.8 ms at 2600^2 (8.4), FP64 ones
// 15.0 (6.7) and 20.0 ms (13.2).
// Entries are requested ahead of the barrier that they are waited for at: the
// next tile's window before a tile's last plane is applied and, PLANES, the next
// planes' first entries before a plane is.
// Bound by the operator's bytes and the mirrored reads that miss the L2.  64^3
// elements p = 3: FP32 50 us with the direction (5.5 TB/s), FP64 118 us with it
// (5.7 TB/s), FP64 residual 110 us (159 us reading all slots).  75^3 p = 2, FP64:
// 54.5 us with the direction (89 + 7 us reading all slots).
// ---------------------------------------------------------------------------
template <int D, int P, typename V, typename T, int KIND, int MODE, int STAGED, int Q, int PLANES>
// (windows of degree 4 in FP64: within the registers of four waves a SIMD)
__global__ __launch_bounds__(256 * Q, D == 3 && P == 4 && sizeof(T) == 8 && STAGED < 2 ? 4 : 1) void k_cg2_spmv(int nfree, const int *__restrict__ free2grid, int sy, int sz,
                                                  int m0, int m1, const V *__restrict__ sval,
                                                  const T *__restrict__ x, const T *__restrict__ po,
                                                  T *__restrict__ pn, T *__restrict__ y, const T *__restrict__ b,
                                                  double *__restrict__ partial, CGStep cs,
                                                  CGState *__restrict__ st, SpmvStage sg)
{
    extern __shared__ double sp_smem[];
    __shared__ double s[8 * Q];
    __shared__ T sq[Q > 1 ? Q - 1 : 1][256];
    constexpr int NT = 256 * Q;
    const int t = threadIdx.x & 255, q = Q > 1 ? threadIdx.x >> 8 : 0;   // row, group
    constexpr int W = 2 * P + 1;
    constexpr int NS = (D == 3) ? W * W * W : W * W;
    constexpr int C = NS / 2, SL = KIND == 0 ? stencil_half(NS) : NS;   // slots of the stored layout
    constexpr int UP = KIND == 0 ? 0 : C;                               // stored index of the centre slot
    static_assert(kStencilTile == 256, "one block applies one row tile");
    constexpr int UNR = STAGED == 2 && D == 2 && PLANES && P <= 2 && sizeof(T) == 4 ? 2 : 1;   // lines whose loads are in flight together
    if (MODE == 1 && (st->done || (st->flag_next && st->flag_next <= cs.k))) return;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    // staged entry i of a plane: entry i from w0 on.  STAGED = 2: entry j of line
    // i / sg.line from w0 on (one line where sg.magic is 0); with sg.plane a tile's
    // rows from `cut` on, which lie in the next plane of rows, have a window of
    // their own (w1) behind the first
    constexpr bool LINES = STAGED == 2;
    const int line_stride = LINES ? sg.line : sy, halo = LINES ? sg.halo : P * sy + P;
    int w0 = 0, w1 = 0, l0 = 0, l1 = 0, behind = 0, total = 0, cut = 0;
    auto window = [&](int r0) {
        const int g0 = free2grid[r0], rb = min(r0 + 256, nfree);
        cut = LINES && D == 3 && sg.plane ? min(rb, (r0 / sg.plane + 1) * sg.plane) : rb;
        w0 = g0 - P * sy - P;
        l0 = free2grid[cut - 1] - g0 + 1 + 2 * halo;
        behind = total = LINES && sg.magic ? W * sg.line : l0;
        if (LINES && D == 3 && cut < rb) {
            const int g1 = free2grid[cut];
            w1 = g1 - P * sy - P;
            l1 = free2grid[rb - 1] - g1 + 1 + 2 * halo;
            total += sg.magic ? W * sg.line : l1;
        }
    };
    auto source = [&](int i, bool &in) {
        in = true;
        if (!LINES) return w0 + i;
        const bool second = D == 3 && i >= behind;
        if (second) i -= behind;
        const int l = (int)__umulhi((unsigned)i, sg.magic), j = i - l * sg.line;
        in = j < (second ? l1 : l0);
        return (second ? w1 : w0) + l * sy + j;
    };
    // a tile's window is requested ahead: the first one's before the sums that
    // give beta, the next one's before the tile's last plane is applied
    constexpr int NB = LINES && D == 2 && PLANES && sizeof(T) == 4 && P > 1 ? 6 : PLANES > 4 ? PLANES : 4;
    constexpr int NPRE = MODE == 1 && STAGED ? (Q > 1 ? 1 : NB) : 0, NPA = NPRE ? NPRE : 1;
    constexpr bool AHEAD = NPRE > 0 && PLANES > 0 && (D == 3 || LINES);
    T prx[NPA], prp[NPA];
    auto request = [&](int first) {
        window(first);
#pragma unroll
        for (int u = 0; u < NPRE; ++u) {
            const int i = (int)threadIdx.x + NT * u;
            bool in;
            const int g = source(i, in);
            in = in && i < total;
            prx[u] = in ? x[g] : (T)0;
            prp[u] = in ? po[g] : (T)0;
        }
    };
    if (NPRE > 0) request(blk * 256);
    T tb = 0;
    if (MODE == 1) {
        double rr = 0.0, rzn = 0.0;
        for (int i = threadIdx.x; i < cs.np; i += NT) {
            rr += cs.part_rr[i];
            rzn += cs.part_rz[i];
        }
        bsum2<NT>(rr, rzn, s);
        const double err = sqrt(rr) / st->bnorm;
        // restart > 0: the residual has just been formed and tested in FP64
        const bool conv = !cs.restart && !cs.mixed && err < st->tol;
        const bool due = !cs.restart && cs.mixed && (rr < st->rel_since_update * st->rr_ref || err < st->tol);
        const double beta = cs.restart == 2 ? 0.0 : rzn / st->rzs[(cs.k + 1) & 1];
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            st->it = cs.k;
            st->rr = rr;
            st->err = err;
            if (cs.hist && !cs.restart) cs.hist[cs.k] = err;
            if (conv) st->done = 1;
            if (due) {
                // iterations from k on wait for the reliable update
                st->need_update = 1;
                st->flag_next = cs.k;
            }
            if (!conv && !due) {
                st->beta = beta;
                st->rzs[cs.k & 1] = rzn;
            }
        }
        // every block takes the same decision from the same partials, whether
        // or not it has seen block 0's record of it
        if (conv || due) return;
        tb = (T)beta;
    }
    const bool first = MODE == 1 && cs.restart == 2;   // the old direction is not read
    auto input = [&](int i) -> T {
        if (MODE == 2) return x[i];
        return first ? x[i] : x[i] + tb * po[i];
    };
    T *sA = reinterpret_cast<T *>(sp_smem), *sB = sA + sg.entries;
    double contrib = 0.0;
    for (int r0 = blk * 256; r0 < nfree; r0 += gridDim.x * 256) {
        const int r = r0 + t;
        const bool act = r < nfree, pre = NPRE > 0 && (AHEAD || r0 == blk * 256);
        if (STAGED && !pre) window(r0);
        const int g = act ? free2grid[r] : 0;
        const int ia = r % m0, ib = (r / m0) % m1, ic = (D == 3) ? r / (m0 * m1) : 0;
        const V *vb = sval + stencil_index(UP, r, SL);   // from the centre slot up
        // entry (dy, dx) around row r: c + dy line_stride + dx
        const int c = g - P * sy + P * line_stride - (LINES && D == 3 && r >= cut ? w1 - behind : w0);
        T acc = 0, own = 0;
        // the first entries of planes dz and -dz, requested before the plane
        // before them is applied
        constexpr int NPL = PLANES ? (Q > 1 ? 1 : PLANES) : 1;
        T ax[NPL], ap[NPL], mx[NPL], mp[NPL];
        auto request_plane = [&](int dz) {
#pragma unroll
            for (int u = 0; u < NPL; ++u) {
                bool in;
                const int i = (int)threadIdx.x + NT * u, from = source(i, in);
                in = in && i < total;
                ax[u] = in ? x[from + dz * sz] : (T)0;
                mx[u] = in ? x[from - dz * sz] : (T)0;
                if (MODE == 1) {
                    ap[u] = in ? po[from + dz * sz] : (T)0;
                    mp[u] = in ? po[from - dz * sz] : (T)0;
                }
            }
        };
        auto plane = [&](int dz) {
            if (STAGED) {
                __syncthreads();   // the readers of the last planes are done
                int i = threadIdx.x;
                if (pre && dz == 0) {
#pragma unroll
                    for (int u = 0; u < NPRE; ++u, i += NT)
                        if (i < total) sA[i] = first ? prx[u] : prx[u] + tb * prp[u];
                }
                if (PLANES && dz > 0) {
#pragma unroll
                    for (int u = 0; u < NPL; ++u, i += NT)
                        if (i < total) {
                            sA[i] = MODE == 2 || first ? ax[u] : ax[u] + tb * ap[u];
                            sB[i] = MODE == 2 || first ? mx[u] : mx[u] + tb * mp[u];
                        }
                }
                // stretches of lines, more entries than a window has, in batches of
                // loads; a window's without the registers of one
                constexpr int U = !LINES ? 1 : Q > 1 ? 2 : 4;
                for (; i < total; i += U * NT) {
                    T a[U], m[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        bool in;
                        const int from = source(i + u * NT, in);
                        in = in && i + u * NT < total;
                        a[u] = in ? input(from + dz * sz) : (T)0;
                        m[u] = D == 3 && dz > 0 && in ? input(from - dz * sz) : (T)0;
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        if (i + u * NT >= total) break;
                        sA[i + u * NT] = a[u];
                        if (D == 3 && dz > 0) sB[i + u * NT] = m[u];
                    }
                }
                __syncthreads();
            }
        };
        // entry (dy, dx) around the row in plane +dz / -dz
        auto xa = [&](int dz, int dy, int dx) -> T {
            return STAGED ? sA[c + dy * line_stride + dx] : input(g + dz * sz + dy * sy + dx);
        };
        auto xm = [&](int dz, int dy, int dx) -> T {
            if (!STAGED) return input(g - dz * sz + dy * sy + dx);
            return D == 3 && dz > 0 ? sB[c + dy * line_stride + dx] : sA[c + dy * line_stride + dx];
        };
        // upper line (dz, dy) and its mirror (-dz, -dy)
        auto line = [&](int dz, int dy) {
            const int h0 = (D == 3 ? ((dz + P) * W + (dy + P)) * W : (dy + P) * W) - C;   // (dz, dy, -P) from the centre
#pragma unroll
            for (int dx = -P; dx <= P; ++dx) acc += (T)vb[(h0 + dx + P) * kStencilTile] * xa(dz, dy, dx);
            if (KIND == 2) {
#pragma unroll
                for (int dx = -P; dx <= P; ++dx)
                    acc += (T)vb[-(h0 - dx + P) * kStencilTile] * xm(dz, -dy, dx);
            } else {
                const bool okyz = ib - dy >= 0 && ib - dy < m1 && ic - dz >= 0;
                const int rm = r - m0 * (dy + m1 * dz);
#pragma unroll
                for (int dx = -P; dx <= P; ++dx) {
                    const bool ok = okyz && ia + dx >= 0 && ia + dx < m0;
                    acc += (T)(ok ? sval[stencil_index(UP + h0 - dx + P, rm + dx, SL)] : (V)0) * xm(dz, -dy, dx);
                }
            }
        };
        plane(0);
        const bool more = AHEAD && r0 + (int)gridDim.x * 256 < nfree;
        if (D == 2 && more) request(r0 + gridDim.x * 256);
        if (PLANES) request_plane(1);
        if (act) {
            own = xa(0, 0, 0);
            // centre line: own slots dx = 0..P, mirrors dx = -P..-1
            if (q == 0) {
#pragma unroll
                for (int dx = 0; dx <= P; ++dx) acc += (T)vb[dx * kStencilTile] * xa(0, 0, dx);
#pragma unroll
                for (int dx = -P; dx < 0; ++dx) {
                    if (KIND == 2) acc += (T)vb[dx * kStencilTile] * xa(0, 0, dx);
                    else acc += (T)(ia + dx >= 0 ? sval[stencil_index(UP - dx, r + dx, SL)] : (V)0) * xa(0, 0, dx);
                }
            }
#pragma unroll(UNR)
            for (int dy = Q > 1 && q == 0 ? Q : (Q > 1 ? q : 1); dy <= P; dy += Q) line(0, dy);
        }
        if (D == 3) {
#pragma unroll 1
            for (int dz = 1; dz <= P; ++dz) {
                plane(dz);
                if (PLANES && dz < P) request_plane(dz + 1);
                if (dz == P && more) request(r0 + gridDim.x * 256);
                if (act) {
#pragma unroll(UNR)
                    for (int dy = -P + (q + dz) % Q; dy <= P; dy += Q) line(dz, dy);
                }
            }
        }
        if (Q > 1) {
            if (q) sq[q - 1][t] = acc;
            __syncthreads();
            if (q == 0)
#pragma unroll
                for (int u = 0; u + 1 < Q; ++u) acc += sq[u][t];
        }
        if (act && q == 0) {
            if (MODE == 2) {
                const T v = b[g] - acc;
                y[g] = v;
                contrib += (double)v * (double)v;
            } else {
                pn[g] = own;
                y[g] = acc;
                contrib += (double)own * (double)acc;
            }
        }
    }
    const double tot = bsum<NT>(contrib, s);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// ---------------------------------------------------------------------------
// grid-layout CG vector kernels (n = grid size; diag = 1 at eliminated
// functions so z stays 0 there)
// ---------------------------------------------------------------------------
// x += alpha p; r -= alpha t; z = tau r / diag; partials (r, r), (r, z).
// Every block derives alpha = rz_k / (p, A p) from the SpMV's partials
// itself (a bounded count, summed in a fixed order).
template <typename T, typename TX>
__global__ __launch_bounds__(kVecThreads) void k_cg2_update(int n, TX *__restrict__ x, T *__restrict__ r,
                                                            const T *__restrict__ p, const T *__restrict__ t,
                                                            T *__restrict__ z, const T *__restrict__ diag,
                                                            double tau, const double *__restrict__ pap_parts,
                                                            int npap, double *__restrict__ part_rr,
                                                            double *__restrict__ part_rz,
                                                            CGState *__restrict__ st, int k)
{
    __shared__ double s[2 * kVecThreads / 64];
    if (st->done || (st->flag_next && st->flag_next <= k)) return;
    // the first entries are requested before the sum that gives alpha
    int i = blockIdx.x * kVecThreads + threadIdx.x;
    T pi = 0, ti = 0, ri = 0, di = 1;
    TX xi = 0;
    auto load = [&]() {
        if (i < n) {
            pi = p[i];
            ti = t[i];
            ri = r[i];
            xi = x[i];
            if (diag) di = diag[i];
        }
    };
    load();
    const double pap = sum_partials<kVecThreads>(pap_parts, npap, s);
    const double alpha_d = st->rzs[k & 1] / pap;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->pap = pap;
        st->alpha = alpha_d;
    }
    const T alpha = (T)alpha_d;
    const T ta = (T)tau;
    double rr = 0.0, rz = 0.0;
    while (i < n) {
        x[i] = xi + (TX)(alpha * pi);
        const T rn = ri - alpha * ti;
        r[i] = rn;
        const T zi = diag ? ta * rn / di : rn;
        z[i] = zi;
        rr += (double)rn * (double)rn;
        rz += (double)rn * (double)zi;
        i += gridDim.x * kVecThreads;
        load();
    }
    bsum2<kVecThreads>(rr, rz, s);
    if (threadIdx.x == 0) {
        part_rr[blockIdx.x] = rr;
        part_rz[blockIdx.x] = rz;
    }
}

// The stop test of k_cg2_spmv on its own, after the last iteration of a chunk
// of launches: k iterations are complete.  MIXED == 0: reference stopping rule
// (err < tol stops).  MIXED == 1: FP32 recurrence of the mixed solver: never
// stops on its own residual, flags a reliable update instead and pauses until
// it has run.
__global__ __launch_bounds__(256) void k_cg2_check(CGStep cs, CGState *__restrict__ st)
{
    __shared__ double s[4];
    if (st->done || (st->flag_next && st->flag_next <= cs.k)) return;
    const double rr = sum_partials<256>(cs.part_rr, cs.np, s);
    if (threadIdx.x != 0) return;
    const double err = sqrt(rr) / st->bnorm;
    st->it = cs.k;
    st->rr = rr;
    st->err = err;
    if (cs.hist) cs.hist[cs.k] = err;
    if (!cs.mixed && err < st->tol) {
        st->done = 1;
    } else {
        if (cs.mixed && (rr < st->rel_since_update * st->rr_ref || err < st->tol)) {
            st->need_update = 1;
            st->flag_next = cs.k;
        }
        if (cs.k >= st->maxit) st->done = 2;
    }
}

// z = tau r / diag (or z = r), partials (r, r) and (r, z)
template <typename T>
__global__ __launch_bounds__(kVecThreads) void k_cg2_precond(int n, const T *__restrict__ r, T *__restrict__ z,
                                                             const T *__restrict__ diag, double tau,
                                                             double *__restrict__ part_rr,
                                                             double *__restrict__ part_rz)
{
    __shared__ double s[2 * kVecThreads / 64];
    double rr = 0.0, rz = 0.0;
    for (int i = blockIdx.x * kVecThreads + threadIdx.x; i < n; i += gridDim.x * kVecThreads) {
        const T ri = r[i];
        const T zi = diag ? (T)tau * ri / diag[i] : ri;
        z[i] = zi;
        rr += (double)ri * (double)ri;
        rz += (double)ri * (double)zi;
    }
    bsum2<kVecThreads>(rr, rz, s);
    if (threadIdx.x == 0) {
        part_rr[blockIdx.x] = rr;
        part_rz[blockIdx.x] = rz;
    }
}

// partial (a, b) in the grid solvers' block layout (a preconditioner that
// is not fused into the update writes z, then this gives the (r, z) partials)
template <typename T>
__global__ __launch_bounds__(kVecThreads) void k_cg2_dot(int n, const T *__restrict__ a, const T *__restrict__ b,
                                                         double *__restrict__ part, const CGState *__restrict__ st)
{
    __shared__ double s[kVecThreads / 64];
    if (st && st->done) return;
    double v = 0.0;
    for (int i = blockIdx.x * kVecThreads + threadIdx.x; i < n; i += gridDim.x * kVecThreads)
        v += (double)a[i] * (double)b[i];
    const double c = bsum<kVecThreads>(v, s);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
}

template <typename S, typename Dt>
__global__ void k_copy_convert(int64_t n, const S *__restrict__ a, Dt *__restrict__ b)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (Dt)a[i];
}

// x64 += xc32; xc32 = 0 (grid)
__global__ void k_accum_grid(int64_t n, double *__restrict__ x, float *__restrict__ xc)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        x[i] += (double)xc[i];
        xc[i] = 0.0f;
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline unsigned blocks_for(int64_t n, int nt, int cap)
{
    int64_t b = (n + nt - 1) / nt;
    if (b > cap) b = cap;
    if (b < 1) b = 1;
    return (unsigned)b;
}

int sspmv_blocks(int nfree) { return (int)blocks_for(nfree, 256, kMaxPartials); }
int vec_blocks(int64_t n) { return (int)blocks_for(n, kVecThreads, 512); }

template <typename T>
hipError_t launch_fill_t(T *a, int64_t n, T v, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL((k_fill<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, n, v);
    return hipGetLastError();
}

hipError_t launch_fill_f64(double *a, int64_t n, double v, hipStream_t s) { return launch_fill_t<double>(a, n, v, s); }
hipError_t launch_fill_f32(float *a, int64_t n, float v, hipStream_t s) { return launch_fill_t<float>(a, n, v, s); }

hipError_t launch_csr_to_stencil(int d, int p, int nfree, const int *rp, const int *ci,
                                 const double *v, const int *f2g, int nbx, int nby, double *s64,
                                 float *s32, hipStream_t s)
{
    const dim3 grid((nfree + 255) / 256), blk(256);
#define GSX_C(D, P) if (d == D && p == P) { hipLaunchKernelGGL((k_csr_to_stencil<D, P>), grid, blk, 0, s, nfree, rp, ci, v, f2g, nbx, nby, s64, s32); return hipGetLastError(); }
    GSX_C(2, 1) GSX_C(2, 2) GSX_C(2, 3) GSX_C(2, 4)
    GSX_C(3, 1) GSX_C(3, 2) GSX_C(3, 3) GSX_C(3, 4)
#undef GSX_C
    return hipErrorInvalidValue;
}

hipError_t launch_stencil_diag(int nfree, int ns, const int *f2g, const double *s64, double *diag_grid,
                              hipStream_t s)
{
    if (nfree <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stencil_diag, dim3((nfree + 255) / 256), dim3(256), 0, s, nfree, ns, (ns - 1) / 2, f2g, s64,
                       diag_grid);
    return hipGetLastError();
}

hipError_t launch_scatter_f64_to_grid(int nfree, const int *f2g, const double *src, double *dst, hipStream_t s)
{
    hipLaunchKernelGGL((k_scatter_to_grid<double, double>), dim3((nfree + 255) / 256), dim3(256), 0, s, nfree, f2g, src, dst);
    return hipGetLastError();
}

hipError_t launch_gather_f64_from_grid(int nfree, const int *f2g, const double *src, double *dst, hipStream_t s)
{
    hipLaunchKernelGGL((k_gather_from_grid<double>), dim3((nfree + 255) / 256), dim3(256), 0, s, nfree, f2g, src, dst);
    return hipGetLastError();
}

constexpr size_t kWindowLds = 64 * 1024;   // LDS of a tile's staged input

SpmvStage sspmv_stage(int d, int p, int nfree, int m0, int m1, int sy, int sz)
{
    auto grid = [&](int r) { return (int64_t)(r % m0) + (int64_t)sy * ((r / m0) % m1) + (int64_t)sz * (r / (m0 * m1)); };
    // span: grid entries that the rows of a tile in one plane reach over, whole:
    // the sum over its planes
    auto stage = [&](int plane) {
        int64_t span = 0, whole = 0, parts = 1;
        const int64_t halo = (int64_t)p * sy + p;
        for (int64_t r0 = 0; r0 < nfree; r0 += 256) {
            const int64_t e = std::min<int64_t>(r0 + 256, nfree);
            int64_t cut = plane ? std::min(e, (r0 / plane + 1) * (int64_t)plane) : e;
            const int64_t a = grid((int)cut - 1) - grid((int)r0) + 1;
            const int64_t b = cut < e ? grid((int)e - 1) - grid((int)cut) + 1 : 0;
            span = std::max({span, a, b});
            whole = std::max(whole, a + 2 * halo + (b ? b + 2 * halo : 0));
            if (b) parts = 2;
        }
        const int64_t line = span + 2 * p, lines = parts * line * (2 * p + 1);
        if (lines < whole)
            return SpmvStage{(int)std::min<int64_t>(lines, INT32_MAX), (int)line, p,
                             (unsigned)(((uint64_t)1 << 32) / (uint64_t)line + 1), plane};
        return SpmvStage{(int)std::min<int64_t>(whole, INT32_MAX), sy, (int)halo, 0u, plane};
    };
    SpmvStage g = stage(0);
    const int plane = m0 * m1;
    if (d == 3 && plane >= 256 && (size_t)g.entries * 2 * sizeof(double) > kWindowLds) g = stage(plane);
    return g;
}

// An FP64 operator of at most this many bytes (all slots) is read whole: it
// stays in the eight 4 MB L2s, where the mirrored reads' index operations cost
// more than the bytes they save.  Whole solves, all slots against mirrored:
// 64^2 p = 2 (0.8 MB) 1788 / 1967 us, 18^3 p = 3 (20 MB) 3662 / 4392 us;
// 75^3 p = 2 (422 MB) 12.5 / 7.4 ms.
constexpr int64_t kMirrorBytes = (int64_t)24 << 20;

// A 3D operator of at most a tile per CU leaves most of the chip idle: four
// groups of 256 threads then share a tile's stencil lines and one sums the
// parts.  CG solves, one group / four: 12^3 p = 4 mixed 25.5 / 16.3 ms, 32^3 p =
// 4 mixed 30.1 / 18.0 and FP64 31.5 / 22.6, 30^3 p = 3 mixed 5.3 / 3.9, 40^3 p =
// 2 mixed (250 tiles) 1.76 / 1.66; beyond the line 40^3 p = 3 FP64 (270 tiles)
// 6.5 / 7.5, 60^3 p = 3 mixed 8.6 / 12.0.  2D stencils have too few lines: 64^2
// p = 2 1.50 / 1.66 ms, 300^2 p = 4 mixed 8.4 / 10.4.
constexpr int kSplit = 4, kSplitTiles = 256;
// One such block runs on a CU, so its window may take more LDS: 1 x 1 x 500 p = 4
// FP64, 32 iterations, entry by entry 2.62 ms, staged 1.40; 1 x 1 x 600 p = 3 1.70
// and 1.21.
constexpr size_t kSplitLds = 128 * 1024;

// Entries per thread requested ahead for the next planes of a 3D tile: they hide
// two waits a plane, at registers.  Up to a tile for each of the four blocks a CU
// holds, waits bound the kernel; with more tiles only p = 2 in FP32 gains.
// 32 CG iterations without / with them: 50^3 p = 3 mixed (518 tiles) 2.10 / 1.91
// ms, 100 x 30 x 30 p = 2 mixed 1.20 / 1.10, 45^3 p = 2 FP64 1.05 / 0.96; 64^3 p =
// 3 mixed (1073 tiles) 3.08 / 3.41, 64^3 p = 2 FP64 (1024) 1.55 / 1.73, mixed 1.60
// / 1.49, 100^3 p = 1 mixed 1.81 / 2.00.  Six entries instead of four: 200 x 200 x
// 3 p = 2 mixed 1.31 / 1.23, 64^3 p = 2 mixed 1.50 / 1.83.
constexpr int kPlaneTiles = 1000;

template <int D, int P, typename V, typename T, int KIND, int MODE>
static hipError_t sspmv_launch(const SpmvGrid &G, const V *sv, const T *x, const T *po, T *pn, T *y, const T *b,
                               double *part, const CGStep &cs, CGState *st, hipStream_t s)
{
    const dim3 grid(sspmv_blocks(G.nfree));
    const size_t lds = (size_t)G.stage.entries * (D == 3 ? 2 : 1) * sizeof(T);
    // 0: entry by entry; 1: a window; 2: stretches of lines, or a window per plane
    const bool split = D == 3 && (int)grid.x <= kSplitTiles;
    const int staged = lds > (split ? kSplitLds : kWindowLds) ? 0 : G.stage.magic || G.stage.plane ? 2 : 1;
    constexpr bool f32 = sizeof(T) == 4;
    constexpr int FEW = D == 2 ? 0 : f32 && P == 2 ? 6 : f32 || P <= 2 ? 4 : 0;
    // 2D: the next tile's stretches are requested where a block has further tiles
    // (2600^2 p = 2 mixed 9.3 / 8.4 ms); below, the registers of it cost a wave per
    // SIMD (600^2 p = 2 mixed 1.04 ms without, 1.12 with them)
    constexpr int MANY = D == 2 ? 1 : f32 && P == 2 ? 4 : 0;
#define GSX_Q(STAGED, Q, PLANES)                                                                                      \
    hipLaunchKernelGGL((k_cg2_spmv<D, P, V, T, KIND, MODE, STAGED, Q, PLANES>), grid, dim3(256 * Q),                  \
                       STAGED ? lds : 0, s, G.nfree, G.f2g, G.sy, G.sz, G.m0, G.m1, sv, x, po, pn, y, b, part, cs,    \
                       st, G.stage)
#define GSX_ST(Q, PLANES)                                                                                             \
    {                                                                                                                 \
        if (staged == 2) GSX_Q(2, Q, PLANES);                                                                         \
        else if (staged) GSX_Q(1, Q, PLANES);                                                                         \
        else GSX_Q(0, Q, 0);                                                                                          \
    }
    if (split) {
        constexpr int Q = D == 3 ? kSplit : 1;
        GSX_ST(Q, FEW)
    } else if (D == 3 ? (int)grid.x <= kPlaneTiles : (G.nfree + 255) / 256 <= kMaxPartials) {
        GSX_ST(1, FEW)
    } else {
        GSX_ST(1, MANY)
    }
#undef GSX_ST
#undef GSX_Q
    return hipGetLastError();
}

#define GSX_SALL(KIND, MODE)                                                                                      \
    GSX_S(2, 1, KIND, MODE) GSX_S(2, 2, KIND, MODE) GSX_S(2, 3, KIND, MODE) GSX_S(2, 4, KIND, MODE)               \
    GSX_S(3, 1, KIND, MODE) GSX_S(3, 2, KIND, MODE) GSX_S(3, 3, KIND, MODE) GSX_S(3, 4, KIND, MODE)
#define GSX_S(D, P, KIND, MODE)                                                                                   \
    if (G.d == D && G.p == P) return sspmv_launch<D, P, SV, ST, KIND, MODE>(G, sv, x, po, pn, y, b, part, cs, st, s);

template <int MODE>
static hipError_t sspmv_f64(const SpmvGrid &G, const double *sv, const double *x, const double *po, double *pn,
                            double *y, const double *b, double *part, const CGStep &cs, CGState *st, hipStream_t s)
{
    using SV = double;
    using ST = double;
    const int w = 2 * G.p + 1, slots = G.d == 3 ? w * w * w : w * w;
    if ((int64_t)G.nfree * slots * 8 <= kMirrorBytes) {
        GSX_SALL(2, MODE)
    } else {
        GSX_SALL(1, MODE)
    }
    return hipErrorInvalidValue;
}

hipError_t launch_sspmv_residual(const SpmvGrid &G, const double *sv, const double *x, double *y, const double *b,
                                 double *part, hipStream_t s)
{
    return sspmv_f64<2>(G, sv, x, nullptr, nullptr, y, b, part, CGStep{}, nullptr, s);
}

hipError_t launch_cg2_spmv_f64(const SpmvGrid &G, const double *sv, const double *z, const double *po, double *pn,
                               double *t, double *part, const CGStep &cs, CGState *st, hipStream_t s)
{
    return sspmv_f64<1>(G, sv, z, po, pn, t, nullptr, part, cs, st, s);
}

hipError_t launch_cg2_spmv_f32(const SpmvGrid &G, const float *sv, const float *x, const float *po, float *pn,
                               float *y, double *part, const CGStep &cs, CGState *st, hipStream_t s)
{
    using SV = float;
    using ST = float;
    const float *b = nullptr;
    GSX_SALL(0, 1)
    return hipErrorInvalidValue;
}
#undef GSX_S
#undef GSX_SALL

hipError_t launch_cg2_check(const CGStep &cs, CGState *st, hipStream_t s)
{
    hipLaunchKernelGGL(k_cg2_check, dim3(1), dim3(256), 0, s, cs, st);
    return hipGetLastError();
}

hipError_t launch_cg2_update_f64(int n, double *x, double *r, const double *p, const double *t,
                                 double *z, const double *diag, double tau, const double *pap,
                                 int npap, double *prr, double *prz, CGState *st, int k, hipStream_t s)
{
    hipLaunchKernelGGL((k_cg2_update<double, double>), dim3(vec_blocks(n)), dim3(kVecThreads), 0, s, n, x, r, p, t, z,
                       diag, tau, pap, npap, prr, prz, st, k);
    return hipGetLastError();
}

hipError_t launch_cg2_update_f32(int n, float *x, float *r, const float *p, const float *t, float *z,
                                 const float *diag, double tau, const double *pap, int npap,
                                 double *prr, double *prz, CGState *st, int k, hipStream_t s)
{
    hipLaunchKernelGGL((k_cg2_update<float, float>), dim3(vec_blocks(n)), dim3(kVecThreads), 0, s, n, x, r, p, t, z,
                       diag, tau, pap, npap, prr, prz, st, k);
    return hipGetLastError();
}

hipError_t launch_cg2_dot_f64(int n, const double *a, const double *b, double *part, const CGState *st,
                              hipStream_t s)
{
    hipLaunchKernelGGL((k_cg2_dot<double>), dim3(vec_blocks(n)), dim3(kVecThreads), 0, s, n, a, b, part, st);
    return hipGetLastError();
}

hipError_t launch_cg2_dot_f32(int n, const float *a, const float *b, double *part, const CGState *st,
                              hipStream_t s)
{
    hipLaunchKernelGGL((k_cg2_dot<float>), dim3(vec_blocks(n)), dim3(kVecThreads), 0, s, n, a, b, part, st);
    return hipGetLastError();
}

hipError_t launch_cg2_precond_f64(int n, const double *r, double *z, const double *diag, double tau, double *prr,
                                  double *prz, hipStream_t s)
{
    hipLaunchKernelGGL((k_cg2_precond<double>), dim3(vec_blocks(n)), dim3(kVecThreads), 0, s, n, r, z, diag, tau, prr,
                       prz);
    return hipGetLastError();
}

hipError_t launch_cg2_precond_f32(int n, const float *r, float *z, const float *diag, double tau, double *prr,
                                  double *prz, hipStream_t s)
{
    hipLaunchKernelGGL((k_cg2_precond<float>), dim3(vec_blocks(n)), dim3(kVecThreads), 0, s, n, r, z, diag, tau, prr,
                       prz);
    return hipGetLastError();
}

hipError_t launch_grid_f64_to_f32(int64_t n, const double *a, float *b, hipStream_t s)
{
    hipLaunchKernelGGL((k_copy_convert<double, float>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, a, b);
    return hipGetLastError();
}

hipError_t launch_accum_grid(int64_t n, double *x, float *xc, hipStream_t s)
{
    hipLaunchKernelGGL(k_accum_grid, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, x, xc);
    return hipGetLastError();
}

}  // namespace gsx
