// Sum-factorised assembly of 2D patches (libgsx, gfx950): the stiffness matrix
// and the load row by row, without element matrices.
//
// Reference: igrad(u,G)*igrad(u,G).tr()*meas(G) [* kappa] and u*ff*meas(G) of
// gsExprAssembler (src/gsAssembler/gsExpressions.h:2737-3890, 946-970), summed
// over the elements and Gauss points of each patch
// (gsExprAssembler.h:553-630, 754-833).
//
// For a tensor-product basis the entry of row i = (ix, iy), column i + o is
//   A(i, i + o) = sum_ab sum_gx X^ab(ix, ox, gx) T_ab(iy, oy, gx),
//   T_ab(iy, oy, gx) = sum_gy D^ab(gx, gy) Y^ab(iy, oy, gy)
// with D^ab = w kappa |det J| (J^-1 J^-T)_ab at the Gauss point and X, Y the
// products of the row's and the column's 1D values (derivatives where the flag
// of that direction is set): the element-by-element sum regrouped by Gauss
// point columns.
//
// k_sf2_rows: a block takes a range of basis rows ix and walks a chunk of iy.
// A thread owns one Gauss point column gx and goes up the elements in y: the
// geometry from control rows contracted once (the last p + 1 in registers), D
// per point, and the sums T for the (p + 1)(p + 2) / 2 pairs (iy, iy + oy) of
// functions alive on the element, in registers.  When element ey is done the
// pairs of row iy = ey are complete: they go to LDS and the block contracts x,
// one thread per (ix, oy).  Only oy >= 0 is formed; rows overlapping into the
// neighbouring block recompute p elements.  No Gauss point data or element
// matrix touches memory: the element matrices of 1 M elements at p = 3 took
// 2.1 GB each way.  Raw rows: [function][oy][ox], lines padded to a multiple
// of four entries, of every basis function of every patch.
// Bound by FP64 arithmetic and LDS reads.  3 x 3 patches of 181^2 elements, p =
// 2: element matrices 494 us + gather from them 874 us before, raw rows 71 us +
// gather 156 us now; one patch of 64^2, p = 2 (latency): 14 + 29 us before, 16 +
// 7.6 us now.
//
// The CSR rows are gathered from the raw rows (entries with oy < 0, or oy = 0
// and ox < 0, from their mirrors, so that the matrix is bitwise symmetric):
// k_sf2_finish for one patch, k_sf2_gather for glued patches.
#include "gsx_common.h"
#include "gsx_kernels.h"
#include "gsx_basis.h"

namespace gsx {

template <int P>
struct Sf2Cfg {
    static constexpr int NB1 = P + 1, W = 2 * P + 1, NS = W * W;
    static constexpr int NL = P + 1;                    // lines oy = 0 .. p
    static constexpr int OXP = (W + 3) / 4 * 4, ROW = NL * OXP;
    static constexpr int EB = 256 / NB1;                // elements per block
    static constexpr int RB = EB - P;                   // rows per block
    static constexpr int CYM = 16;                      // rows iy per chunk, at most
    static_assert(RB * NL <= 256, "one thread per (row, line)");
};

template <int P>
__global__ __launch_bounds__(256) void k_sf2_rows(const PatchDev *__restrict__ patches,
                                                  const int *__restrict__ gpatch,
                                                  const int64_t *__restrict__ bprefix, int ng, int cy, GaussTab gt,
                                                  double *__restrict__ raw, double *__restrict__ rawf,
                                                  double *__restrict__ detmin)
{
    using C = Sf2Cfg<P>;
    constexpr int NB1 = C::NB1, NL = C::NL, OXP = C::OXP, ROW = C::ROW, EB = C::EB, RB = C::RB;
    constexpr int EYM = C::CYM + P, NPAIR = NB1 * (NB1 + 1) / 2;
    __shared__ double sX[2][NB1][NB1][EB];          // [derivative][q][m][e]
    __shared__ double sY[EYM * NB1][2 * NB1 + 1];   // values, derivatives, weight
    __shared__ double sT[NL][4][NB1][EB], sF[NB1][EB];
    __shared__ double sMin[4];
    int lo = 0, hi = ng - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (bprefix[mid] <= (int64_t)blockIdx.x) lo = mid; else hi = mid - 1;
    }
    const PatchDev &pd = patches[gpatch[lo]];
    const int lb = (int)(blockIdx.x - bprefix[lo]);
    const int nbx = pd.nb[0], nby = pd.nb[1], nelx = pd.nel[0], nely = pd.nel[1];
    const int nxb = (nbx + RB - 1) / RB;
    const int x0 = (lb % nxb) * RB, x1 = min(x0 + RB, nbx);
    const int c0 = (lb / nxb) * cy, c1 = min(c0 + cy, nby);
    const int exa = max(0, x0 - P), exb = min(nelx, x1);   // elements [exa, exb)
    const int ya = max(0, c0 - P), yb = min(nely, c1);
    const int t = threadIdx.x;
    // 1D tables: the y elements of the chunk, the block's columns
    for (int k = t; k < (yb - ya) * NB1; k += 256) {
        const int span = P + ya + k / NB1, q = k % NB1;
        const double *U = pd.knots[1];
        const double a = U[span], b = U[span + 1], h = (b - a) / 2.0;
        double N[NB1], dN[NB1];
        deboor_ders<P>(U, span, h * (gt.x[NB1][q] + 1.0) + a, N, dN);
#pragma unroll
        for (int m = 0; m < NB1; ++m) {
            sY[k][m] = N[m];
            sY[k][NB1 + m] = dN[m];
        }
        sY[k][2 * NB1] = (0.0 == h ? 0.5 : h) * gt.w[NB1][q];
    }
    const int le = t / NB1, q = t % NB1, ex = min(exa + le, nelx - 1);
    const bool act = le < EB && exa + le < exb;
    double vx[NB1], dx[NB1], wx;
    {
        const int span = P + ex;
        const double *U = pd.knots[0];
        const double a = U[span], b = U[span + 1], h = (b - a) / 2.0;
        deboor_ders<P>(U, span, h * (gt.x[NB1][q] + 1.0) + a, vx, dx);
        wx = (0.0 == h ? 0.5 : h) * gt.w[NB1][q];
        if (le < EB)
#pragma unroll
            for (int m = 0; m < NB1; ++m) {
                sX[0][q][m][le] = vx[m];
                sX[1][q][m][le] = dx[m];
            }
    }
    __syncthreads();
    // contracted control rows: value and x derivative of both coordinates,
    // relative to a control point of the column, so that the Jacobian's
    // differences cancel over the chunk's extent and not over the coordinates
    double hv[NB1][2], hx[NB1][2];
    const double2 ref = reinterpret_cast<const double2 *>(pd.ctrl)[ex + (int64_t)nbx * ya];
    auto load = [&](int y, int m) {
        const double2 *c = reinterpret_cast<const double2 *>(pd.ctrl) + ex + (int64_t)nbx * y;
        double a0 = 0.0, a1 = 0.0, b0 = 0.0, b1 = 0.0;
#pragma unroll
        for (int b = 0; b < NB1; ++b) {
            const double px = c[b].x - ref.x, py = c[b].y - ref.y;
            a0 += px * vx[b];
            a1 += py * vx[b];
            b0 += px * dx[b];
            b1 += py * dx[b];
        }
        hv[m][0] = a0;
        hv[m][1] = a1;
        hx[m][0] = b0;
        hx[m][1] = b1;
    };
    // pair (m1, m2), m1 <= m2, of the element's functions
    auto pair = [](int m1, int m2) { return m1 * NB1 - m1 * (m1 - 1) / 2 + (m2 - m1); };
    double acc[NPAIR][4], accf[NB1], dmin = 1e300;
#pragma unroll
    for (int k = 0; k < NPAIR; ++k) acc[k][0] = acc[k][1] = acc[k][2] = acc[k][3] = 0.0;
#pragma unroll
    for (int m = 0; m < NB1; ++m) accf[m] = 0.0;
#pragma unroll
    for (int m = 1; m < NB1; ++m) load(ya + m - 1, m);
    for (int iy = ya; iy < c1; ++iy) {
        if (iy < nely) {
#pragma unroll
            for (int m = 0; m < P; ++m)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    hv[m][c] = hv[m + 1][c];
                    hx[m][c] = hx[m + 1][c];
                }
            load(iy + P, P);
            const int64_t el = ex + (int64_t)nelx * iy;
            const double kap = pd.kappa ? pd.kappa[el] : 1.0;
#pragma unroll 1
            for (int qy = 0; qy < NB1; ++qy) {
                const double *y = sY[(iy - ya) * NB1 + qy];
                double bv[NB1], bd[NB1];
                double X[2] = {ref.x, ref.y}, J00 = 0.0, J01 = 0.0, J10 = 0.0, J11 = 0.0;
#pragma unroll
                for (int m = 0; m < NB1; ++m) {
                    bv[m] = y[m];
                    bd[m] = y[NB1 + m];
                    X[0] += hv[m][0] * bv[m];
                    X[1] += hv[m][1] * bv[m];
                    J00 += hx[m][0] * bv[m];
                    J10 += hx[m][1] * bv[m];
                    J01 += hv[m][0] * bd[m];
                    J11 += hv[m][1] * bd[m];
                }
                const double det = J00 * J11 - J01 * J10, w = wx * y[2 * NB1], ad = fabs(det);
                if (act) dmin = fmin(dmin, pd.orient * det);
                const double S = w * (source_value(pd.fkind, 2, X, pd.felem, el) * ad);
                // J^-1 = cof / det: D = w kappa / |det| cof cof^T
                const double sc = w * kap / ad;
                const double d00 = sc * (J11 * J11 + J01 * J01), d01 = -sc * (J11 * J10 + J01 * J00),
                             d11 = sc * (J10 * J10 + J00 * J00);
#pragma unroll
                for (int m1 = 0; m1 < NB1; ++m1) {
                    accf[m1] += bv[m1] * S;
                    const double u00 = d00 * bv[m1], u01 = d01 * bv[m1], u10 = d01 * bd[m1], u11 = d11 * bd[m1];
#pragma unroll
                    for (int m2 = m1; m2 < NB1; ++m2) {
                        double *a = acc[pair(m1, m2)];
                        a[0] += u00 * bv[m2];
                        a[1] += u01 * bd[m2];
                        a[2] += u10 * bv[m2];
                        a[3] += u11 * bd[m2];
                    }
                }
            }
        }
        if (iy >= c0) {
            // row iy is complete: its pairs to LDS, then the x contraction
            if (le < EB) {
#pragma unroll
                for (int oy = 0; oy < NL; ++oy)
#pragma unroll
                    for (int ab = 0; ab < 4; ++ab) sT[oy][ab][q][le] = acc[pair(0, oy)][ab];
                sF[q][le] = accf[0];
            }
            __syncthreads();
            const int rx = t % RB, oy = t / RB, ix = x0 + rx;
            if (oy < NL && ix < x1) {
                double out[OXP];
#pragma unroll
                for (int k = 0; k < OXP; ++k) out[k] = 0.0;
                double f = 0.0;
#pragma unroll
                for (int m1 = P; m1 >= 0; --m1) {   // elements ascending
                    const int e = ix - m1 - exa;
                    if (ix - m1 < 0 || ix - m1 >= nelx) continue;
#pragma unroll 1
                    for (int qx = 0; qx < NB1; ++qx) {
                        const double v1 = sX[0][qx][m1][e], d1 = sX[1][qx][m1][e];
                        const double u0 = d1 * sT[oy][0][qx][e] + v1 * sT[oy][2][qx][e];
                        const double u1 = d1 * sT[oy][1][qx][e] + v1 * sT[oy][3][qx][e];
#pragma unroll
                        for (int m2 = 0; m2 < NB1; ++m2)
                            out[m2 - m1 + P] += sX[1][qx][m2][e] * u0 + sX[0][qx][m2][e] * u1;
                        if (oy == 0) f += v1 * sF[qx][e];
                    }
                }
                const int64_t row = ix + (int64_t)nbx * iy;
                double2 *o = reinterpret_cast<double2 *>(raw + pd.r_off + row * ROW + oy * OXP);
#pragma unroll
                for (int k = 0; k < OXP / 2; ++k) o[k] = double2{out[2 * k], out[2 * k + 1]};
                if (oy == 0) rawf[pd.b_off + row] = f;
            }
            __syncthreads();
        }
#pragma unroll
        for (int m1 = 0; m1 < NB1; ++m1) {
#pragma unroll
            for (int m2 = m1; m2 < NB1; ++m2)
#pragma unroll
                for (int ab = 0; ab < 4; ++ab)
                    acc[pair(m1, m2)][ab] = m2 < P ? acc[pair(m1 + 1, m2 + 1 < NB1 ? m2 + 1 : m2)][ab] : 0.0;
            accf[m1] = m1 < P ? accf[m1 < P ? m1 + 1 : m1] : 0.0;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) dmin = fmin(dmin, __shfl_xor(dmin, off, 64));
    if ((t & 63) == 0) sMin[t >> 6] = dmin;
    __syncthreads();
    if (t == 0) detmin[blockIdx.x] = fmin(fmin(sMin[0], sMin[1]), fmin(sMin[2], sMin[3]));
}

// entry of patch function l (of a patch at raw) at offset (ox, oy)
template <int P>
__device__ inline double sf2_entry(const double *__restrict__ raw, int64_t l, int nbx, int ox, int oy)
{
    using C = Sf2Cfg<P>;
    if (oy > 0 || (oy == 0 && ox >= 0)) return raw[l * C::ROW + oy * C::OXP + ox + P];
    return raw[(l + ox + (int64_t)nbx * oy) * C::ROW - oy * C::OXP + P - ox];
}

// One patch whose free functions form the box: blocks of up to R rows of an
// x-line through LDS, as k_sf_finish3d does in 3D.
template <int P>
__global__ __launch_bounds__(256) void k_sf2_finish(SfBox bx, int nfree, const int *__restrict__ rowptr,
                                                    const double *__restrict__ raw, const double *__restrict__ rawf,
                                                    double *__restrict__ s64, float *__restrict__ s32,
                                                    double *__restrict__ val, double *__restrict__ rhs,
                                                    const int *__restrict__ dofs, const double *__restrict__ fixed,
                                                    int *__restrict__ err)
{
    using C = Sf2Cfg<P>;
    constexpr int W = C::W, NS = C::NS, CE = NS / 2, NH = stencil_half(NS), R = 32, LD = R + 1;
    __shared__ double L[NS * LD];
    const int t = threadIdx.x;
    const int nseg = (bx.m[0] + R - 1) / R, seg = blockIdx.x % nseg, jy = blockIdx.x / nseg;
    const int j0 = (int)((int64_t)bx.m[0] * seg / nseg), nr = (int)((int64_t)bx.m[0] * (seg + 1) / nseg) - j0;
    const int r0 = j0 + bx.m[0] * jy, ix0 = bx.flo[0] + j0, iy = bx.flo[1] + jy, nbx = bx.nb[0];
    auto is_free = [&](int x, int y) { return x >= bx.flo[0] && x <= bx.fhi[0] && y >= bx.flo[1] && y <= bx.fhi[1]; };
    for (int k = t; k < NS * LD; k += 256) L[k] = 0.0;
    __syncthreads();
    // own lines, then the lower entries from their mirrors (row jx of line
    // iy - oy, upper offset ox: the entry of row jx + ox at (-ox, -oy))
    for (int k = t; k < nr * C::ROW; k += 256) {
        const int j = k % C::OXP, oy = (k / C::OXP) % C::NL, rr = k / C::ROW;
        if (j < W && (oy > 0 || j >= P) && is_free(ix0 + rr + j - P, iy + oy))
            L[((oy + P) * W + j) * LD + rr] = raw[(ix0 + (int64_t)nbx * iy) * C::ROW + k];
    }
    constexpr int RS = R + 2 * P;
    for (int k = t; k < C::NL * RS * C::OXP; k += 256) {
        const int j = k % C::OXP, rs = (k / C::OXP) % RS, oy = k / (C::OXP * RS);
        const int ox = j - P, jx = ix0 - P + rs, rr = jx + ox - ix0;
        if (j >= W || rr < 0 || rr >= nr || (oy == 0 && ox <= 0) || !is_free(jx, iy - oy)) continue;
        L[((P - oy) * W + P - ox) * LD + rr] =
            raw[(jx + (int64_t)nbx * (iy - oy)) * C::ROW + oy * C::OXP + j];
    }
    __syncthreads();
    const int ylo = max(-P, bx.flo[1] - iy), ny = min(P, bx.fhi[1] - iy) - ylo + 1;
    for (int k = t; k < nr * NS; k += 256) {
        const int rr = k / NS, sl = k % NS, ox = sl % W - P, oy = sl / W - P - ylo;
        const int lo = max(-P, bx.flo[0] - ix0 - rr), nx = min(P, bx.fhi[0] - ix0 - rr) - lo + 1;
        const int base = rowptr[r0 + rr];
        if (nx * ny != rowptr[r0 + rr + 1] - base) {
            if (sl == 0) atomicOr(err, 1);
        } else if (oy >= 0 && oy < ny && ox >= lo && ox < lo + nx) {
            val[base + oy * nx + ox - lo] = L[sl * LD + rr];
        }
    }
    if (s64 && t % R < nr)
        for (int sl = t / R; sl < NS; sl += 256 / R) {
            const double v = L[sl * LD + t % R];
            s64[stencil_index(sl, r0 + t % R, NS)] = v;
            if (s32 && sl >= CE) s32[stencil_index(sl - CE, r0 + t % R, NH)] = (float)v;
        }
    if (t < nr) {
        const int64_t l = ix0 + t + (int64_t)nbx * iy;
        double f = rawf[l];
        if (fixed)
            for (int sl = 0; sl < NS; ++sl) {
                const int ox = sl % W - P, oy = sl / W - P, jx = ix0 + t + ox, ky = iy + oy;
                if (jx < 0 || jx >= nbx || ky < 0 || ky >= bx.nb[1] || is_free(jx, ky)) continue;
                f -= sf2_entry<P>(raw, l, nbx, ox, oy) * fixed[dofs[jx + (int64_t)nbx * ky] - nfree];
            }
        rhs[r0 + t] = f;
    }
}

// Glued patches: a wavefront per CSR row.  The row's window of every
// occurrence (patch, function) is read from that patch's raw rows, a lane per
// stencil slot.  A row of one occurrence whose columns ascend along the window
// (all but the neighbours of interfaces) places entry k at its rank among the
// free lanes; other rows find the column by bisection in LDS and sum their
// occurrences there in patch order.
template <int P, int MAXROW>
__global__ __launch_bounds__(256) void k_sf2_gather(const PatchDev *__restrict__ patches,
                                                    const int *__restrict__ occ_ptr,
                                                    const int *__restrict__ occ_patch,
                                                    const int64_t *__restrict__ occ_local, int nfree,
                                                    const int *__restrict__ rowptr, const int *__restrict__ col,
                                                    const double *__restrict__ raw, const double *__restrict__ rawf,
                                                    double *__restrict__ val, double *__restrict__ rhs,
                                                    const double *__restrict__ fixed, int *__restrict__ err)
{
    using C = Sf2Cfg<P>;
    constexpr int W = C::W, NS = C::NS, NP = (NS + 63) / 64;
    __shared__ int sCol[4][MAXROW];
    __shared__ double sAcc[4][MAXROW];
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int r = blockIdx.x * 4 + w;
    if (r >= nfree) return;
    const int rb = rowptr[r], len = rowptr[r + 1] - rb;
    const int o0 = occ_ptr[r], o1 = occ_ptr[r + 1];
    if (patches[occ_patch[o0]].p[0] != P) return;   // a row of another degree's patches
    double racc = 0.0, elim = 0.0;
    bool placed = false;
    for (int o = o0; o < o1; ++o) {
        const PatchDev &pd = patches[occ_patch[o]];
        const int nbx = pd.nb[0], nby = pd.nb[1];
        const int64_t l = occ_local[o];
        const int lx = (int)(l % nbx), ly = (int)(l / nbx);
        const double *base = raw + pd.r_off;
        int g[NP];
        double v[NP];
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int sl = lane + 64 * u, ox = sl % W - P, oy = sl / W - P, jx = lx + ox, jy = ly + oy;
            g[u] = -1;
            v[u] = 0.0;
            if (sl < NS && jx >= 0 && jx < nbx && jy >= 0 && jy < nby) {
                const int d = pd.dofs[l + ox + (int64_t)nbx * oy];
                v[u] = sf2_entry<P>(base, l, nbx, ox, oy);
                if (d < nfree) g[u] = d;
                else if (fixed) elim += v[u] * fixed[d - nfree];
            }
        }
        if (rhs) racc += rawf[pd.b_off + l];
        if (o1 - o0 == 1) {
            int rank[NP], done = 0, last = -1;
            bool up = true;
#pragma unroll
            for (int u = 0; u < NP; ++u) {
                const unsigned long long m = __ballot(g[u] >= 0), below = m & ((1ull << lane) - 1);
                rank[u] = done + __popcll(below);
                const int prev = __shfl(g[u], below ? 63 - __clzll(below) : 0, 64);
                up = up && (g[u] < 0 || g[u] > (below ? prev : last));
                if (m) last = __shfl(g[u], 63 - __clzll(m), 64);
                done += __popcll(m);
            }
            if (__all(up) && done == len) {
                placed = true;
#pragma unroll
                for (int u = 0; u < NP; ++u)
                    if (g[u] >= 0) val[rb + rank[u]] = v[u];
                break;
            }
        }
        if (o == o0) {
            for (int k = lane; k < len; k += kWave) {
                sCol[w][k] = col[rb + k];
                sAcc[w][k] = 0.0;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            if (g[u] < 0) continue;
            int a = 0, b = len - 1;
            while (a < b) {
                const int mid = (a + b) >> 1;
                if (sCol[w][mid] < g[u]) a = mid + 1; else b = mid;
            }
            if (len == 0 || sCol[w][a] != g[u]) atomicOr(err, 1);
            else sAcc[w][a] += v[u];   // the window's columns are distinct
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (!placed && o1 > o0)
        for (int k = lane; k < len; k += kWave) val[rb + k] = sAcc[w][k];
    if (rhs) {
        if (fixed)
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) elim += __shfl_xor(elim, off, 64);
        if (lane == 0) rhs[r] = racc - elim;
    }
}

bool sf2_supported(int p) { return p >= 2 && p <= 4; }

// Galerkin product of raw rows under bisection, the coarse raw rows from the
// fine ones:  Kc(I, J) = sum_ij T(i, I) K(i, j) T(j, J),  T a product of the
// directions' transfers.  The coarse function I of a direction is a sum of the
// p + 2 fine ones 2 I - p .. 2 I + 1, T[I][k] their weights (zero outside).
// k_sf2_galerkin_x contracts x, a thread per (Ix, line (iy, iy + oy)), oy >= 0;
// k_sf2_galerkin_y contracts y, a thread per coarse entry, lines with oy < 0
// read as the mirrors of stored ones (both indices swapped).  Bound by the
// bytes of the raw rows and of the half-contracted lines.  16 patches of 256^2
// elements, p = 3: x 268 us (element matrices formed 3.7 ms, coarsened 1.9 ms);
// with the raw rows' own 0.45 ms and gathers of 0.7 ms instead of 5.2 ms the
// hierarchy's set-up and solve takes 33 ms instead of 44.
template <int P>
__global__ __launch_bounds__(256) void k_sf2_galerkin_x(const PatchDev *__restrict__ cpatches,
                                                        const PatchDev *__restrict__ fpatches,
                                                        const Sf2Coarse *__restrict__ meta, int ng,
                                                        const double *__restrict__ T, const double *__restrict__ raw,
                                                        double *__restrict__ mid)
{
    using C = Sf2Cfg<P>;
    constexpr int W = C::W, NT = P + 2;
    int lo = 0, hi = ng - 1;
    while (lo < hi) {
        const int m = (lo + hi + 1) >> 1;
        if (meta[m].bx <= (int64_t)blockIdx.x) lo = m; else hi = m - 1;
    }
    const Sf2Coarse mt = meta[lo];
    const PatchDev &fp = fpatches[mt.patch], &cp = cpatches[mt.patch];
    const int nbx = fp.nb[0], nby = fp.nb[1], cnx = cp.nb[0];
    const int64_t u = ((int64_t)blockIdx.x - mt.bx) * 256 + threadIdx.x;
    const int Ix = (int)(u % cnx), oy = (int)((u / cnx) % C::NL), iy = (int)(u / ((int64_t)cnx * C::NL));
    if (iy + oy >= nby) return;   // also the threads beyond the last line
    const double *Tx = T + mt.tx;
    double v[NT][W], tk[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const int ix = 2 * Ix - P + k;
        const bool in = ix >= 0 && ix < nbx;
        tk[k] = Tx[Ix * NT + k];
        const double *row = raw + fp.r_off + ((in ? ix : 0) + (int64_t)nbx * iy) * C::ROW + oy * C::OXP;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const int jx = ix + j - P;
            v[k][j] = in && jx >= 0 && jx < nbx ? row[j] : 0.0;
        }
    }
    double *out = mid + mt.m_off + ((int64_t)(iy * C::NL + oy) * cnx + Ix) * C::OXP;
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const int J = Ix + j - P;
        if (J < 0 || J >= cnx) continue;
        double tl[NT], sum = 0.0;
#pragma unroll
        for (int l = 0; l < NT; ++l) tl[l] = Tx[J * NT + l];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            double a = 0.0;
#pragma unroll
            for (int l = 0; l < NT; ++l) {
                constexpr int N = W;
                const int o = 2 * (j - P) + l - k + P;   // jx - ix + P
                if (o >= 0 && o < N) a += tl[l] * v[k][o];
            }
            sum += tk[k] * a;
        }
        out[j] = sum;
    }
}

template <int P>
__global__ __launch_bounds__(256) void k_sf2_galerkin_y(const PatchDev *__restrict__ cpatches,
                                                        const PatchDev *__restrict__ fpatches,
                                                        const Sf2Coarse *__restrict__ meta, int ng,
                                                        const double *__restrict__ T, const double *__restrict__ mid,
                                                        double *__restrict__ craw)
{
    using C = Sf2Cfg<P>;
    constexpr int W = C::W, NT = P + 2;
    int lo = 0, hi = ng - 1;
    while (lo < hi) {
        const int m = (lo + hi + 1) >> 1;
        if (meta[m].by <= (int64_t)blockIdx.x) lo = m; else hi = m - 1;
    }
    const Sf2Coarse mt = meta[lo];
    const PatchDev &fp = fpatches[mt.patch], &cp = cpatches[mt.patch];
    const int nby = fp.nb[1], cnx = cp.nb[0], cny = cp.nb[1];
    const int64_t u = ((int64_t)blockIdx.x - mt.by) * 256 + threadIdx.x;
    const int j = (int)(u % C::OXP), Ix = (int)((u / C::OXP) % cnx);
    const int64_t rest = u / ((int64_t)C::OXP * cnx);
    const int OY = (int)(rest % C::NL), Iy = (int)(rest / C::NL);
    const int Jx = Ix + j - P, Jy = Iy + OY;
    if (j >= W || Jx < 0 || Jx >= cnx || Jy >= cny) return;
    const double *Ty = T + mt.ty, *M = mid + mt.m_off;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const int iy = 2 * Iy - P + k;
        if (iy < 0 || iy >= nby) continue;
        double a = 0.0;
#pragma unroll
        for (int l = 0; l < NT; ++l) {
            const int jy = 2 * Jy - P + l, o = jy - iy;
            if (o < -P || o > P || jy < 0 || jy >= nby) continue;
            const double m = o >= 0 ? M[((int64_t)(iy * C::NL + o) * cnx + Ix) * C::OXP + j]
                                    : M[((int64_t)(jy * C::NL - o) * cnx + Jx) * C::OXP + 2 * P - j];
            a += Ty[Jy * NT + l] * m;
        }
        sum += Ty[Iy * NT + k] * a;
    }
    craw[cp.r_off + (Ix + (int64_t)cnx * Iy) * C::ROW + OY * C::OXP + j] = sum;
}

// doubles of the half-contracted lines, and blocks of the two kernels
void sf2_galerkin_sizes(int p, const int *fnb, const int *cnb, int64_t *mid, int64_t *bx, int64_t *by)
{
    const int64_t nl = p + 1, oxp = (2 * p + 1 + 3) / 4 * 4;
    *mid = (int64_t)fnb[1] * nl * cnb[0] * oxp;
    *bx = ((int64_t)fnb[1] * nl * cnb[0] + 255) / 256;
    *by = ((int64_t)cnb[1] * nl * cnb[0] * oxp + 255) / 256;
}

hipError_t launch_sf2_galerkin(int p, const PatchDev *cpatches, const PatchDev *fpatches, const Sf2Coarse *meta,
                               int ng, int64_t nbx, int64_t nby, const double *T, const double *raw, double *mid,
                               double *craw, hipStream_t s)
{
#define GSX_G(P)                                                                                                      \
    if (p == P) {                                                                                                     \
        hipLaunchKernelGGL((k_sf2_galerkin_x<P>), dim3((unsigned)nbx), dim3(256), 0, s, cpatches, fpatches, meta, ng, \
                           T, raw, mid);                                                                              \
        hipLaunchKernelGGL((k_sf2_galerkin_y<P>), dim3((unsigned)nby), dim3(256), 0, s, cpatches, fpatches, meta, ng, \
                           T, mid, craw);                                                                             \
        return hipGetLastError();                                                                                     \
    }
    GSX_G(2) GSX_G(3) GSX_G(4)
#undef GSX_G
    return hipErrorInvalidValue;
}

int64_t sf2_raw_doubles(int p, int64_t nbasis)
{
    return nbasis * (p == 2 ? Sf2Cfg<2>::ROW : p == 3 ? Sf2Cfg<3>::ROW : Sf2Cfg<4>::ROW);
}

int64_t sf2_blocks(int p, const int *nb, int cy)
{
    const int rb = p == 2 ? Sf2Cfg<2>::RB : p == 3 ? Sf2Cfg<3>::RB : Sf2Cfg<4>::RB;
    return (int64_t)((nb[0] + rb - 1) / rb) * ((nb[1] + cy - 1) / cy);
}

hipError_t launch_sf2_rows(int p, const PatchDev *patches, const int *gpatch, const int64_t *bprefix, int ng,
                           int64_t nblocks, int cy, const GaussTab &gt, double *raw, double *rawf, double *detmin,
                           hipStream_t s)
{
    if (nblocks <= 0) return hipSuccess;
    if (cy < 1 || cy > Sf2Cfg<3>::CYM) return hipErrorInvalidValue;
    const dim3 grid((unsigned)nblocks), blk(256);
    switch (p) {
    case 2: hipLaunchKernelGGL((k_sf2_rows<2>), grid, blk, 0, s, patches, gpatch, bprefix, ng, cy, gt, raw, rawf, detmin); break;
    case 3: hipLaunchKernelGGL((k_sf2_rows<3>), grid, blk, 0, s, patches, gpatch, bprefix, ng, cy, gt, raw, rawf, detmin); break;
    case 4: hipLaunchKernelGGL((k_sf2_rows<4>), grid, blk, 0, s, patches, gpatch, bprefix, ng, cy, gt, raw, rawf, detmin); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_sf2_finish(int p, const SfBox &bx, int nfree, const int *rowptr, const double *raw,
                             const double *rawf, double *s64, float *s32, double *val, double *rhs, const int *dofs,
                             const double *fixed, int *err, hipStream_t s)
{
    if (nfree <= 0) return hipSuccess;
    const dim3 grid((unsigned)((int64_t)((bx.m[0] + 31) / 32) * bx.m[1])), blk(256);
    switch (p) {
    case 2: hipLaunchKernelGGL((k_sf2_finish<2>), grid, blk, 0, s, bx, nfree, rowptr, raw, rawf, s64, s32, val, rhs, dofs, fixed, err); break;
    case 3: hipLaunchKernelGGL((k_sf2_finish<3>), grid, blk, 0, s, bx, nfree, rowptr, raw, rawf, s64, s32, val, rhs, dofs, fixed, err); break;
    case 4: hipLaunchKernelGGL((k_sf2_finish<4>), grid, blk, 0, s, bx, nfree, rowptr, raw, rawf, s64, s32, val, rhs, dofs, fixed, err); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int P>
static hipError_t sf2_gather(const PatchDev *patches, const int *occ_ptr, const int *occ_patch,
                             const int64_t *occ_local, int nfree, const int *rowptr, const int *col,
                             const double *raw, const double *rawf, double *val, double *rhs, int maxrow,
                             const double *fixed, int *err, hipStream_t s)
{
    const dim3 grid((nfree + 3) / 4), blk(256);
    switch (gather_maxrow_bucket(maxrow)) {
    case 128: hipLaunchKernelGGL((k_sf2_gather<P, 128>), grid, blk, 0, s, patches, occ_ptr, occ_patch, occ_local, nfree, rowptr, col, raw, rawf, val, rhs, fixed, err); break;
    case 512: hipLaunchKernelGGL((k_sf2_gather<P, 512>), grid, blk, 0, s, patches, occ_ptr, occ_patch, occ_local, nfree, rowptr, col, raw, rawf, val, rhs, fixed, err); break;
    case 1024: hipLaunchKernelGGL((k_sf2_gather<P, 1024>), grid, blk, 0, s, patches, occ_ptr, occ_patch, occ_local, nfree, rowptr, col, raw, rawf, val, rhs, fixed, err); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_sf2_gather(int p, const PatchDev *patches, const int *occ_ptr, const int *occ_patch,
                             const int64_t *occ_local, int nfree, const int *rowptr, const int *col,
                             const double *raw, const double *rawf, double *val, double *rhs, int maxrow,
                             const double *fixed, int *err, hipStream_t s)
{
    if (nfree <= 0) return hipSuccess;
    switch (p) {
    case 2: return sf2_gather<2>(patches, occ_ptr, occ_patch, occ_local, nfree, rowptr, col, raw, rawf, val, rhs, maxrow, fixed, err, s);
    case 3: return sf2_gather<3>(patches, occ_ptr, occ_patch, occ_local, nfree, rowptr, col, raw, rawf, val, rhs, maxrow, fixed, err, s);
    case 4: return sf2_gather<4>(patches, occ_ptr, occ_patch, occ_local, nfree, rowptr, col, raw, rawf, val, rhs, maxrow, fixed, err, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace gsx
