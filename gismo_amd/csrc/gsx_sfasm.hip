// Sum-factorised assembly of single 3D patches (libgsx, gfx950): the
// stiffness matrix row by row, without element matrices.
//
// Reference: the bilinear form igrad(u,G)*igrad(u,G).tr()*meas(G) [* kappa]
// of gsExprAssembler (src/gsAssembler/gsExpressions.h:2737-3890) summed over
// the elements and Gauss points of the patch (gsExprAssembler.h:754-833),
// and the load vector u*ff*meas(G) (gsExpressions.h:946-970) pushed into the
// rhs (gsExprAssembler.h:553-630).
//
// For a tensor-product basis the entry of row i = (ix, iy, iz) and column
// j = i + o is
//   A(i, j) = sum_ab sum_g D^ab(g) X^ab(ix, ox, gx) Y^ab(iy, oy, gy) Z^ab(iz, oz, gz)
// where g = (gx, gy, gz) runs over the Gauss points of the patch (g_k =
// e_k (p+1) + q_k), D^ab(g) = w_g kappa_e |det J_g| (J^-1 J^-T)_ab, and
// X^ab(i, o, g) = B^[a==0](i, g) B^[b==0](i+o, g) with B^0 the 1D basis value
// and B^1 its derivative (Y, Z likewise for directions 1, 2).  This is the
// element-by-element sum grad(N_i) D grad(N_j) regrouped: the same terms,
// summed point column by point column instead of element by element.
//
// A block owns a 2 x 2 tile of basis rows in (y, z) and walks the elements
// along x.  Per Gauss point column gx it computes the geometry of its (y, z)
// support by sum factorisation over the control points, then D, then
// contracts z, then y (folding the nine (a, b) pairs into the four classes
// of their x flags), then x into the accumulators of the p + 1 rows
// ix = e .. e + p that element e touches.  Row e is complete after element e
// and leaves the registers.  Only the upper half of the stencil (o >= 0
// lexicographically in (z, y, x)) is accumulated, into raw rows (SfRaw) of all
// basis functions, eliminated ones too: k_sf_finish3d takes the lower half of a
// free row from the raw rows that mirror it, so the FP64 stencil is bitwise
// symmetric.
#include "gsx_common.h"
#include "gsx_kernels.h"
#include "gsx_basis.h"

namespace gsx {

constexpr int kGeoChunk = 8;   // elements along z of one k_geo3d block, at most

template <int P>
struct SfCfg {
    static constexpr int NB1 = P + 1, W = 2 * P + 1, NS = W * W * W;
    static constexpr int TY = 2, TZ = 2, NT = TY * TZ;
    static constexpr int NEY = TY + P, NGY = NEY * NB1, NCY = NEY + P;   // y support: elements, points, ctrl
    static constexpr int NEZ = TZ + P, NGZ = NEZ * NB1, NCZ = NEZ + P;
    static constexpr int NYZ = W * P + P + 1;          // upper (oy, oz) pairs: oz > 0, or oz = 0 and oy >= 0
    static constexpr int KPR = (NYZ - 1) * W + NB1;    // upper (oy, oz, ox) per row
    static constexpr int NCOMBO = NT * KPR;
    static constexpr int CPT = (NCOMBO + 255) / 256;   // accumulator combos per thread
};

// Raw rows: lines of OXP entries (ox + p = 0 .. 2p, padded)
template <int P>
struct SfRaw {
    static constexpr int W = 2 * P + 1, NYZ = W * P + P + 1, OXP = (W + 3) / 4 * 4, ROW = NYZ * OXP;
    // line of (oy, oz) with oz > 0, or oz = 0 and oy >= 0 (sf_pair's order)
    static __device__ inline int line(int oy, int oz) { return oz == 0 ? oy : P + 1 + (oz - 1) * W + oy + P; }
};

// (oy, oz) of upper pair u: u <= P: (u, 0); else oz = 1 + (u - P - 1) / W,
// oy = (u - P - 1) % W - P.
template <int P>
__device__ inline void sf_pair(int u, int &oy, int &oz)
{
    constexpr int W = 2 * P + 1;
    if (u <= P) {
        oy = u;
        oz = 0;
    } else {
        oz = 1 + (u - P - 1) / W;
        oy = (u - P - 1) % W - P;
    }
}

// 1D tables of the patch's Gauss points, per direction k at offset off_k:
// [g][m] values, then [g][m] derivatives (G_k x (p+1) each), then [g]
// mapped weights, for g = e (p+1) + q (the quantities of basis_tables).
template <int P>
__global__ void k_sf_tables(const PatchDev *__restrict__ patches, GaussTab gt, double *__restrict__ tab, int g0,
                            int g1, int g2)
{
    constexpr int NB1 = P + 1;
    const PatchDev &pd = patches[0];
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int G[3] = {g0, g1, g2};
    int k = 0;
    int64_t off = 0;
    while (k < 3 && t >= G[k]) {
        off += (int64_t)G[k] * (2 * NB1 + 1);
        t -= G[k];
        ++k;
    }
    if (k >= 3) return;
    const int e = t / NB1, q = t % NB1;
    const double *U = pd.knots[k];
    const int span = P + e;
    const double a = U[span], b = U[span + 1];
    const double h = (b - a) / 2.0;
    const double u = h * (gt.x[NB1][q] + 1.0) + a;
    double N[NB1], dN[NB1];
    deboor_ders<P>(U, span, u, N, dN);
#pragma unroll
    for (int m = 0; m < NB1; ++m) {
        tab[off + (int64_t)t * NB1 + m] = N[m];
        tab[off + (int64_t)G[k] * NB1 + (int64_t)t * NB1 + m] = dN[m];
    }
    tab[off + 2 * (int64_t)G[k] * NB1 + t] = (0.0 == h ? 0.5 : h) * gt.w[NB1][q];
}

template <int P>
__global__ __launch_bounds__(256) void k_sfasm3d(const PatchDev *__restrict__ patches,
                                                 const double *__restrict__ tab, SfBox bx,
                                                 double *__restrict__ raw)
{
    using C = SfCfg<P>;
    constexpr int NB1 = C::NB1, W = C::W, TY = C::TY, TZ = C::TZ, NT = C::NT;
    constexpr int NGY = C::NGY, NGZ = C::NGZ, NCY = C::NCY, NCZ = C::NCZ, NYZ = C::NYZ, KPR = C::KPR;
    constexpr int NCOMBO = C::NCOMBO, CPT = C::CPT;
    __shared__ double sVy[NGY][NB1], sDy[NGY][NB1], sWy[NGY];
    __shared__ double sVz[NGZ][NB1], sDz[NGZ][NB1], sWz[NGZ];
    __shared__ double sVx[NB1][NB1], sDx[NB1][NB1], sWx[NB1];
    __shared__ double sC[NB1][NCZ][NCY][3];
    __shared__ double sK[C::NEZ][C::NEY];
    __shared__ double sGX[NCZ][NCY][6];
    __shared__ double sGY[NCZ][NGY][9];
    __shared__ double sD[6][NGZ][NGY];
    __shared__ double sT1[8][NGY][TZ][NB1];
    __shared__ double sT3[4][NT][NYZ];

    const PatchDev &pd = patches[0];
    const int t = threadIdx.x;
    const int ty = blockIdx.x % bx.nty, tz = blockIdx.x / bx.nty;
    const int Y0 = ty * TY, Z0 = tz * TZ;
    const int nbx = bx.nb[0], nby = bx.nb[1], nbz = bx.nb[2];
    const int nelx = bx.nel[0], nely = bx.nel[1], nelz = bx.nel[2];
    const int ey_lo = max(0, Y0 - P), ey_hi = min(nely - 1, Y0 + TY - 1);
    const int ez_lo = max(0, Z0 - P), ez_hi = min(nelz - 1, Z0 + TZ - 1);
    const int ney = ey_hi - ey_lo + 1, nez = ez_hi - ez_lo + 1;
    const int ngy = ney * NB1, ngz = nez * NB1, ncy = ney + P, ncz = nez + P;
    const double *tx = tab + bx.toff[0], *tyb = tab + bx.toff[1], *tzb = tab + bx.toff[2];
    const int Gx = bx.g[0], Gy = bx.g[1], Gz = bx.g[2];

    for (int k = t; k < ngy * NB1; k += 256) {
        const int gy = k / NB1, m = k % NB1;
        const int g = ey_lo * NB1 + gy;
        sVy[gy][m] = tyb[(int64_t)g * NB1 + m];
        sDy[gy][m] = tyb[(int64_t)Gy * NB1 + (int64_t)g * NB1 + m];
    }
    for (int k = t; k < ngz * NB1; k += 256) {
        const int gz = k / NB1, m = k % NB1;
        const int g = ez_lo * NB1 + gz;
        sVz[gz][m] = tzb[(int64_t)g * NB1 + m];
        sDz[gz][m] = tzb[(int64_t)Gz * NB1 + (int64_t)g * NB1 + m];
    }
    for (int k = t; k < ngy; k += 256) sWy[k] = tyb[2 * (int64_t)Gy * NB1 + ey_lo * NB1 + k];
    for (int k = t; k < ngz; k += 256) sWz[k] = tzb[2 * (int64_t)Gz * NB1 + ez_lo * NB1 + k];

    // accumulators: combo c = t + 256 ci -> row (iyl, izl) = c / KPR, pair
    // and ox from c % KPR; acc[ci][r] belongs to row ix = e + r
    double acc[CPT][NB1];
    int cu[CPT], cox[CPT], crow[CPT];
#pragma unroll
    for (int ci = 0; ci < CPT; ++ci) {
        const int c = t + 256 * ci;
        crow[ci] = -1;
        cu[ci] = 0;
        cox[ci] = 0;
        if (c < NCOMBO) {
            crow[ci] = c / KPR;
            const int k = c % KPR;
            if (k < NB1) {
                cu[ci] = 0;
                cox[ci] = k;
            } else {
                cu[ci] = 1 + (k - NB1) / W;
                cox[ci] = (k - NB1) % W - P;
            }
        }
#pragma unroll
        for (int r = 0; r < NB1; ++r) acc[ci][r] = 0.0;
    }

    // entry (i, o) of the upper half
    auto store = [&](int ix, int iy, int iz, int ox, int oy, int oz, double v) {
        if (ix >= nbx || iy >= nby || iz >= nbz) return;
        const int64_t row = ix + (int64_t)nbx * (iy + (int64_t)nby * iz);
        raw[row * SfRaw<P>::ROW + SfRaw<P>::line(oy, oz) * SfRaw<P>::OXP + ox + P] = v;
    };

    for (int ex = 0; ex < nelx; ++ex) {
        __syncthreads();   // previous element's readers of sVx/sC are done
        for (int k = t; k < NB1 * NB1; k += 256) {
            const int q = k / NB1, m = k % NB1;
            const int g = ex * NB1 + q;
            sVx[q][m] = tx[(int64_t)g * NB1 + m];
            sDx[q][m] = tx[(int64_t)Gx * NB1 + (int64_t)g * NB1 + m];
        }
        if (t < NB1) sWx[t] = tx[2 * (int64_t)Gx * NB1 + ex * NB1 + t];
        for (int k = t; k < NB1 * ncz * ncy * 3; k += 256) {
            const int c = k % 3, by = (k / 3) % ncy, bz = (k / (3 * ncy)) % ncz, bxl = k / (3 * ncy * ncz);
            const int64_t m = (int64_t)(ex + bxl) + (int64_t)nbx * ((ey_lo + by) + (int64_t)nby * (ez_lo + bz));
            sC[bxl][bz][by][c] = pd.ctrl[m * 3 + c];
        }
        for (int k = t; k < nez * ney; k += 256) {
            const int eyl = k % ney, ezl = k / ney;
            sK[ezl][eyl] = pd.kappa ? pd.kappa[ex + (int64_t)nelx * ((ey_lo + eyl) + (int64_t)nely * (ez_lo + ezl))]
                                    : 1.0;
        }
        __syncthreads();
        for (int qx = 0; qx < NB1; ++qx) {
            // A: x contraction of the control points (value and derivative)
            for (int k = t; k < ncz * ncy * 6; k += 256) {
                const int c = k % 3, f = (k / 3) % 2, by = (k / 6) % ncy, bz = k / (6 * ncy);
                double s = 0.0;
#pragma unroll
                for (int bxl = 0; bxl < NB1; ++bxl) s += sC[bxl][bz][by][c] * (f ? sDx[qx][bxl] : sVx[qx][bxl]);
                sGX[bz][by][f * 3 + c] = s;
            }
            __syncthreads();
            // B: y contraction: (xv yv), (xd yv), (xv yd) per coordinate
            for (int k = t; k < ncz * ngy * 9; k += 256) {
                const int c = k % 3, cb = (k / 3) % 3, gy = (k / 9) % ngy, bz = k / (9 * ngy);
                const int eyl = gy / NB1;
                const int fx = cb == 1, fy = cb == 2;
                double s = 0.0;
#pragma unroll
                for (int m = 0; m < NB1; ++m)
                    s += sGX[bz][eyl + m][fx * 3 + c] * (fy ? sDy[gy][m] : sVy[gy][m]);
                sGY[bz][gy][cb * 3 + c] = s;
            }
            __syncthreads();
            // C: z contraction -> Jacobian at every (gy, gz), then D
            for (int k = t; k < ngy * ngz; k += 256) {
                const int gy = k % ngy, gz = k / ngy;
                const int ezl = gz / NB1, eyl = gy / NB1;
                double J[3][3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    double j0 = 0.0, j1 = 0.0, j2 = 0.0;
#pragma unroll
                    for (int m = 0; m < NB1; ++m) {
                        const double vz = sVz[gz][m], dz = sDz[gz][m];
                        j0 += sGY[ezl + m][gy][3 + c] * vz;
                        j1 += sGY[ezl + m][gy][6 + c] * vz;
                        j2 += sGY[ezl + m][gy][c] * dz;
                    }
                    J[c][0] = j0;
                    J[c][1] = j1;
                    J[c][2] = j2;
                }
                const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
                const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
                const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
                const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
                double inv[3][3];
                inv[0][0] = c00 / det;
                inv[1][0] = c01 / det;
                inv[2][0] = c02 / det;
                inv[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) / det;
                inv[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) / det;
                inv[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) / det;
                inv[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) / det;
                inv[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) / det;
                inv[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / det;
                const double w = sWx[qx] * sWy[gy] * sWz[gz];
                double cq = w * fabs(det);
                if (pd.kappa) cq *= sK[ezl][eyl];
                int s = 0;
#pragma unroll
                for (int a = 0; a < 3; ++a)
#pragma unroll
                    for (int b = a; b < 3; ++b) {
                        const double m = inv[a][0] * inv[b][0] + inv[a][1] * inv[b][1] + inv[a][2] * inv[b][2];
                        sD[s++][gz][gy] = cq * m;
                    }
            }
            __syncthreads();
            // D: z contraction of D for oz >= 0.  Arrays: (a,b) = 00, 01 (= 10),
            // 11 with z flags (0,0); 20, 21 with (1,0); 02, 12 with (0,1); 22.
            for (int k = t; k < 8 * ngy * TZ * NB1; k += 256) {
                const int oz = k % NB1, izl = (k / NB1) % TZ, gy = (k / (NB1 * TZ)) % ngy, arr = k / (NB1 * TZ * ngy);
                const int iz = Z0 + izl;
                const int sidx = arr == 0 ? 0 : arr == 1 ? 1 : arr == 2 ? 3 : (arr == 3 || arr == 5) ? 2
                                 : (arr == 4 || arr == 6) ? 4 : 5;
                const int fa = arr == 3 || arr == 4 || arr == 7, fb = arr == 5 || arr == 6 || arr == 7;
                double s = 0.0;
                if (iz < nbz) {
                    const int e0 = max(ez_lo, iz + oz - P), e1 = min(ez_hi, iz);
                    for (int ez = e0; ez <= e1; ++ez)
#pragma unroll
                        for (int q = 0; q < NB1; ++q) {
                            const int gz = (ez - ez_lo) * NB1 + q;
                            const double ba = fa ? sDz[gz][iz - ez] : sVz[gz][iz - ez];
                            const double bb = fb ? sDz[gz][iz + oz - ez] : sVz[gz][iz + oz - ez];
                            s += (ba * bb) * sD[sidx][gz][gy];
                        }
                }
                sT1[arr][gy][izl][oz] = s;
            }
            __syncthreads();
            // E: y contraction, (a, b) folded into the x-flag classes
            // 0: (0,0); 1: (0,1),(0,2); 2: (1,0),(2,0); 3: (1,1),(1,2),(2,1),(2,2)
            for (int k = t; k < 4 * NT * NYZ; k += 256) {
                const int u = k % NYZ, trow = (k / NYZ) % NT, cls = k / (NYZ * NT);
                const int iyl = trow % TY, izl = trow / TY;
                const int iy = Y0 + iyl, iz = Z0 + izl;
                int oy, oz;
                sf_pair<P>(u, oy, oz);
                double s = 0.0;
                if (iy < nby && iz < nbz) {
                    const int e0 = max(ey_lo, max(iy, iy + oy) - P), e1 = min(ey_hi, min(iy, iy + oy));
                    const int npair = cls == 0 ? 1 : cls == 3 ? 4 : 2;
                    for (int pp = 0; pp < npair; ++pp) {
                        int a, b;
                        if (cls == 0) { a = 0; b = 0; }
                        else if (cls == 1) { a = 0; b = 1 + pp; }
                        else if (cls == 2) { a = 1 + pp; b = 0; }
                        else { a = 1 + (pp >> 1); b = 1 + (pp & 1); }
                        const int arr = (a == 0 && b == 0) ? 0 : (a + b == 1) ? 1 : (a == 1 && b == 1) ? 2
                                        : (a == 2 && b == 0) ? 3 : (a == 2 && b == 1) ? 4 : (a == 0 && b == 2) ? 5
                                        : (a == 1 && b == 2) ? 6 : 7;
                        const int fa = a == 1, fb = b == 1;
                        for (int ey = e0; ey <= e1; ++ey)
#pragma unroll
                            for (int q = 0; q < NB1; ++q) {
                                const int gy = (ey - ey_lo) * NB1 + q;
                                const double ba = fa ? sDy[gy][iy - ey] : sVy[gy][iy - ey];
                                const double bb = fb ? sDy[gy][iy + oy - ey] : sVy[gy][iy + oy - ey];
                                s += (ba * bb) * sT1[arr][gy][izl][oz];
                            }
                    }
                }
                sT3[cls][trow][u] = s;
            }
            __syncthreads();
            // F: x contraction into the rows e .. e + P
#pragma unroll
            for (int ci = 0; ci < CPT; ++ci) {
                if (crow[ci] < 0) continue;
                const double t0 = sT3[0][crow[ci]][cu[ci]], t1 = sT3[1][crow[ci]][cu[ci]];
                const double t2 = sT3[2][crow[ci]][cu[ci]], t3 = sT3[3][crow[ci]][cu[ci]];
                const int ox = cox[ci];
#pragma unroll
                for (int r = 0; r < NB1; ++r) {
                    const int r2 = r + ox;
                    if (r2 < 0 || r2 > P) continue;
                    const double va = sVx[qx][r], da = sDx[qx][r], vb = sVx[qx][r2], db = sDx[qx][r2];
                    acc[ci][r] += (((da * db) * t0 + (da * vb) * t1) + (va * db) * t2) + (va * vb) * t3;
                }
            }
        }
        // row ix = ex is complete (all rows at the last element)
        const int nrow = ex == nelx - 1 ? NB1 : 1;
#pragma unroll
        for (int ci = 0; ci < CPT; ++ci) {
            if (crow[ci] < 0) continue;
            const int iyl = crow[ci] % TY, izl = crow[ci] / TY;
            int oy, oz;
            sf_pair<P>(cu[ci], oy, oz);
            for (int r = 0; r < nrow; ++r) store(ex + r, Y0 + iyl, Z0 + izl, cox[ci], oy, oz, acc[ci][r]);
#pragma unroll
            for (int r = 0; r < P; ++r) acc[ci][r] = acc[ci][r + 1];
            acc[ci][P] = 0.0;
        }
    }
}

// ---------------------------------------------------------------------------
// The same row assembly with the three contractions on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64; operand layout: A[i][k] in lane i + 16 k, B[k][j]
// in lane j + 16 k, result [i][j] in lane j + 16 (i % 4), element i / 4).
// D comes precomputed per Gauss point (k_geo3d).  A block of 8 waves owns a
// 4 x 4 tile of basis rows in (y, z); per Gauss point column gx:
//   z:  T1_arr[gy][c]   = sum_gz D_s(arr)[gz][gy] Wz_f(arr)[gz][c]        (c = (izl, oz >= 0))
//   y:  T3_cls[e][c]    = sum_(a,b) in cls sum_gy Wy_f(a,b)[e][gy] T1_arr(a,b)[gy][c]   (e = (iyl, oy))
//   x:  acc[(ox, r)][(e, c)] += sum_cls X_cls[(ox, r)] T3_cls[e][c]
// with Wz, Wy the products of the 1D basis values/derivatives of row and
// column (x-independent, built once per block) and X_cls the same products
// along x for the current point.  The x result rows are i = 4 r + g with
// ox = 4 t + g - p: element r of a lane's result register is the ring
// position (row ix = e + r), so moving to the next element shifts the four
// elements of each register -- no data crosses lanes.
// ---------------------------------------------------------------------------
typedef double sf_d4 __attribute__((ext_vector_type(4)));

template <int P>
struct SfmCfg {
    static constexpr int NB1 = P + 1, W = 2 * P + 1, NS = W * W * W;
    // row tile in (y, z): 4 x 4 up to degree 3; 2 x 3 at degree 4 (the z
    // stage's 16 columns hold TZ (p + 1) <= 16, and the LDS arrays fit)
    static constexpr int TY = P == 4 ? 2 : 4, TZ = P == 4 ? 3 : 4;
    static constexpr int NGY = (TY + P) * NB1, NGZ = (TZ + P) * NB1;
    static constexpr int KZ = (NGZ + 3) / 4 * 4;       // z contraction depth (gz)
    static constexpr int MY = (NGY + 15) / 16 * 16;    // z stage rows (gy)
    static constexpr int KY = (NGY + 3) / 4 * 4;       // y contraction depth (gy)
    static constexpr int NE = TY * W;                  // y stage rows (iyl, oy)
    static constexpr int ME = (NE + 15) / 16 * 16;
    static constexpr int NC = TZ * NB1;                // columns (izl, oz >= 0)
    static constexpr int MTF = (W + 3) / 4;            // x stage row tiles (ox)
    static constexpr int NTF = NE;                     // x stage column tiles (one per e)
    static constexpr int NWAVE = 8;
    static constexpr int FPW = (MTF * NTF + NWAVE - 1) / NWAVE;
    static_assert(NC <= 16 && P <= 4, "one column tile; the ring holds at most five rows");
};

// A block computes the rows ix in [E0, E1) of its tile (the last block along x
// the p rows after them too) from the elements E0 - p .. E1 - 1: blocks along x
// balance the tiles over the CUs and fill the chip for small patches, at p
// extra elements each (sf_xblocks).  The z stage's operands stay in registers:
// its 1D products are the same for every column, D is requested from memory
// one column ahead (192 VGPRs at degree 3; two blocks a CU would leave 128 and
// spill: 5.2 ms).  Bound by the matrix instructions and the latency of the two
// barriers per column: 64^3 elements p = 3, 1.67 ms (3.04 ms with one block per
// tile, D and the z products in LDS and entries stored in the final layout).
// Giving an XCD neighbouring tiles took 1.78 ms.
template <int P>
__global__ __launch_bounds__(512, 2) void k_sfasm3d_mfma(const double *__restrict__ tab,
                                                         const double *__restrict__ Dq, SfBox bx,
                                                         double *__restrict__ raw)
{
    using C = SfmCfg<P>;
    constexpr int NB1 = C::NB1, W = C::W, TY = C::TY, TZ = C::TZ;
    constexpr int KZ = C::KZ, MY = C::MY, KY = C::KY, NE = C::NE, ME = C::ME, NC = C::NC;
    constexpr int MTF = C::MTF, NTF = C::NTF, FPW = C::FPW, NT_D = MY / 16;
    __shared__ double sWy[4][NE][KY];
    __shared__ double sT1[8][KY][16];
    __shared__ double sT3[5][NE][16];
    __shared__ double sVx[NB1][NB1], sDx[NB1][NB1];

    const int t = threadIdx.x, w = t / kWave, l = t % kWave;
    const int tiles = bx.nty * bx.ntz, xb = blockIdx.x / tiles, nxb = gridDim.x / tiles;
    const int ty = blockIdx.x % tiles % bx.nty, tz = blockIdx.x % tiles / bx.nty;
    const int Y0 = ty * TY, Z0 = tz * TZ;
    const int nbx = bx.nb[0], nby = bx.nb[1], nbz = bx.nb[2];
    const int nelx = bx.nel[0], nely = bx.nel[1], nelz = bx.nel[2];
    const int E0 = (int)((int64_t)nelx * xb / nxb), E1 = (int)((int64_t)nelx * (xb + 1) / nxb);
    const int exs = max(0, E0 - P);
    const int ey_lo = max(0, Y0 - P), ey_hi = min(nely - 1, Y0 + TY - 1);
    const int ez_lo = max(0, Z0 - P), ez_hi = min(nelz - 1, Z0 + TZ - 1);
    const int ngy = (ey_hi - ey_lo + 1) * NB1, ngz = (ez_hi - ez_lo + 1) * NB1;
    const double *tx = tab + bx.toff[0], *tyb = tab + bx.toff[1], *tzb = tab + bx.toff[2];
    const int Gx = bx.g[0], Gy = bx.g[1], Gz = bx.g[2];
    const int li = l % 16, lk = l / 16;

    // z stage: wave w forms array w of (a,b) = 00, 01 (= 10), 11 [z flags 00];
    // 20, 21 [10]; 02, 12 [01]; 22 [11].  wz: Bz^fa(iz, gz) Bz^fb(iz + oz, gz)
    // for this lane's column c = li = izl (p+1) + oz and gz = 4 ks + lk
    const int arr = w;
    const int sidx = arr == 0 ? 0 : arr == 1 ? 1 : arr == 2 ? 3 : (arr == 3 || arr == 5) ? 2
                     : (arr == 4 || arr == 6) ? 4 : 5;
    double wz[KZ / 4];
    {
        const int f = ((arr == 3 || arr == 4 || arr == 7) ? 2 : 0) + ((arr == 5 || arr == 6 || arr == 7) ? 1 : 0);
        const int iz = Z0 + li / NB1, jz = iz + li % NB1;
#pragma unroll
        for (int ks = 0; ks < KZ / 4; ++ks) {
            const int gz = 4 * ks + lk, ez = ez_lo + gz / NB1, m1 = iz - ez, m2 = jz - ez;
            double v = 0.0;
            if (li < NC && gz < ngz && iz < nbz && jz < nbz && m1 >= 0 && m1 <= P && m2 >= 0 && m2 <= P) {
                const int64_t g = (int64_t)ez_lo * NB1 + gz;
                const double a = (f & 2) ? tzb[(int64_t)Gz * NB1 + g * NB1 + m1] : tzb[g * NB1 + m1];
                const double b = (f & 1) ? tzb[(int64_t)Gz * NB1 + g * NB1 + m2] : tzb[g * NB1 + m2];
                v = a * b;
            }
            wz[ks] = v;
        }
    }
    // Wy[f][e][gy]: By^fa(iy, gy) By^fb(iy + oy, gy), e = iyl (2p+1) + oy + p
    for (int k = t; k < 4 * NE * KY; k += 512) {
        const int gy = k % KY, e = (k / KY) % NE, f = k / (KY * NE);
        double v = 0.0;
        if (gy < ngy) {
            const int iyl = e / W, oy = e % W - P;
            const int iy = Y0 + iyl, jy = iy + oy, ey = ey_lo + gy / NB1;
            const int m1 = iy - ey, m2 = jy - ey;
            if (iy < nby && jy >= 0 && jy < nby && m1 >= 0 && m1 <= P && m2 >= 0 && m2 <= P) {
                const int64_t g = (int64_t)ey_lo * NB1 + gy;
                const double a = (f & 2) ? tyb[(int64_t)Gy * NB1 + g * NB1 + m1] : tyb[g * NB1 + m1];
                const double b = (f & 1) ? tyb[(int64_t)Gy * NB1 + g * NB1 + m2] : tyb[g * NB1 + m2];
                v = a * b;
            }
        }
        sWy[f][e][gy] = v;
    }

    // ring positions 0..3 in the four elements of acc; at degree 4 the fifth
    // (row ex + 4, first touched by element ex) accumulates in element 0 of
    // acc4 and moves into element 3 of acc when the ring shifts
    // (only ox <= 0, the x tiles 0 and 1, reach position 4: fi = w + 8 u < 2 NTF)
    constexpr int NA4 = P == 4 ? (2 * NTF + 7) / 8 : 1;
    sf_d4 acc[FPW], acc4[NA4];
#pragma unroll
    for (int u = 0; u < FPW; ++u) acc[u] = sf_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < NA4; ++u) acc4[u] = sf_d4{0.0, 0.0, 0.0, 0.0};

    // D of column gc at gz = 4 ks + lk, gy = 16 mt + li.  Beyond the tile's
    // window the last entry is read: the 1D products there are 0.
    double dn[KZ / 4][NT_D];
    auto d_load = [&](int gc) {
        const double *q = Dq + (((int64_t)min(gc, Gx - 1) * 6 + sidx) * Gz + ez_lo * NB1) * Gy + ey_lo * NB1;
#pragma unroll
        for (int ks = 0; ks < KZ / 4; ++ks)
#pragma unroll
            for (int mt = 0; mt < NT_D; ++mt)
                dn[ks][mt] = q[(int64_t)min(4 * ks + lk, ngz - 1) * Gy + min(16 * mt + li, ngy - 1)];
    };
    auto x_tables = [&](int ex) {
        if (t < NB1 * NB1) {
            const int q = t / NB1, m = t % NB1;
            const int64_t g = (int64_t)ex * NB1 + q;
            sVx[q][m] = tx[g * NB1 + m];
            sDx[q][m] = tx[(int64_t)Gx * NB1 + g * NB1 + m];
        }
    };
    d_load(exs * NB1);
    x_tables(exs);
    __syncthreads();

    // y-stage work units: (class, row tile, pair subset); class 3 in two halves
    // (planes 3 and 4 of sT3, summed when the x stage reads them)
    constexpr int NMT = ME / 16, NUNIT = 5 * NMT;
    for (int ex = exs; ex < E1; ++ex) {
        for (int qx = 0; qx < NB1; ++qx) {
            // z: the wave's row tiles interleaved (independent accumulators)
            {
                sf_d4 a4[NT_D];
#pragma unroll
                for (int mt = 0; mt < NT_D; ++mt) a4[mt] = sf_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < KZ / 4; ++ks)
#pragma unroll
                    for (int mt = 0; mt < NT_D; ++mt)
                        a4[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(dn[ks][mt], wz[ks], a4[mt], 0, 0, 0);
#pragma unroll
                for (int mt = 0; mt < NT_D; ++mt)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int gy = 16 * mt + 4 * q + lk;
                        if (gy < KY) sT1[arr][gy][li] = a4[mt][q];
                    }
            }
            __syncthreads();
            d_load(ex * NB1 + qx + 1);
            if (qx == 0) x_tables(ex);   // the previous element's x stage is done
            // y: x-flag classes 0: (0,0); 1: (0,1),(0,2); 2: (1,0),(2,0); 3: (1,1),(1,2) | (2,1),(2,2)
            for (int unit = w; unit < NUNIT; unit += 8) {
                const int plane = (unit < 4 * NMT) ? 1 + unit / NMT : 0;   // units 0..: planes 1,2,3,4 then 0
                const int mt = unit % NMT;
                const int npair = plane == 0 ? 1 : 2;
                const int e = min(16 * mt + li, NE - 1);   // rows beyond the tile are not stored
                sf_d4 a4 = sf_d4{0.0, 0.0, 0.0, 0.0}, b4 = sf_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int pp = 0; pp < 2; ++pp) {
                    if (pp >= npair) break;
                    int a, b;
                    if (plane == 0) { a = 0; b = 0; }
                    else if (plane == 1) { a = 0; b = 1 + pp; }
                    else if (plane == 2) { a = 1 + pp; b = 0; }
                    else if (plane == 3) { a = 1; b = 1 + pp; }
                    else { a = 2; b = 1 + pp; }
                    const int ar = (a == 0 && b == 0) ? 0 : (a + b == 1) ? 1 : (a == 1 && b == 1) ? 2
                                   : (a == 2 && b == 0) ? 3 : (a == 2 && b == 1) ? 4 : (a == 0 && b == 2) ? 5
                                   : (a == 1 && b == 2) ? 6 : 7;
                    const int f = (a == 1 ? 2 : 0) + (b == 1 ? 1 : 0);
#pragma unroll
                    for (int ks = 0; ks < KY / 4; ++ks) {
                        const double av = sWy[f][e][4 * ks + lk];
                        const double bv = sT1[ar][4 * ks + lk][li];
                        if (ks & 1) b4 = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, b4, 0, 0, 0);
                        else a4 = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, a4, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (16 * mt + 4 * q + lk < NE) sT3[plane][16 * mt + 4 * q + lk][li] = a4[q] + b4[q];
            }
            __syncthreads();
            // x: rows i = 4 r + g (ox = 4 t + g - p), depth = the four classes
            double xa[MTF], xa4[MTF];
#pragma unroll
            for (int tt = 0; tt < MTF; ++tt) {
                const int r = li / 4, g = li % 4, ox = 4 * tt + g - P, r2 = r + ox, cls = lk;
                const bool fa = cls == 0 || cls == 1, fb = cls == 0 || cls == 2;
                double v = 0.0;
                if (r <= P && ox <= P && r2 >= 0 && r2 <= P)
                    v = (fa ? sDx[qx][r] : sVx[qx][r]) * (fb ? sDx[qx][r2] : sVx[qx][r2]);
                xa[tt] = v;
                // degree 4: rows g of the second operand hold ring position 4
                const int r4 = P, s2 = r4 + ox;
                double v4 = 0.0;
                if (P == 4 && li < 4 && ox <= P && s2 >= 0 && s2 <= P)
                    v4 = (fa ? sDx[qx][r4] : sVx[qx][r4]) * (fb ? sDx[qx][s2] : sVx[qx][s2]);
                xa4[tt] = v4;
            }
#pragma unroll
            for (int u = 0; u < FPW; ++u) {
                const int fi = w + 8 * u;
                if (fi < MTF * NTF) {
                    const int tt = fi / NTF, n = fi % NTF;
                    const double bv = lk == 3 ? sT3[3][n][li] + sT3[4][n][li] : sT3[lk][n][li];
                    acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[tt], bv, acc[u], 0, 0, 0);
                    if constexpr (P == 4)
                        if (u < NA4 && tt < 2)
                            acc4[u < NA4 ? u : 0] =
                                __builtin_amdgcn_mfma_f64_16x16x4f64(xa4[tt], bv, acc4[u < NA4 ? u : 0], 0, 0, 0);
                }
            }
        }
        // rows complete after this element: ring position 0 (all at the last element)
        const int nrow = ex < E0 ? 0 : ex == nelx - 1 ? NB1 : 1;
        // opaque copies: the stores' indices are worked out here, once per
        // element, and not kept in registers across the loop
        int we = w, lie = li, lke = lk;
        asm volatile("" : "+v"(we), "+v"(lie), "+v"(lke));
#pragma unroll
        for (int u = 0; u < FPW; ++u) {
            const int fi = we + 8 * u;
            if (fi < MTF * NTF) {
                const int tt = fi / NTF, n = fi % NTF;
                const int iyl = n / W, oy = n % W - P, izl = lie / NB1, oz = lie % NB1;
                const int iy = Y0 + iyl, iz = Z0 + izl;
                // whole lines, the padding and (centre line) ox < 0 included
                if (nrow > 0 && lie < NC && (oz > 0 || oy >= 0) && iy < nby && iz < nbz) {
                    const int64_t row = ex + (int64_t)nbx * (iy + (int64_t)nby * iz);
                    double *q = raw + row * SfRaw<P>::ROW + SfRaw<P>::line(oy, oz) * SfRaw<P>::OXP + 4 * tt + lke;
#pragma unroll
                    for (int r = 0; r < NB1; ++r) {
                        if (r >= nrow) break;
                        double v;
                        if constexpr (P == 4) v = r < 4 ? acc[u][r < 4 ? r : 0] : (u < NA4 && tt < 2 ? acc4[u < NA4 ? u : 0][0] : 0.0);
                        else v = acc[u][r];
                        q[(int64_t)r * SfRaw<P>::ROW] = v;
                    }
                }
                if constexpr (P == 4) {
                    const bool has4 = u < NA4 && tt < 2;
                    acc[u] = sf_d4{acc[u][1], acc[u][2], acc[u][3], has4 ? acc4[u < NA4 ? u : 0][0] : 0.0};
                    if (has4) acc4[u < NA4 ? u : 0] = sf_d4{0.0, 0.0, 0.0, 0.0};
                } else {
                    acc[u] = sf_d4{acc[u][1], acc[u][2], acc[u][3], 0.0};
                }
            }
        }
    }
}

// Blocks along x for `tiles` row tiles: the split of the elements that takes
// the fewest element steps on the busiest of the 256 CUs (one block each),
// counting the p repeated elements and about two steps of set-up per block.
// One block per tile took 1347 us at 21^3 elements p = 4 (117 tiles), split
// 512 us.
static int sf_xblocks(int p, int tiles, int nelx)
{
    constexpr int slots = 256;
    int best = 1;
    int64_t cost = INT64_MAX;
    for (int c = 1; c <= nelx; ++c) {
        const int64_t rounds = ((int64_t)tiles * c + slots - 1) / slots;
        const int64_t k = rounds * ((nelx + c - 1) / c + (c > 1 ? p : 0) + 2);
        if (k < cost) {
            cost = k;
            best = c;
        }
    }
    return best;
}

// Geometry, load and oriented minimum of det J of a patch, by Gauss point
// columns.  A thread owns the column (gx, gy) and walks a chunk of elements
// along z: it contracts each new plane of control points with its own x and y
// values once (the last p + 1 contracted planes stay in registers), so a point
// costs three (p + 1)-term sums per coordinate and derivative.  Per point it
// writes D_ab = w |det J| kappa (J^-1 J^-T)_ab as [gx][ab][gz][gy] (whole lines:
// the lanes run along gy), and sums the load density w f |det J| against the z
// functions; function iz of chunk k goes to R1[k (ch + p) + iz - k ch][gx][gy].
// Bound by the D it writes and by FP64 arithmetic.  64^3
// elements p = 3: 324 us (0.85 GB written); one element per block took 1099 us.
template <int P>
__global__ __launch_bounds__(256) void k_geo3d(const PatchDev *__restrict__ patches, const double *__restrict__ tab,
                                               SfBox bx, int ch, double *__restrict__ detmin,
                                               double *__restrict__ Dq, double *__restrict__ R1)
{
    constexpr int NB1 = P + 1, KT = kGeoChunk * NB1;
    __shared__ double sV[KT][NB1], sD[KT][NB1], sW[KT];
    __shared__ double sMin[4];
    const PatchDev &pd = patches[0];
    const int t = threadIdx.x;
    const int Gx = bx.g[0], Gy = bx.g[1], Gz = bx.g[2];
    const double *tx = tab + bx.toff[0], *ty = tab + bx.toff[1], *tz = tab + bx.toff[2];
    const int ncb = (int)(((int64_t)Gx * Gy + 255) / 256), kz = blockIdx.x / ncb;   // chunks after columns
    const int e0 = kz * ch, e1 = min(e0 + ch, bx.nel[2]);
    for (int k = t; k < (e1 - e0) * NB1 * NB1; k += 256) {
        const int q = k / NB1, m = k % NB1;
        const int64_t g = (int64_t)e0 * NB1 + q;
        sV[q][m] = tz[g * NB1 + m];
        sD[q][m] = tz[(int64_t)Gz * NB1 + g * NB1 + m];
        if (m == 0) sW[q] = tz[2 * (int64_t)Gz * NB1 + g];
    }
    __syncthreads();
    const int64_t col = (int64_t)(blockIdx.x % ncb) * 256 + t;
    double dmin = 1e300;
    if (col < (int64_t)Gx * Gy) {
        const int gy = (int)(col % Gy), gx = (int)(col / Gy);
        const int ex = gx / NB1, ey = gy / NB1;
        double vx[NB1], dx[NB1];
#pragma unroll
        for (int m = 0; m < NB1; ++m) {
            vx[m] = tx[(int64_t)gx * NB1 + m];
            dx[m] = tx[(int64_t)Gx * NB1 + (int64_t)gx * NB1 + m];
        }
        const double *vyp = ty + (int64_t)gy * NB1, *dyp = vyp + (int64_t)Gy * NB1;
        const double wxy = tx[2 * (int64_t)Gx * NB1 + gx] * ty[2 * (int64_t)Gy * NB1 + gy];
        double hv[NB1][3], hx[NB1][3], hy[NB1][3], acc[NB1];
        auto load = [&](int z, int m) {
#pragma unroll
            for (int c = 0; c < 3; ++c) hv[m][c] = hx[m][c] = hy[m][c] = 0.0;
#pragma unroll 1
            for (int by = 0; by < NB1; ++by) {
                const double vy = vyp[by], dy = dyp[by];
                const double *q = pd.ctrl + 3 * (ex + (int64_t)bx.nb[0] * ((ey + by) + (int64_t)bx.nb[1] * z));
                double a0[3] = {0.0, 0.0, 0.0}, a1[3] = {0.0, 0.0, 0.0};
#pragma unroll
                for (int b = 0; b < NB1; ++b)
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const double v = q[3 * b + c];
                        a0[c] += v * vx[b];
                        a1[c] += v * dx[b];
                    }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    hv[m][c] += a0[c] * vy;
                    hx[m][c] += a1[c] * vy;
                    hy[m][c] += a0[c] * dy;
                }
            }
        };
        double *r1 = R1 + ((int64_t)kz * (ch + P) * Gx + gx) * Gy + gy;
        const int64_t r1s = (int64_t)Gx * Gy;
#pragma unroll
        for (int m = 0; m < NB1; ++m) acc[m] = 0.0;
#pragma unroll
        for (int m = 1; m < NB1; ++m) load(e0 + m - 1, m);
        for (int e = e0; e < e1; ++e) {
#pragma unroll
            for (int m = 0; m < P; ++m)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    hv[m][c] = hv[m + 1][c];
                    hx[m][c] = hx[m + 1][c];
                    hy[m][c] = hy[m + 1][c];
                }
            load(e + P, P);
            const int64_t el = ex + (int64_t)bx.nel[0] * (ey + (int64_t)bx.nel[1] * e);
            const double kap = pd.kappa ? pd.kappa[el] : 1.0;
#pragma unroll 1
            for (int q = 0; q < NB1; ++q) {
                const int qi = (e - e0) * NB1 + q;
                double x[3], J[3][3];
#pragma unroll
                for (int c = 0; c < 3; ++c) x[c] = J[c][0] = J[c][1] = J[c][2] = 0.0;
#pragma unroll
                for (int m = 0; m < NB1; ++m) {
                    const double bv = sV[qi][m], bd = sD[qi][m];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        x[c] += hv[m][c] * bv;
                        J[c][0] += hx[m][c] * bv;
                        J[c][1] += hy[m][c] * bv;
                        J[c][2] += hv[m][c] * bd;
                    }
                }
                const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
                const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
                const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
                const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
                const double w = wxy * sW[qi];
                dmin = fmin(dmin, pd.orient * det);
                const double S = w * (source_value(pd.fkind, 3, x, pd.felem, el) * fabs(det));
#pragma unroll
                for (int m = 0; m < NB1; ++m) acc[m] += sV[qi][m] * S;
                if (Dq) {
                    // J^-1 = cof / det: D = w kappa / |det| cof cof^T
                    const double cof[3][3] = {
                        {c00, J[0][2] * J[2][1] - J[0][1] * J[2][2], J[0][1] * J[1][2] - J[0][2] * J[1][1]},
                        {c01, J[0][0] * J[2][2] - J[0][2] * J[2][0], J[0][2] * J[1][0] - J[0][0] * J[1][2]},
                        {c02, J[0][1] * J[2][0] - J[0][0] * J[2][1], J[0][0] * J[1][1] - J[0][1] * J[1][0]}};
                    const double cq = w * kap / fabs(det);
                    double *dq = Dq + ((int64_t)gx * 6 * Gz + (e * NB1 + q)) * Gy + gy;
#pragma unroll
                    for (int a = 0; a < 3; ++a)
#pragma unroll
                        for (int b = a; b < 3; ++b) {
                            *dq = cq * (cof[a][0] * cof[b][0] + cof[a][1] * cof[b][1] + cof[a][2] * cof[b][2]);
                            dq += (int64_t)Gz * Gy;
                        }
                }
            }
            // function e is complete within the chunk
            *r1 = acc[0];
            r1 += r1s;
#pragma unroll
            for (int m = 0; m < P; ++m) acc[m] = acc[m + 1];
            acc[P] = 0.0;
        }
#pragma unroll
        for (int m = 0; m < P; ++m) {
            *r1 = acc[m];
            r1 += r1s;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) dmin = fmin(dmin, __shfl_xor(dmin, off, 64));
    if ((t & 63) == 0) sMin[t >> 6] = dmin;
    __syncthreads();
    if (t == 0) detmin[blockIdx.x] = fmin(fmin(sMin[0], sMin[1]), fmin(sMin[2], sMin[3]));
}

// Load vector of the free rows from k_geo3d's z sums: a block takes up to 64
// rows of one x-line (iy, iz) and contracts y into LDS, then x.  Chunks and
// Gauss points in ascending order.
template <int P>
__global__ __launch_bounds__(256) void k_load3d(const double *__restrict__ tab, SfBox bx, int ch,
                                                const double *__restrict__ R1, double *__restrict__ rhs)
{
    constexpr int NB1 = P + 1;
    __shared__ double sT[(64 + P) * NB1];
    const int Gx = bx.g[0], Gy = bx.g[1];
    const double *tx = tab + bx.toff[0], *ty = tab + bx.toff[1];
    const int nseg = (bx.m[0] + 63) / 64;
    const int seg = blockIdx.x % nseg, jy = (blockIdx.x / nseg) % bx.m[1], jz = blockIdx.x / nseg / bx.m[1];
    const int iy = bx.flo[1] + jy, iz = bx.flo[2] + jz;
    const int ix0 = bx.flo[0] + seg * 64, ix1 = min(ix0 + 64, bx.fhi[0] + 1);
    const int ea = max(0, ix0 - P), eb = min(bx.nel[0], ix1);   // elements of the segment
    const int g0 = ea * NB1, ng = (eb - ea) * NB1;
    const int ya = max(0, iy - P), yb = min(bx.nel[1] - 1, iy);
    const int nch = (bx.nel[2] + ch - 1) / ch;
    for (int k = threadIdx.x; k < ng; k += 256) {
        double s = 0.0;
        for (int c = max(0, iz - P) / ch; c < nch && c * ch <= iz; ++c) {
            const int sl = iz - c * ch, len = min(ch, bx.nel[2] - c * ch);
            if (sl >= len + P) continue;
            const double *q = R1 + (((int64_t)c * (ch + P) + sl) * Gx + g0 + k) * Gy;
            for (int e = ya; e <= yb; ++e)
#pragma unroll
                for (int j = 0; j < NB1; ++j) s += ty[(int64_t)(e * NB1 + j) * NB1 + iy - e] * q[e * NB1 + j];
        }
        sT[k] = s;
    }
    __syncthreads();
    const int ix = ix0 + threadIdx.x;
    if (threadIdx.x < 64 && ix < ix1) {
        double s = 0.0;
        for (int e = max(0, ix - P); e <= min(bx.nel[0] - 1, ix); ++e)
#pragma unroll
            for (int j = 0; j < NB1; ++j) s += tx[(int64_t)(e * NB1 + j) * NB1 + ix - e] * sT[(e - ea) * NB1 + j];
        rhs[(ix - bx.flo[0]) + (int64_t)bx.m[0] * (jy + (int64_t)bx.m[1] * jz)] = s;
    }
}

// rows of one block of k_sf_finish3d
template <int P> struct SfFinish { static constexpr int R = P >= 4 ? 8 : 16; };

// Free rows from the raw rows: CSR values (free columns in slot order =
// ascending columns), the FP64 stencil (0 at columns outside the free box), the
// FP32 upper half, and minus K_ij g_j over the eliminated columns on the rhs.
// A block takes up to R rows of one x-line into LDS: their own upper lines, one
// contiguous range, and each lower line (-oy, -oz) from the rows of the line
// (iy - oy, iz - oz) whose upper entries mirror it (p rows more on both sides).
// The CSR values are written row by row and the stencils slot by slot in runs
// of R rows.  A thread keeps its stencil offsets (its entries of a raw row, its
// slots of a CSR row, its row of a stencil run) over all rows, so the loops
// hold no divisions; with them the kernel was bound by integer arithmetic.
// Bound by the bytes and the latency of the mirrored reads: 64^3 elements p = 3,
// about 900 us for 2.8 GB (with divisions 1178 us; neighbouring lines on one XCD 1071
// us).
template <int P>
__global__ __launch_bounds__(256) void k_sf_finish3d(SfBox bx, int nfree, const int *__restrict__ rowptr,
                                                     const double *__restrict__ raw, double *__restrict__ s64,
                                                     float *__restrict__ s32, double *__restrict__ val,
                                                     double *__restrict__ rhs, const int *__restrict__ dofs,
                                                     const double *__restrict__ fixed, int *__restrict__ err)
{
    using Q = SfRaw<P>;
    constexpr int W = 2 * P + 1, NS = W * W * W, C = NS / 2, NH = stencil_half(NS);
    constexpr int R = SfFinish<P>::R, LD = R + 1;   // LD: odd stride in doubles against bank conflicts
    __shared__ double L[NS * LD];
    __shared__ int sBase[R + 1];
    const int t = threadIdx.x;
    // segments of an x-line, as even as they come
    const int nseg = (bx.m[0] + R - 1) / R;
    const int seg = blockIdx.x % nseg, jy = (blockIdx.x / nseg) % bx.m[1], jz = blockIdx.x / nseg / bx.m[1];
    const int j0 = (int)((int64_t)bx.m[0] * seg / nseg), nr = (int)((int64_t)bx.m[0] * (seg + 1) / nseg) - j0;
    const int r0 = j0 + bx.m[0] * (jy + bx.m[1] * jz);
    const int ix0 = bx.flo[0] + j0, iy = bx.flo[1] + jy, iz = bx.flo[2] + jz;
    const int64_t nbx = bx.nb[0], nbxy = nbx * bx.nb[1];
    if (t <= nr) sBase[t] = rowptr[r0 + t];
    auto free_x = [&](int x) { return x >= bx.flo[0] && x <= bx.fhi[0]; };
    auto free_yz = [&](int y, int z) {
        return y >= bx.flo[1] && y <= bx.fhi[1] && z >= bx.flo[2] && z <= bx.fhi[2];
    };
    const bool inner = free_x(ix0 - P) && free_x(ix0 + nr - 1 + P) && free_yz(iy - P, iz - P) && free_yz(iy + P, iz + P);
    if (!inner) {
        for (int k = t; k < NS * LD; k += 256) L[k] = 0.0;
        __syncthreads();
    }
    // own upper lines: slots C .. NS - 1 (the centre line from ox = 0)
    const double *own = raw + (ix0 + nbx * iy + nbxy * iz) * Q::ROW;
#pragma unroll
    for (int i0 = 0; i0 < Q::ROW; i0 += 256) {
        const int i = i0 + t, j = i % Q::OXP, u = i / Q::OXP;
        const int oz = u <= P ? 0 : 1 + (u - P - 1) / W, oy = u <= P ? u : (u - P - 1) % W - P;
        const int slot = ((oz + P) * W + (oy + P)) * W + j, x = ix0 + j - P;
        if (i < Q::ROW && j < W && slot >= C && free_yz(iy + oy, iz + oz))
            for (int rr = 0; rr < nr; ++rr)
                if (free_x(x + rr)) L[slot * LD + rr] = own[rr * Q::ROW + i];
    }
    // lower entries from their mirrors: row jx, upper offset ox = j - p of line
    // (oy, oz) is the entry of row jx + ox at (-ox, -oy, -oz)
    constexpr int RS = R + 2 * P;
    static_assert(RS * Q::OXP <= 256, "one thread per (row, ox) of a line");
    {
        const int j = t % Q::OXP, rs = t / Q::OXP, ox = j - P, jx = ix0 - P + rs, rr = jx + ox - ix0;
        const double *q = raw + (jx + nbx * iy + nbxy * iz) * Q::ROW + j;
        if (rs < RS && j < W && rr >= 0 && rr < nr && free_x(jx)) {
            double *d = L + rr - ox * LD;   // slot (P - oz, P - oy, P - ox)
            if (ox > 0) d[C * LD] = q[0];
            for (int u = 1; u < Q::NYZ; ++u) {
                const int oz = u <= P ? 0 : 1 + (u - P - 1) / W, oy = u <= P ? u : (u - P - 1) % W - P;
                if (free_yz(iy - oy, iz - oz))
                    d[(((P - oz) * W + (P - oy)) * W + P) * LD] = q[u * Q::OXP - (oy * nbx + oz * nbxy) * Q::ROW];
            }
        }
    }
    __syncthreads();
    // CSR values: this thread's slots of every row, at their place in the row's
    // window of free columns
    const int ylo = max(-P, bx.flo[1] - iy), ny = min(P, bx.fhi[1] - iy) - ylo + 1;
    const int zlo = max(-P, bx.flo[2] - iz), nz = min(P, bx.fhi[2] - iz) - zlo + 1;
#pragma unroll
    for (int s0 = 0; s0 < NS; s0 += 256) {
        const int sl = s0 + t, ox = sl % W - P, oy = (sl / W) % W - P - ylo, oz = sl / (W * W) - P - zlo;
        const bool on = sl < NS && oy >= 0 && oy < ny && oz >= 0 && oz < nz;
        const int yz = oz * ny + oy;
        for (int rr = 0; rr < nr; ++rr) {
            const int lo = max(-P, bx.flo[0] - ix0 - rr), nx = min(P, bx.fhi[0] - ix0 - rr) - lo + 1;
            const int base = sBase[rr];
            if (nx * ny * nz != sBase[rr + 1] - base) {
                if (t == 0) atomicOr(err, 1);
            } else if (on && ox >= lo && ox < lo + nx) {
                val[base + yz * nx + ox - lo] = L[sl * LD + rr];
            }
        }
    }
    if (s64 && t % R < nr) {
        double *q64 = s64 + stencil_index(0, r0 + t % R, NS);
        float *q32 = s32 ? s32 + stencil_index(0, r0 + t % R, NH) : nullptr;
        for (int sl = t / R; sl < NS; sl += 256 / R) {
            const double v = L[sl * LD + t % R];
            q64[sl * kStencilTile] = v;
            if (q32 && sl >= C) q32[(sl - C) * kStencilTile] = (float)v;
        }
    }
    if (!fixed || inner) return;
    // eliminated columns' K_ij g_j, read from the raw rows: 16 lanes per row,
    // then their sums in order
    __shared__ double sC[R][16];
    const int rw = t / 16, lane = t % 16;
    if (rw < R) {
        double g = 0.0;
        if (rw < nr)
            for (int sl = lane; sl < NS; sl += 16) {
                const int ox = sl % W - P, oy = (sl / W) % W - P, oz = sl / (W * W) - P;
                const int jx = ix0 + rw + ox, ky = iy + oy, kz = iz + oz;
                if (jx < 0 || jx >= bx.nb[0] || ky < 0 || ky >= bx.nb[1] || kz < 0 || kz >= bx.nb[2]) continue;
                if (free_x(jx) && free_yz(ky, kz)) continue;
                const int64_t col = jx + nbx * ky + nbxy * kz;
                const double v = sl >= C ? own[rw * Q::ROW + Q::line(oy, oz) * Q::OXP + ox + P]
                                         : raw[col * Q::ROW + Q::line(-oy, -oz) * Q::OXP + P - ox];
                g += v * fixed[dofs[col] - nfree];
            }
        sC[rw][lane] = g;
    }
    __syncthreads();
    if (t < nr) {
        double corr = 0.0;
        for (int j = 0; j < 16; ++j) corr += sC[t][j];
        rhs[r0 + t] -= corr;
    }
}

bool sf_supported(int d, int p) { return d == 3 && p >= 1 && p <= 4; }

int64_t sf_table_doubles(int p, const int *nel)
{
    int64_t n = 0;
    for (int k = 0; k < 3; ++k) n += (int64_t)nel[k] * (p + 1) * (2 * (p + 1) + 1);
    return n;
}

bool sf_mfma(int p) { return p >= 2 && p <= 4; }

int64_t sf_dq_doubles(int p, const int *nel)
{
    if (!sf_mfma(p)) return 0;
    return (int64_t)nel[0] * (p + 1) * 6 * ((int64_t)nel[1] * (p + 1)) * ((int64_t)nel[2] * (p + 1));
}

int64_t sf_raw_doubles(int p, const int *nb)
{
    const int64_t row = p == 1 ? SfRaw<1>::ROW : p == 2 ? SfRaw<2>::ROW : p == 3 ? SfRaw<3>::ROW : SfRaw<4>::ROW;
    return row * nb[0] * nb[1] * nb[2];
}

// elements per chunk of k_geo3d: shorter chunks (p planes more each) until two
// blocks per CU run
static int sf_chunk(int p, const int *nel)
{
    const int64_t cols = ((int64_t)nel[0] * (p + 1) * nel[1] * (p + 1) + 255) / 256;
    int ch = kGeoChunk;
    while (ch > 2 && cols * ((nel[2] + ch - 1) / ch) < 512) ch /= 2;
    return ch;
}

int64_t sf_load_doubles(int p, const int *nel)
{
    const int ch = sf_chunk(p, nel);
    return (int64_t)((nel[2] + ch - 1) / ch) * (ch + p) * nel[0] * (p + 1) * nel[1] * (p + 1);
}

int64_t sf_det_count(int p, const int *nel)
{
    const int ch = sf_chunk(p, nel);
    return ((int64_t)nel[0] * (p + 1) * nel[1] * (p + 1) + 255) / 256 * ((nel[2] + ch - 1) / ch);
}

hipError_t launch_sf_assemble(int p, const PatchDev *patches, const GaussTab &gt, double *tab, SfBox bx, double *R1,
                              double *detmin, double *Dq, double *raw, double *rhs, hipStream_t s)
{
    const int G = bx.g[0] + bx.g[1] + bx.g[2];
    const int ch = sf_chunk(p, bx.nel);
    const int64_t nload = (int64_t)((bx.m[0] + 63) / 64) * bx.m[1] * bx.m[2];
    const dim3 ggeo((unsigned)sf_det_count(p, bx.nel));
#define GSX_SF(PP)                                                                                              \
    if (p == PP) {                                                                                              \
        hipLaunchKernelGGL((k_sf_tables<PP>), dim3((G + 255) / 256), dim3(256), 0, s, patches, gt, tab, bx.g[0], \
                           bx.g[1], bx.g[2]);                                                                   \
        hipLaunchKernelGGL((k_geo3d<PP>), ggeo, dim3(256), 0, s, patches, tab, bx, ch, detmin,                  \
                           sf_mfma(PP) ? Dq : nullptr, R1);                                                     \
        hipLaunchKernelGGL((k_load3d<PP>), dim3((unsigned)nload), dim3(256), 0, s, tab, bx, ch, R1, rhs);       \
        if (sf_mfma(PP)) {                                                                                      \
            bx.nty = (bx.nb[1] + SfmCfg<(PP > 1 ? PP : 2)>::TY - 1) / SfmCfg<(PP > 1 ? PP : 2)>::TY;            \
            bx.ntz = (bx.nb[2] + SfmCfg<(PP > 1 ? PP : 2)>::TZ - 1) / SfmCfg<(PP > 1 ? PP : 2)>::TZ;            \
            hipLaunchKernelGGL((k_sfasm3d_mfma<(PP > 1 ? PP : 2)>),                                             \
                               dim3(bx.nty * bx.ntz * sf_xblocks(PP, bx.nty * bx.ntz, bx.nel[0])), dim3(512),   \
                               0, s, tab, Dq, bx, raw);                                                         \
        } else {                                                                                                \
            bx.nty = (bx.nb[1] + 1) / 2;                                                                        \
            bx.ntz = (bx.nb[2] + 1) / 2;                                                                        \
            hipLaunchKernelGGL((k_sfasm3d<PP>), dim3(bx.nty * bx.ntz), dim3(256), 0, s, patches, tab, bx, raw); \
        }                                                                                                       \
        return hipGetLastError();                                                                               \
    }
    GSX_SF(1) GSX_SF(2) GSX_SF(3) GSX_SF(4)
#undef GSX_SF
    return hipErrorInvalidValue;
}

hipError_t launch_sf_finish(int p, const SfBox &bx, int nfree, const int *rowptr, const double *raw, double *s64,
                            float *s32, double *val, double *rhs, const int *dofs, const double *fixed, int *err,
                            hipStream_t s)
{
    if (nfree <= 0) return hipSuccess;
#define GSX_SFF(PP)                                                                                             \
    if (p == PP) {                                                                                              \
        const int64_t nseg = (bx.m[0] + SfFinish<PP>::R - 1) / SfFinish<PP>::R;                                 \
        hipLaunchKernelGGL((k_sf_finish3d<PP>), dim3((unsigned)(nseg * bx.m[1] * bx.m[2])), dim3(256), 0, s, bx, \
                           nfree, rowptr, raw, s64, s32, val, rhs, dofs, fixed, err);                           \
        return hipGetLastError();                                                                               \
    }
    GSX_SFF(1) GSX_SFF(2) GSX_SFF(3) GSX_SFF(4)
#undef GSX_SFF
    return hipErrorInvalidValue;
}

}  // namespace gsx
