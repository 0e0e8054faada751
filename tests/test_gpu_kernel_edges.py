"""Kernels at the sizes where their tiling can go wrong (remainders, chunk and
tile edges, the smallest sizes), against the oracle or a plain reference."""
import numpy as np
import pytest

import oracle as O
from gismo_amd import gsx, problems

pytestmark = pytest.mark.gpu


def _noisy_box(d, p, n, seed=3, kappa=True):
    """Single noisy patch, n elements per direction (int or per direction)."""
    P = problems.box_patch(d, p, n)
    problems.perturb_interior(P, 0.1 / np.max(n), seed)
    if kappa:
        P.kappa = problems.lognormal_kappa(P.nelem, 0.5, seed)
    P.fkind = 1
    return problems.Problem([P], problems.all_sides(d), [], name=f"box-d{d}-p{p}-n{n}")


# one Gauss point column per thread (blocks of 256 columns), chunks of 1 to 8
# elements along the last direction, longer ones the more columns there are
@pytest.mark.parametrize("d,p,n", [(2, 1, (1, 1)), (2, 1, (128, 8)), (2, 2, (85, 9)), (2, 2, (86, 7)),
                                   (2, 3, (65, 17)), (2, 4, (3, 16)), (3, 1, (8, 17, 9)), (3, 2, (5, 6, 8)),
                                   (3, 3, (4, 4, 1)), (3, 3, (5, 3, 10)), (3, 4, (2, 3, 9)), (2, 1, (9000, 17)),
                                   (2, 2, (5000, 70)), (3, 1, (60, 50, 21)), (3, 2, (60, 61, 13))])
def test_error_norms_columns(ctx, d, p, n):
    prob = _noisy_box(d, p, n, kappa=False)
    dofs, nfree = O.mapper(prob.patches, prob.dir_sides, prob.ifaces)
    u = np.prod(np.sin(np.pi * prob.patches[0].ctrl), axis=1)
    sol = np.zeros(max(1, nfree))
    sol[dofs[dofs < nfree]] = u[dofs < nfree]
    gp = gsx.Problem(ctx, prob)
    x = ctx.to_device(sol)
    l2, h1 = gp.error_norms(x)
    # both sums have positive terms: rounding stays near 1e-15 per term
    assert l2 == pytest.approx(O.l2_error(prob.patches, dofs, nfree, sol), rel=1e-11)
    assert h1 == pytest.approx(O.h1_error(prob.patches, dofs, nfree, sol), rel=1e-11)
    x.close()
    gp.close()


# strips and tiles of 16 outputs; one mode product per launch where a box exceeds
# the strips' LDS (530 functions) or is thin (on both sides of that line)
@pytest.mark.parametrize("d,p,n", [(2, 1, (2, 2)), (2, 1, (17, 16)), (2, 2, (15, 33)), (2, 3, (3, 130)),
                                   (3, 1, (2, 2, 2)), (3, 2, (16, 15, 17)), (3, 3, (5, 31, 2)), (3, 4, (14, 2, 15)),
                                   (2, 1, (530, 3)), (2, 2, (270, 9)), (2, 3, (258, 18)), (3, 2, (4, 5, 200)), (3, 2, (17, 15, 193)), (3, 1, (300, 3, 4)),
                                   (3, 3, (255, 2, 5))])
def test_fd_apply_tiles(ctx, d, p, n):
    prob = _noisy_box(d, p, n, kappa=False)
    sides = [s for _, s in prob.dir_sides]
    gp = gsx.Problem(ctx, prob)
    fd = gsx.FastDiag(gp)
    r = np.random.default_rng(7).standard_normal(gp.nfree)
    want = O.fd_operator(prob.patches[0], sides)(r)
    rd, zd = ctx.to_device(r), ctx.array(gp.nfree)
    fd.apply(rd, zd)
    # sums of up to 2 (m0 + m1 + m2) terms of both eigenbases in FP64; an eigensolver
    # perturbs a direction's operator by a few eps of its norm, which the inverse
    # weighs against the smallest sum of eigenvalues (1.6e-11 for 300 x 3 x 4)
    import scipy.linalg as sla
    lam = [sla.eigvalsh(*O.tensor_1d(prob.patches[0].knots[k], p, *O._free_range(prob.patches[0], k, sides)))
           for k in range(d)]
    tol = max(1e-11, 4 * 2.2e-16 * max(l[-1] for l in lam) / sum(l[0] for l in lam))
    assert np.abs(zd.download() - want).max() <= tol * np.abs(want).max()
    for o in (rd, zd, fd, gp):
        o.close()


@pytest.mark.parametrize("d,p,n", [(2, 2, (17, 31)), (3, 2, (16, 5, 15)), (3, 3, (6, 14, 7))])
def test_fd_pcg_fp32_tiles(ctx, d, p, n):
    """FP32 iterations (FP32 factors) reach the FP64 solution."""
    prob = _noisy_box(d, p, n)
    dofs, nfree = O.mapper(prob.patches, prob.dir_sides, prob.ifaces)
    Ao, bo = O.assemble(prob.patches, dofs, nfree, 0)
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_EXPR, gsx.MIXED)
    fd = gsx.FastDiag(gp)
    its = []
    for prec in (gsx.FP64, gsx.MIXED):
        x = ctx.array(gp.nfree).zero()
        it, rel, ok = gsx.fd_cg_solve(A, fd, b, x, tol=1e-10, maxit=300, precision=prec)
        xs = x.download()
        assert ok and np.linalg.norm(bo - Ao @ xs) <= 1.1e-10 * np.linalg.norm(bo)
        its.append(it)
        x.close()
    assert its[1] <= its[0] + 5, its   # wrong FP32 factors would not precondition
    for o in (A, b, fd, gp):
        o.close()


# the structured CG: row tiles of 256 with staged windows, all slots read below
# 24 MB of operator and mirrored upper ones above, stretches of lines where these
# are long, a window for each plane of a tile where one for both is too large,
# direct reads where neither fits the LDS, several tiles a block above 524,288
# rows, four groups of threads a tile for 3D operators of up to 256 tiles, planes
# requested ahead in up to 1000
@pytest.mark.parametrize("d,p,n", [(2, 1, (2, 2)), (2, 2, (16, 17)), (2, 4, (300, 9)), (2, 1, (740, 731)),
                                   (3, 1, (9, 8, 7)), (3, 2, (3, 3, 600)), (3, 3, (2, 2, 450)), (3, 3, (19, 18, 19)),
                                   (3, 3, (21, 19, 20)), (3, 4, (13, 11, 12)), (3, 4, (2, 40, 3)),
                                   (3, 1, (42, 41, 43)), (3, 2, (42, 40, 41)),
                                   (2, 2, (700, 40)), (2, 3, (1100, 500)), (2, 4, (160, 30)), (3, 1, (900, 5, 4)),
                                   (3, 2, (700, 6, 5)), (3, 3, (130, 40, 3)), (3, 4, (300, 3, 2)),
                                   (3, 2, (1500, 40, 3)), (3, 1, (700, 30, 30)), (3, 1, (100, 90, 80))])
def test_structured_cg_tiles(ctx, d, p, n):
    """FP64 and mixed solves on the structured operator reach the CSR
    operator's solution in its iterations."""
    P = problems.box_patch(d, p, n)
    P.kappa = problems.lognormal_kappa(P.nelem, 0.3, 5)
    P.fkind = 1
    prob = problems.Problem([P], problems.all_sides(d), [])
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_EXPR, gsx.MIXED)
    # Ten FP64 iterations: the recurrences perturb each step by a few eps and
    # a perturbation grows at most with the Krylov polynomials, of norm up to
    # about sqrt(cond) <= 1e5 here before orthogonality is lost, so the two
    # operators' iterates agree to 10 * 1e-16 * 1e5 = 1e-10.  (After 120 the
    # flat boxes' iterates differ by 1e-5: orthogonality is gone there.)
    few = []
    for structured in (False, True):
        A.set_operator(structured)
        x = ctx.array(gp.nfree).zero()
        it, rel, ok = A.cg_solve(b, x, tol=1e-30, maxit=10)
        few.append((x.download(), it, A.history()))
        x.close()
    assert few[0][1] == few[1][1]
    assert np.linalg.norm(few[1][0] - few[0][0]) <= 1e-10 * np.linalg.norm(few[0][0])
    assert np.allclose(few[1][2], few[0][2], rtol=1e-9, atol=1e-13)
    # solves to 1e-9, the mixed one through FP32 iterations
    r = b.download()
    M = A.to_scipy()
    for prec in (gsx.FP64, gsx.MIXED):
        x = ctx.array(gp.nfree).zero()
        it, rel, ok = A.cg_solve(b, x, tol=1e-9, maxit=20000, precision=prec)
        assert ok and np.linalg.norm(r - M @ x.download()) <= 1.01e-9 * np.linalg.norm(r), (prec, it, rel)
        x.close()
    for o in (A, b, gp):
        o.close()


# CSR row sums: waves of 64 / L rows, entries in pairs, LDS chunks of 512
@pytest.mark.parametrize("n,lo,hi", [(1, 1, 1), (3, 0, 2), (65, 1, 9), (513, 0, 40), (1000, 30, 60), (301, 90, 420),
                                     (37, 700, 1300), (70000, 0, 12), (20000, 30, 60), (9000, 90, 300),
                                     (1500, 450, 900)])
def test_csr_products(ctx, n, lo, hi):
    """gsx_spmv on matrices with ragged, empty and long rows, and Jacobi
    sweeps of a multigrid hierarchy over them."""
    import scipy.sparse as sp
    rng = np.random.default_rng(n)
    m = max(n, 1400)   # distinct columns for the longest rows come from a window
    lens = rng.integers(lo, hi + 1, n)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(min(n, m), min(k, n), replace=False)) if k else np.zeros(0, int)
                         for k in lens]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(np.minimum(lens, n))]).astype(np.int32)
    va = rng.standard_normal(rp[-1])
    M = sp.csr_matrix((va, ci, rp), shape=(n, n))
    A = gsx.Matrix.from_csr(ctx, rp, ci, va)
    x = rng.standard_normal(n)
    xd, yd = ctx.to_device(x), ctx.array(n)
    A.spmv(xd, yd)
    # each row sum rounds by at most its length times eps of its absolute sum
    bound = 1e-16 * (1 + np.minimum(lens, n)) * (abs(M) @ abs(x)) + 1e-300
    assert np.all(np.abs(yd.download() - M @ x) <= 4 * bound)
    for o in (xd, yd, A):
        o.close()


# level operators in slices of 64 rows from 65,536 rows up (CSR rows below): four
# waves per slice below 131,072 rows, several slices per block above, uniform
# slices (inside a patch), a last slice of one row (257^2), rows next to
# interfaces; against the cycle written out in scipy
@pytest.mark.parametrize("gx,gy,n,p,levels", [(1, 1, 16, 2, 2), (2, 1, 12, 3, 2), (3, 2, 24, 3, 3), (2, 2, 8, 4, 2),
                                              (1, 1, 374, 2, 2), (2, 2, 60, 2, 3), (1, 1, 82, 3, 2), (2, 1, 52, 4, 2),
                                              (1, 1, 256, 3, 4), (2, 1, 184, 3, 4), (2, 2, 200, 2, 4), (2, 2, 136, 4, 4)])
@pytest.mark.parametrize("prec", [gsx.FP64, gsx.MIXED])
def test_multigrid_level_slices(ctx, gx, gy, n, p, levels, prec):
    prob = problems.square_grid(gx, gy, n, p)
    for k, P in enumerate(prob.patches):
        problems.perturb_interior(P, 0.1 / n, 30 + k)
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_FULL | gsx.ASM_KEEP_ELEMENTS, prec)
    mg = gsx.Multigrid(gp, A, levels, 2, 1, 0.7, precision=prec)
    ops = [mg.level(l) for l in range(levels)]
    import scipy.sparse.linalg as spla

    def cycle(l, rhs):
        M = ops[l][0]
        if l == 0:
            return spla.spsolve(M.tocsc(), rhs)
        d = M.diagonal()
        x = np.zeros_like(rhs)
        for _ in range(2):
            x = x + 0.7 * (rhs - M @ x) / d
        P = ops[l - 1][1]
        x = x + P @ cycle(l - 1, P.T @ (rhs - M @ x))
        return x + 0.7 * (rhs - M @ x) / d
    r = np.random.default_rng(4).standard_normal(gp.nfree)
    want = cycle(levels - 1, r)
    rd, zd = ctx.to_device(r), ctx.array(gp.nfree)
    mg.apply(rd, zd)
    # FP64: sums of at most 81 entries per smoothing step, cond(A_0) < 1e4;
    # mixed: level values and coarse vectors rounded to FP32 (6e-8), amplified
    # by the cycle's bounded operators
    tol = 1e-10 if prec == gsx.FP64 else 2e-5
    assert np.linalg.norm(zd.download() - want) <= tol * np.linalg.norm(want)
    x = ctx.array(gp.nfree).zero()
    it, rel, ok = gsx.mg_cg_solve(A, mg, b, x, tol=1e-9)
    bb = b.download()
    assert ok and np.linalg.norm(bb - A.to_scipy() @ x.download()) <= 1.01e-9 * np.linalg.norm(bb)
    for o in (rd, zd, x, mg, A, b, gp):
        o.close()


# the row assembly: tiles of 4 x 4 (2 x 3) rows in (y, z) split along x, Gauss
# point columns in chunks along z, x-line segments of 64 and of 16 (8) rows;
# boxes thinner than a chunk, a tile or the stencil, and eliminated columns
# moved to the right-hand side
@pytest.mark.parametrize("p,n", [(1, (1, 2, 3)), (1, (70, 4, 5)), (2, (1, 1, 1)), (2, (2, 5, 17)), (2, (67, 3, 2)),
                                 (3, (1, 1, 9)), (3, (17, 5, 4)), (3, (4, 18, 3)), (4, (1, 2, 1)), (4, (9, 2, 5)),
                                 (4, (2, 7, 9))])
@pytest.mark.parametrize("sides", [(1, 2, 3, 4, 5, 6), (2, 5)])
def test_row_assembly_tiles(ctx, p, n, sides):
    P = problems.box_patch(3, p, n)
    problems.perturb_interior(P, 0.1 / max(n), 9)
    P.kappa = problems.lognormal_kappa(P.nelem, 0.5, 9)
    P.fkind = 1
    prob = problems.Problem([P], [(0, s) for s in sides], [])
    gp = gsx.Problem(ctx, prob)
    if gp.nfree == 0:
        gp.close()
        pytest.skip("no free functions")
    gp.set_bc([(0, s, gsx.BC_DIRICHLET, gsx.BCF_AFFINE, (0.5, 1.0, -2.0, 0.25)) for s in sides])
    out = []
    for mode in (gsx.ASM_ROWWISE, gsx.ASM_ELEMENTWISE):
        A, b = gp.assemble(gsx.PATTERN_FULL | mode, gsx.MIXED)
        rp, ci, va = A.download()
        x = ctx.array(gp.nfree).zero()
        it, rel, ok = A.cg_solve(b, x, tol=1e-10, maxit=5000, precision=gsx.MIXED)   # on the stencils
        assert ok
        out.append((rp, ci, va, b.download()[:gp.nfree], gp.min_detj(), A.to_scipy(), x.download()))
        for o in (x, A, b):
            o.close()
    r, e = out
    assert np.array_equal(r[0], e[0]) and np.array_equal(r[1], e[1])
    # the same products grouped differently: up to (p+1)^3 27 9 terms per entry
    # at eps, judged against the row's largest entry
    scale = np.maximum.reduceat(np.abs(e[2]), e[0][:-1])
    assert np.all(np.abs(r[2] - e[2]) <= 1e-12 * np.repeat(scale, np.diff(e[0])))
    assert np.abs(r[3] - e[3]).max() <= 1e-12 * np.abs(e[3]).max()
    assert r[4] == pytest.approx(e[4], rel=1e-12)
    assert (r[5] != r[5].T).nnz == 0   # bitwise symmetric
    assert np.linalg.norm(r[3] - r[5] @ r[6]) <= 1.01e-10 * np.linalg.norm(r[3])
    gp.close()


# the 2D row assembly: blocks of 83 / 61 / 47 rows along x, chunks of 2 to 16
# rows along y, x-line segments of 32 rows, thin patches, glued patches with
# interface and corner rows, eliminated columns moved to the right-hand side
@pytest.mark.parametrize("p,n,gx,gy", [(2, (1, 1), 1, 1), (2, (82, 3), 1, 1), (2, (84, 17), 1, 1), (3, (59, 2), 1, 1),
                                       (3, (1, 40), 1, 1), (4, (44, 5), 1, 1), (4, (48, 1), 1, 1), (2, 9, 2, 2),
                                       (3, 63, 2, 1), (3, 5, 3, 3), (4, 7, 1, 2), (2, 90, 4, 4)])
def test_row_assembly_2d(ctx, p, n, gx, gy):
    if gx * gy == 1:
        P = problems.box_patch(2, p, n)
        P.kappa = problems.lognormal_kappa(P.nelem, 0.5, 9)
        prob = problems.Problem([P], problems.all_sides(2)[1:], [])
    else:
        prob = problems.square_grid(gx, gy, n, p)
    for k, P in enumerate(prob.patches):
        problems.perturb_interior(P, 0.1 / np.max(n), 40 + k)
        P.fkind = 1
    gp = gsx.Problem(ctx, prob)
    assert gp.nfree > 0
    gp.set_bc([(k, s, gsx.BC_DIRICHLET, gsx.BCF_AFFINE, (0.5, 1.0, -2.0, 0.25)) for k, s in prob.dir_sides])
    out = []
    for mode in (0, gsx.ASM_ELEMENTWISE):
        A, b = gp.assemble(gsx.PATTERN_FULL | mode, gsx.MIXED)
        rp, ci, va = A.download()
        x = ctx.array(gp.nfree).zero()
        it, rel, ok = A.cg_solve(b, x, tol=1e-10, maxit=20000, precision=gsx.MIXED)
        assert ok
        out.append((rp, ci, va, b.download()[:gp.nfree], gp.min_detj(), A.to_scipy(), x.download()))
        for o in (x, A, b):
            o.close()
    r, e = out
    assert np.array_equal(r[0], e[0]) and np.array_equal(r[1], e[1])
    # the same products grouped differently: up to (p+1)^2 16 4 terms per entry
    # at eps, judged against the row's largest entry (coordinates up to 4)
    scale = np.maximum.reduceat(np.abs(e[2]), e[0][:-1])
    assert np.all(np.abs(r[2] - e[2]) <= 1e-12 * np.repeat(scale, np.diff(e[0])))
    assert np.abs(r[3] - e[3]).max() <= 1e-12 * np.abs(e[3]).max()
    assert r[4] == pytest.approx(e[4], rel=1e-12)
    assert (r[5] != r[5].T).nnz == 0   # bitwise symmetric
    assert np.linalg.norm(r[3] - r[5] @ r[6]) <= 1.01e-10 * np.linalg.norm(r[3])
    gp.close()


def _glued_boxes(d, p, n, g):
    """g boxes per direction, glued; every outer side is a Dirichlet side."""
    patches, sides, ifaces = [], [], []
    at = {i: k for k, i in enumerate(np.ndindex(*g))}
    for i, k in at.items():
        patches.append(problems.box_patch(d, p, n, lo=[float(a) for a in i], hi=[a + 1.0 for a in i]))
        for j in range(d):
            t = [a for a in range(d) if a != j]
            up = at.get(tuple(a + (b == j) for b, a in enumerate(i)))
            if i[j] == 0:
                sides.append((k, 2 * j + 1))
            if up is None:
                sides.append((k, 2 * j + 2))
            else:
                ifaces.append((k, 2 * j + 2, up, 2 * j + 1, t[0], 0) + ((t[1], 0) if d == 3 else (0, 0)))
    return problems.Problem(patches, sides, ifaces)


# pattern kernels: rows of one occurrence by 16 or 64 lanes, coupled rows by
# merging windows (up to 8 patches at a corner), the closed form of a box in
# segments of 32 rows
@pytest.mark.parametrize("d,p,n,g", [(2, 1, (1, 2), (1, 1)), (2, 4, (3, 70), (1, 1)), (3, 1, (2, 1, 2), (1, 1, 1)),
                                     (3, 4, (1, 34, 2), (1, 1, 1)), (3, 2, (65, 3, 2), (1, 1, 1)),
                                     (2, 1, (1, 1), (2, 2)), (2, 3, (5, 2), (3, 2)), (2, 4, (33, 3), (2, 3)),
                                     (3, 1, (2, 2, 1), (2, 2, 2)), (3, 3, (2, 3, 2), (2, 2, 1)), (3, 4, (2, 2, 2), (1, 1, 2))])
@pytest.mark.parametrize("sides", [0, 1, 2])
def test_row_patterns(ctx, d, p, n, g, sides):
    """CSR patterns against the union of the functions' windows."""
    prob = _glued_boxes(d, p, n, g)
    prob.dir_sides = prob.dir_sides[::2] if sides == 1 else prob.dir_sides[:1] if sides == 2 else prob.dir_sides
    gp = gsx.Problem(ctx, prob)
    if gp.nfree == 0:
        gp.close()
        return
    dofs_all, off = gp.dofs(), 0
    want = [set() for _ in range(gp.nfree)]
    for k, P in enumerate(prob.patches):
        nb = [len(u) - P.p[0] - 1 for u in P.knots]
        dofs = dofs_all[off:off + P.nbasis].reshape(nb[::-1])
        off += P.nbasis
        for loc in np.ndindex(*nb[::-1]):
            r = dofs[loc]
            if r < gp.nfree:
                w = dofs[tuple(slice(max(0, i - p), i + p + 1) for i in loc)].ravel()
                want[r].update(w[w < gp.nfree].tolist())
    A, b = gp.assemble(gsx.PATTERN_FULL | gsx.ASM_REBUILD_PATTERN)
    rp, ci, va = A.download()
    assert np.array_equal(np.diff(rp), [len(w) for w in want])
    assert np.array_equal(ci, np.concatenate([sorted(w) for w in want]) if gp.nfree else [])
    for o in (A, b, gp):
        o.close()


# dense inverse: below, at and above the 64 tiles and the 256 pivot blocks, odd
# and even numbers of sweeps
@pytest.mark.parametrize("n", [(2, 2), (8, 10), (9, 9), (6, 14), (4, 44), (13, 17), (17, 17), (2, 258), (17, 33),
                               (25, 26), (34, 41)])
def test_dense_coarse_inverse(ctx, n):
    """A one-level multigrid applies the inverse of its matrix."""
    prob = _noisy_box(2, 1, n)
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_FULL)
    M = A.to_scipy().toarray()
    mg = gsx.Multigrid(gp, A, 1, 1, 1, 1.0)
    r = np.random.default_rng(3).standard_normal(gp.nfree)
    rd, zd = ctx.to_device(r), ctx.array(gp.nfree)
    mg.apply(rd, zd)
    z, zs = zd.download(), np.linalg.solve(M, r)
    # Gauss-Jordan on an SPD matrix: n eps cond
    assert np.linalg.norm(z - zs) <= 1.2e-16 * max(16, gp.nfree) * np.linalg.cond(M) * np.linalg.norm(zs)
    for o in (mg, rd, zd, A, b, gp):
        o.close()


# Galerkin levels from raw rows: one element per direction on the coarsest
# level, lines ending inside a block, interfaces, several levels
@pytest.mark.parametrize("p,n,g,levels", [(2, (2, 2), (1, 1), 2), (3, (2, 8), (1, 1), 2), (4, (4, 2), (1, 1), 2),
                                          (2, (36, 132), (1, 1), 3), (3, (8, 4), (2, 3), 3), (4, (12, 20), (2, 2), 3)])
@pytest.mark.parametrize("keep", [0, gsx.ASM_KEEP_ELEMENTS])
def test_galerkin_rows(ctx, p, n, g, levels, keep):
    """Every level's operator is P^T A P of the next finer one."""
    prob = _glued_boxes(2, p, n, g)
    for k, P in enumerate(prob.patches):
        problems.perturb_interior(P, 0.1 / max(n), 50 + k)
        P.kappa = problems.lognormal_kappa(P.nelem, 0.5, 60 + k)
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_FULL | keep)
    mg = gsx.Multigrid(gp, A, levels, 1, 1, 0.7)
    M = A.to_scipy()
    for l in range(levels - 2, -1, -1):
        Ac, P = mg.level(l)[:2]
        want = (P.T @ M @ P).tocsr()
        # (p + 2)^4 weighted terms per entry, weights at most 1
        D = abs(Ac - want)
        assert D.max() <= 1e-13 * (p + 2) ** 2 * abs(want).max()
        assert (Ac != Ac.T).nnz == 0
        M = Ac
    for o in (mg, A, b, gp):
        o.close()


# patches of one element: more blocks of the row assembly (675, 800 and 768
# determinant minima) than elements (225, 400 and 256), several blocks in the
# reduction of the minima
@pytest.mark.parametrize("p,g", [(4, 15), (2, 20), (3, 16)])
def test_row_assembly_of_one_element_patches(ctx, p, g):
    prob = problems.square_grid(g, g, 1, p)
    for k, P in enumerate(prob.patches):
        problems.perturb_interior(P, 0.1, 70 + k)
    gp = gsx.Problem(ctx, prob)
    out = []
    for mode in (0, gsx.ASM_ELEMENTWISE):
        A, b = gp.assemble(gsx.PATTERN_FULL | mode)
        out.append((*A.download(), b.download()[:gp.nfree], gp.min_detj()))
        A.close()
        b.close()
    r, e = out
    assert np.array_equal(r[0], e[0]) and np.array_equal(r[1], e[1])
    # as test_row_assembly_2d; the geometry's coordinates up to g multiply the
    # element path's rounding of a Jacobian of size 1
    scale = np.maximum.reduceat(np.abs(e[2]), e[0][:-1])
    assert np.all(np.abs(r[2] - e[2]) <= 1e-12 * g * np.repeat(scale, np.diff(e[0])))
    assert np.abs(r[3] - e[3]).max() <= 1e-12 * g * np.abs(e[3]).max()
    assert r[4] == pytest.approx(e[4], rel=1e-12 * g)
    gp.close()
    # a folded patch is found wherever it lies among the blocks
    for k in (0, g * g // 2, g * g - 1):
        ctrl = prob.patches[k].ctrl
        prob.patches[k].ctrl = ctrl.copy()
        prob.patches[k].ctrl[p + 2] += 3.0   # the first interior control point
        gp = gsx.Problem(ctx, prob)
        with pytest.raises(gsx.GsxError) as err:
            gp.assemble(gsx.PATTERN_FULL)
        assert err.value.status == gsx.GSX_ERR_JACOBIAN
        gp.close()
        prob.patches[k].ctrl = ctrl


@pytest.mark.parametrize("prec", [gsx.FP64, gsx.MIXED])
@pytest.mark.parametrize("per_row,lanes", [(60, 32), (150, 64), (300, 64), (700, 64)])
def test_batch_lanes_of_csr_members(ctx, prec, per_row, lanes):
    """A CSR member added without a tile shape sums its rows with the lanes of
    its mean row length, 64 for the longest: its iterates are bitwise those of
    the member given these lanes, and not those of 8 lanes."""
    import scipy.sparse as sp
    n = 900
    rng = np.random.default_rng(per_row)
    M = np.where(rng.random((n, n)) < per_row / n / 2, rng.standard_normal((n, n)), 0.0)
    M = M + M.T
    np.fill_diagonal(M, np.abs(M).sum(axis=1) + rng.uniform(0.5, 1.5, n))
    M = sp.csr_matrix(M)
    A = gsx.Matrix.from_csr(ctx, M.indptr, M.indices, M.data, with_fp32=True)
    b = ctx.to_device(rng.standard_normal(n))
    B = gsx.Batch(ctx, prec, 3)
    xs = [ctx.array(n).zero() for _ in range(3)]
    ids = [B.add(A, b, x, tol=1e-30, maxit=6, tile=t) for x, t in zip(xs, (None, (lanes, 1), (8, 1)))]
    B.run(6)
    got = [x.download() for x in xs]
    assert all(B.result(i)[1] >= 6 for i in ids)
    assert np.array_equal(got[0], got[1])
    assert not np.array_equal(got[0], got[2])
    for o in (B, b, A, *xs):
        o.close()


# patch 0's west and east sides on patch 1's south and west sides, so that the
# ends of patch 0's south side are one function: rows whose window holds both
# ends (up to p + 1 elements) meet that column twice
@pytest.mark.parametrize("p,n", [(2, 2), (2, 3), (3, 2), (3, 4), (4, 3), (4, 5), (3, 6)])
def test_patch_glued_to_itself_around_a_corner(ctx, p, n):
    patches = [problems.box_patch(2, p, (n, 3)), problems.box_patch(2, p, (3, 3), lo=[2.0, 2.0], hi=[3.0, 3.0])]
    for k, P in enumerate(patches):
        problems.perturb_interior(P, 0.1 / n, 80 + k)
        P.fkind = 1
    prob = problems.Problem(patches, [(1, 2), (1, 4)], [(0, 1, 1, 3, 0, 0, 0, 0), (0, 2, 1, 1, 1, 0, 0, 0)])
    dofs, nfree = O.mapper(prob.patches, prob.dir_sides, prob.ifaces)
    assert dofs[0] == dofs[n + p - 1] < nfree
    Ao, bo = O.assemble(prob.patches, dofs, nfree, 0)
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_EXPR)
    # as test_row_assembly_2d; a column listed twice in a row counts once
    assert np.abs(A.to_scipy().toarray() - Ao.toarray()).max() <= 1e-12 * np.abs(Ao.data).max()
    assert np.abs(b.download() - bo).max() <= 1e-12 * np.abs(bo).max()
    for o in (A, b, gp):
        o.close()


@pytest.mark.parametrize("mode", [0, gsx.ASM_ELEMENTWISE])
def test_kept_elements_serve_the_multigrid_setup(ctx, mode):
    """Element matrices or raw rows kept by an assembly are what the set-up
    takes: it forms none of its own."""
    prob = problems.square_grid(2, 2, 8, 3)
    gp = gsx.Problem(ctx, prob)
    for keep, formed in ((gsx.ASM_KEEP_ELEMENTS, 0), (0, 1)):
        A, b = gp.assemble(gsx.PATTERN_FULL | mode | keep)
        ctx.enable_timing(True)
        ctx.reset_timing()
        mg = gsx.Multigrid(gp, A, 2, 1, 1, 0.7)
        ctx.enable_timing(False)
        assert ctx.kernel_stats("mg_elem")[0] == formed
        ops = [mg.level(l) for l in range(2)]
        want = ops[0][1].T @ ops[1][0] @ ops[0][1]
        assert abs(ops[0][0] - want).max() <= 1e-13 * 25 * abs(want).max()   # as test_galerkin_rows
        for o in (mg, A, b):
            o.close()
    gp.close()


def _noisy_grid(g, n, p):
    prob = problems.square_grid(g, g, n, p)
    for k, P in enumerate(prob.patches):
        problems.perturb_interior(P, 0.1 / n, 90 + k)
        P.kappa = problems.lognormal_kappa(P.nelem, 0.5, 90 + k)
    return prob


# budgets in bytes that the element matrices fit (one patch: slabs of them) and
# the raw rows of all patches do not
@pytest.mark.parametrize("g,n,p,budget", [(1, 64, 2, 400_000), (1, 64, 4, 2_000_000), (4, 1, 4, 100_000)])
def test_raw_rows_keep_to_the_element_budget(ctx, g, n, p, budget):
    """Where the raw rows exceed the budget the element path runs: bitwise the
    matrix and load of an assembly that asks for it."""
    gp = gsx.Problem(ctx, _noisy_grid(g, n, p))
    out = []
    for b, mode in ((16 << 30, gsx.ASM_ELEMENTWISE), (budget, 0), (16 << 30, 0)):
        try:
            ctx.set_elem_budget(b)
            A, rhs = gp.assemble(gsx.PATTERN_FULL | mode)
        finally:
            ctx.set_elem_budget(16 << 30)
        out.append([*A.download(), rhs.download()])
        for o in (A, rhs):
            o.close()
    assert all(np.array_equal(u, v) for u, v in zip(out[0], out[1]))
    # the row path's sums round differently, so the comparison tells the paths
    assert not np.array_equal(out[0][2], out[2][2])
    gp.close()


def test_galerkin_rows_keep_to_the_element_budget(ctx):
    """Two levels' element matrices fit (233 KB), their raw rows and the lines
    between them do not (up to 426 KB): the levels come from element matrices."""
    gp = gsx.Problem(ctx, _noisy_grid(3, 2, 4))
    out = []
    for b, mode in ((16 << 30, gsx.ASM_ELEMENTWISE | gsx.ASM_KEEP_ELEMENTS), (270_000, 0), (16 << 30, 0)):
        try:
            ctx.set_elem_budget(b)
            A, rhs = gp.assemble(gsx.PATTERN_FULL | mode)
            mg = gsx.Multigrid(gp, A, 2, 1, 1, 0.7)
        finally:
            ctx.set_elem_budget(16 << 30)
        out.append(mg.level(0)[0].data)
        for o in (mg, A, rhs):
            o.close()
    assert np.array_equal(out[0], out[1]) and not np.array_equal(out[0], out[2])
    gp.close()


@pytest.mark.parametrize("prec", [gsx.FP64, gsx.MIXED])
def test_hierarchy_without_room_for_its_slices(ctx, prec):
    """Level slices are a second copy: where the finest one does not fit (an
    allocation above the CSR values' size fails) that level runs on its CSR
    arrays, and nothing is left of the slices."""
    prob = problems.square_grid(2, 1, 184, 3)
    gp = gsx.Problem(ctx, prob)
    A, b = gp.assemble(gsx.PATTERN_FULL, prec)
    assert gp.nfree >= 65536
    r = ctx.to_device(np.random.default_rng(8).standard_normal(gp.nfree))
    out, held = [], []
    for limit in (0, 8 * A.nnz):
        before = ctx.memory()
        try:
            ctx.set_alloc_limit(limit)
            mg = gsx.Multigrid(gp, A, 4, 2, 2, 0.6, precision=prec)
        finally:
            ctx.set_alloc_limit(0)
        held.append(ctx.memory() - before)
        z, x = ctx.array(gp.nfree), ctx.array(gp.nfree).zero()
        mg.apply(r, z)
        it, rel, ok = gsx.mg_cg_solve(A, mg, b, x, tol=1e-9)
        assert ok
        out.append((z.download(), it, x.download()))
        for o in (z, x, mg):
            o.close()
    # values and columns, of a mixed hierarchy FP32 and FP64 values and columns
    assert held[0] - held[1] >= (16 if prec == gsx.MIXED else 12) * A.nnz
    # both forms sum the same FP64 products of a row, in another order; the
    # mixed cycle rounds its coarse vectors to FP32
    assert np.linalg.norm(out[0][0] - out[1][0]) <= (1e-10 if prec == gsx.FP64 else 2e-5) * np.linalg.norm(out[0][0])
    assert abs(out[0][1] - out[1][1]) <= 1
    assert np.linalg.norm(out[0][2] - out[1][2]) <= 1e-6 * np.linalg.norm(out[0][2])
    for o in (r, b, A, gp):
        o.close()


def test_row_assembly_of_a_long_box(ctx):
    """More chunks of elements along z (65,600 of 8) than a grid's second
    dimension takes blocks."""
    n = (1, 1, 524800)
    P = problems.box_patch(3, 2, n, hi=[1.0, 1.0, 4100.0])
    P.kappa = 1.0 + 0.5 * np.sin(np.arange(P.nelem))
    P.fkind = 1
    gp = gsx.Problem(ctx, problems.Problem([P], problems.all_sides(3), []))
    out = []
    for mode in (0, gsx.ASM_ELEMENTWISE):
        A, b = gp.assemble(gsx.PATTERN_FULL | gsx.ASM_CSR_ONLY | mode)
        out.append((*A.download(), b.download(), gp.min_detj()))
        A.close()
        b.close()
    r, e = out
    assert np.array_equal(r[0], e[0]) and np.array_equal(r[1], e[1])
    # the Jacobian's z entries are differences of coordinates up to 4100 over an
    # element of 1/128: 4100 128 eps = 1e-10 of them in either path
    assert np.abs(r[2] - e[2]).max() <= 4e-10 * np.abs(e[2]).max()
    assert np.abs(r[3] - e[3]).max() <= 4e-10 * np.abs(e[3]).max()
    assert r[4] == pytest.approx(e[4], rel=4e-10)
    gp.close()
