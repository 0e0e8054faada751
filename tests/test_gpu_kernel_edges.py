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


# one Gauss point column per thread (blocks of 256 columns), chunks of 8
# elements along the last direction
@pytest.mark.parametrize("d,p,n", [(2, 1, (1, 1)), (2, 1, (128, 8)), (2, 2, (85, 9)), (2, 2, (86, 7)),
                                   (2, 3, (65, 17)), (2, 4, (3, 16)), (3, 1, (8, 17, 9)), (3, 2, (5, 6, 8)),
                                   (3, 3, (4, 4, 1)), (3, 3, (5, 3, 10)), (3, 4, (2, 3, 9))])
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
