"""GPU test of the multigrid levels under an overset mask: a block of fixed nodes
and a strip of a face, on grids whose levels would go down to 2 or 3 cells without
it.  Through such levels these cycles diverge or take three to four times as many;
the bounds are a third above the counts through levels of 4 cells and more (36, 47
and 27)."""
import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu

D, N, INF = 1, 2, 3


@pytest.fixture(scope="module")
def ctx():
    from incflo_amd import mgx
    c = mgx.Context(0)
    yield c
    c.close()


BLOCK, STRIP = np.s_[2:5, 2:5, 32:64], np.s_[:, 8:16, -1]
CASES = [  # cells, lo, hi, masked nodes (z, y, x), V-cycles
    ((128, 16, 16), (INF, N, N), (D, N, N), BLOCK, 48),
    ((128, 16, 16), (N, N, N), (N, N, N), BLOCK, 62),
    ((40, 24, 32), (N, N, N), (N, N, N), STRIP, 36),
]


@pytest.mark.parametrize("n,lo,hi,at,cycles", CASES)
def test_masked_solve_converges(ctx, n, lo, hi, at, cycles):
    from incflo_amd import mgx
    print(f"case masked levels {n} {lo} {hi}", flush=True)
    per, ph = (0, 0, 0), tuple(m / n[1] for m in n)
    bxs = B.chop_domain(n, 64)
    shape = tuple(m + 1 for m in n[::-1])
    mask = np.ones(shape)
    mask[at] = 0
    rng = np.random.default_rng(3)
    sigma = ctx.array(B.to_boxed(0.5 + rng.random(n[::-1]), bxs, 0))
    nodes = lambda a: ctx.array(B.to_boxed(a, bxs, 0, nodal=True, periodic=per))
    rhs = nodes(rng.standard_normal(shape))
    P = mgx.NodalProjector(ctx, mgx.make_level(n, bxs, periodic=per, prob_hi=ph))
    P.setDomainBC(lo, hi)
    P.set_sigma(sigma, 0)
    flags = B.to_boxed(mask, bxs, 0, nodal=True, periodic=per).astype(np.int32)
    P.setOversetMask(ctx.array(flags, np.int32))
    info = P.solve(nodes(np.zeros(shape)), 0, rhs, 0, 1e-10)
    assert info.nlevels == 3 and info.iters <= cycles
    P.setOversetMask(None)  # without it the levels go on
    if lo[0] == INF:
        assert P.solve(nodes(np.zeros(shape)), 0, rhs, 0, 1e-10).nlevels == 4
    P.close()
