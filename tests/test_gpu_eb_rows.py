"""GPU test of the embedded-boundary level passes: levels whose rows are all in
the table and levels swept by the plain stencil with the rows at cut cells
apart (above 200000 nodes), node counts that are no multiple of a wave or of a
tile, periodic, Dirichlet and Neumann sides, and sweep counts with and without
a first sweep from zero or a sweep after the prolongation.

The check is the answer's residual under the operator apply, which goes cell by
cell and is itself checked against the oracle: the solve stops at rtol in the
assembled rows and the two round differently by a few eps per row, below rtol
here, so 2 rtol bounds it."""
import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu

D = 1
RTOL = 1e-9
CASES = [  # cells, periodic, lo, hi, nu1, nu2
    ((32, 16, 16), (0, 0, 1), (1, 2, 0), (1, 2, 0), 2, 2),
    ((40, 24, 12), (1, 0, 1), (0, 2, 0), (0, 2, 0), 1, 2),
    ((40, 24, 12), (0, 0, 0), (2, 2, 2), (1, 2, 2), 0, 2),
    ((40, 24, 12), (0, 1, 1), (2, 0, 0), (1, 0, 0), 3, 0),
    ((104, 52, 44), (0, 0, 1), (2, 2, 0), (1, 2, 0), 2, 2),   # 244860 nodes
    ((104, 52, 44), (1, 0, 0), (0, 2, 2), (0, 2, 2), 2, 2),
    ((104, 44, 52), (0, 1, 0), (1, 0, 2), (2, 0, 1), 0, 3),
]


@pytest.fixture(scope="module")
def ctx():
    from incflo_amd import mgx
    c = mgx.Context(0)
    yield c
    c.close()


def _solve(ctx, orc, n, per, bclo, bchi, nu1, nu2):
    """solves, checks the residual and returns the V-cycles"""
    from incflo_amd import mgx
    print(f"case eb rows {n} nu {nu1},{nu2}", flush=True)
    ph = tuple(m / n[1] for m in n)
    g = orc.Geom.make(n, periodic=per, bclo=bclo, bchi=bchi, prob_hi=ph)
    bxs = B.chop_domain(n, 32)
    P = mgx.NodalProjector(ctx, mgx.make_level(n, bxs, periodic=per, prob_hi=ph))
    P.setDomainBC(bclo, bchi)
    P.set_options(mgx.default_opts(nu1=nu1, nu2=nu2, maxiter=200))
    cyl = (0.45 * ph[0], 0.52, 0.21)
    P.set_eb_cylinder(*cyl)
    ct, _ = orc.eb_cylinder(g, *cyl)
    rng = np.random.default_rng(sum(n) + nu1)
    sigma = 0.5 + rng.random(g.cell_shape())
    mask = orc.eb_node_mask(g, ct).astype(bool)
    b = np.where(mask, rng.standard_normal(g.node_shape()), 0.0)
    if all(per[d] or (bclo[d] != D and bchi[d] != D) for d in range(3)):
        b = np.where(mask, b - b[mask].mean(), 0.0)
    P.set_sigma(ctx.array(B.to_boxed(sigma, bxs, 0)), 0)
    rd = ctx.array(B.to_boxed(b, bxs, 0, nodal=True, periodic=per))
    xd = ctx.array(B.field_size(bxs, 0, 1, True))
    info = P.solve(xd, 0, rd, 0, RTOL, 0.0, mode=mgx.MODE_FP64)
    od = ctx.array(B.field_size(bxs, 0, 1, True))
    P.apply(xd, 0, od, 0)
    Ax = B.from_boxed(od.download(), bxs, 0, g.node_shape(), nodal=True)
    P.close()
    assert info.converged and info.nlevels > 1
    r = np.where(mask, b - Ax, 0.0)
    assert np.max(np.abs(r)) <= 2 * RTOL * np.max(np.abs(b))
    return info.vcycles


@pytest.mark.parametrize("n,per,bclo,bchi,nu1,nu2", CASES)
def test_eb_passes(ctx, orc, n, per, bclo, bchi, nu1, nu2):
    _solve(ctx, orc, n, per, bclo, bchi, nu1, nu2)


SPLIT = [  # cells, periodic, lo, hi, nu1, nu2: four levels
    ((80, 48, 32), (0, 0, 1), (1, 2, 0), (1, 2, 0), 2, 2),
    ((80, 48, 32), (1, 0, 1), (0, 2, 0), (0, 2, 0), 1, 2),
    ((80, 48, 32), (0, 0, 0), (2, 2, 2), (1, 2, 2), 0, 2),
    ((80, 48, 32), (0, 1, 1), (2, 0, 0), (1, 0, 0), 3, 0),
    ((48, 32, 32), (0, 1, 0), (1, 0, 2), (2, 0, 1), 1, 1),
]


@pytest.mark.parametrize("nodes", [0, 3000])  # every level split; the third one in the table
@pytest.mark.parametrize("n,per,bclo,bchi,nu1,nu2", SPLIT)
def test_split_levels_below_the_first(ctx, orc, n, per, bclo, bchi, nu1, nu2, nodes):
    """Levels 1 and 2 swept by the plain stencil with their cut rows apart, the
    first sweep from zero among them.  The rows are the same either way, so each
    solve takes the cycles of the all-rows one to round-off."""
    from incflo_amd import mgx
    base = mgx.tuning_get()
    lines = [ln for ln in base.splitlines() if not ln.startswith("eb_row_nodes")]
    cycles = []
    try:
        for limit in (10 ** 9, nodes):
            mgx.tuning_set("\n".join(lines + [f"eb_row_nodes {limit}"]) + "\n")
            cycles.append(_solve(ctx, orc, n, per, bclo, bchi, nu1, nu2))
    finally:
        mgx.tuning_set(base)
    assert abs(cycles[0] - cycles[1]) <= 1
