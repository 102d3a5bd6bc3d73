"""GPU test of the cell-centred V-cycle's tile kernels at the level sizes where
the tile changes (register tiles up to 131072 cells, 8 x 8 x 8 up to 400000,
16 x 16 x 8 above) with ragged last tiles, periodic and bounded sides, sweep
counts that need no launch, one or several per leg, FP64 and mixed, and of the
kinds of kernel against each other.

The check is the answer's residual under the oracle's FP64 operator: the solve
stops at rtol in the library's operator and the two round differently by a few
eps per row, below rtol here, so 2 rtol bounds it."""
import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu

D, N = 1, 2
RTOL = 1e-10
CASES = [  # cells, periodic, lo, hi, nu1, nu2, mixed
    ((36, 20, 12), (1, 0, 1), (0, N, 0), (0, D, 0), 2, 2, False),
    ((36, 20, 12), (0, 1, 0), (N, 0, D), (D, 0, N), 0, 1, False),
    ((36, 20, 12), (1, 1, 1), (0, 0, 0), (0, 0, 0), 3, 0, False),
    ((20, 36, 12), (0, 0, 0), (N, N, N), (N, N, N), 1, 4, True),
    ((100, 44, 36), (0, 1, 1), (D, 0, 0), (N, 0, 0), 2, 2, False),    # 158400 cells
    ((100, 44, 36), (1, 1, 1), (0, 0, 0), (0, 0, 0), 2, 2, True),
    ((108, 76, 60), (0, 0, 1), (N, D, 0), (N, N, 0), 2, 2, False),    # 492480 cells
    ((108, 76, 60), (1, 1, 0), (0, 0, N), (0, 0, D), 2, 2, True),
]


@pytest.fixture(scope="module")
def ctx():
    from incflo_amd import mgx
    c = mgx.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,per,bclo,bchi,nu1,nu2,mixed", CASES)
def test_mac_tile_legs(ctx, orc, n, per, bclo, bchi, nu1, nu2, mixed):
    from incflo_amd import mgx
    print(f"case mac tiles {n} nu {nu1},{nu2} mixed {mixed}", flush=True)
    h = 1.0 / n[1]
    ph = tuple(m * h for m in n)
    g = orc.Geom.make(n, periodic=per, bclo=bclo, bchi=bchi, prob_hi=ph)
    rng = np.random.default_rng(sum(n) + nu1)
    beta = [0.5 + rng.random(orc.face_shape(g, d)) for d in range(3)]
    for d in range(3):
        if per[d]:
            lo, hi = [slice(None)] * 3, [slice(None)] * 3
            lo[2 - d], hi[2 - d] = 0, -1
            beta[d][tuple(hi)] = beta[d][tuple(lo)]
    b = rng.standard_normal(g.cell_shape())
    if all(per[d] or (bclo[d] != D and bchi[d] != D) for d in range(3)):
        b -= b.mean()
    bxs = B.chop_domain(n, 64)
    P = mgx.MacProjector(ctx, mgx.make_level(n, bxs, periodic=per, prob_hi=ph))
    P.setDomainBC(bclo, bchi)
    P.set_options(mgx.default_opts(nu1=nu1, nu2=nu2, maxiter=200, bottom_maxiter=200))
    P.set_beta(*[ctx.array(B.faces_to_boxed(beta[d], bxs, 0, d)) for d in range(3)], ng=0)
    rd = ctx.array(B.to_boxed(b, bxs, 0, periodic=per))
    xd = ctx.array(B.field_size(bxs, 0, 1))
    info = P.solve(xd, 0, rd, 0, RTOL, mode=mgx.MODE_MIXED if mixed else mgx.MODE_FP64)
    x = B.from_boxed(xd.download(), bxs, 0, g.cell_shape())
    P.close()
    assert info.converged and info.nlevels > 1
    r = orc.mac_residual(g, beta, b, x)
    assert np.max(np.abs(r)) <= 2 * RTOL * np.max(np.abs(b))


KINDS = {  # mac_tiles lines of the tuning table that give every level one kind
    "register tiles": "1000000000 1000000000 1000000000",
    "8 x 8 x 8 tiles": "0 1000000000 1000000000",
    "16 x 16 x 8 tiles": "0 0 1000000000",
    "one launch per colour": "0 0 0",  # FP32 and rows of a multiple of 32
}
BITS = [  # cells, periodic, lo, hi, nu1, nu2, mixed
    ((36, 20, 12), (1, 0, 1), (0, N, 0), (0, D, 0), 2, 2, False),
    ((36, 20, 12), (0, 0, 0), (D, N, N), (N, D, N), 1, 1, True),
    ((44, 28, 20), (0, 1, 0), (N, 0, D), (D, 0, N), 3, 3, False),
    ((44, 28, 20), (1, 1, 1), (0, 0, 0), (0, 0, 0), 4, 4, True),
    ((44, 28, 20), (0, 0, 1), (N, D, 0), (N, N, 0), 2, 3, False),
    ((44, 28, 20), (0, 0, 1), (N, D, 0), (N, N, 0), 3, 0, True),
    ((44, 28, 20), (1, 1, 0), (0, 0, N), (0, 0, D), 0, 5, False),
    ((64, 36, 20), (1, 0, 1), (0, N, 0), (0, D, 0), 2, 2, True),
    ((64, 36, 20), (0, 0, 0), (N, D, N), (N, N, N), 3, 2, True),
    ((128, 12, 20), (1, 1, 1), (0, 0, 0), (0, 0, 0), 0, 4, True),
    # more than 8.4M cells: blocks in chunks, with a partial round of them
    ((256, 196, 176), (1, 0, 1), (0, N, 0), (0, D, 0), 2, 2, False),
    ((256, 196, 176), (0, 1, 0), (N, 0, D), (N, 0, N), 1, 3, True),
]


@pytest.mark.parametrize("n,per,bclo,bchi,nu1,nu2,mixed", BITS)
def test_kinds_of_tile_agree_bitwise(ctx, n, per, bclo, bchi, nu1, nu2, mixed):
    """Three V-cycles (converged or not) with every level on one kind of kernel."""
    from incflo_amd import mgx
    print(f"case mac tile kinds {n} nu {nu1},{nu2} mixed {mixed}", flush=True)
    ph = tuple(m / n[1] for m in n)
    rng = np.random.default_rng(sum(n) + nu1)
    bxs = B.chop_domain(n, 64)
    rho = ctx.array(B.to_boxed(0.5 + rng.random(n[::-1]), bxs, 0))
    b = rng.standard_normal(n[::-1])
    rd = ctx.array(B.to_boxed(b - b.mean(), bxs, 0))
    base = mgx.tuning_get()
    lines = [ln for ln in base.splitlines() if not ln.startswith("mac_tiles")]
    ref = None
    try:
        for kind, cells in KINDS.items():
            mgx.tuning_set("\n".join(lines + [f"mac_tiles {cells}"]) + "\n")
            P = mgx.MacProjector(ctx, mgx.make_level(n, bxs, periodic=per, prob_hi=ph))
            P.setDomainBC(bclo, bchi)
            P.set_options(mgx.default_opts(nu1=nu1, nu2=nu2, maxiter=3))
            P.set_beta_from_density(rho, 0, 1.0)
            xd = ctx.array(B.field_size(bxs, 0, 1))
            try:
                P.solve(xd, 0, rd, 0, 1e-12, mode=mgx.MODE_MIXED if mixed else mgx.MODE_FP64)
            except mgx.MgxError as e:
                assert e.code == mgx.MGX_ERR_NOT_CONVERGED
            x = xd.download()
            P.close()
            assert np.max(np.abs(x)) > 0.0
            ref = x if ref is None else ref
            assert np.array_equal(x, ref), kind
    finally:
        mgx.tuning_set(base)
