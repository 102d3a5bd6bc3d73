"""GPU test of solves whose V-cycles contract badly or diverge through the levels of
2 and 3 cells: anisotropic cells and coefficients that jump by 1000.  The bounds
are the cycle counts without those levels (max_coarsening_level one lower) plus
15% and two cycles, for the other choice of levels has to be found on the way;
twice the count in the mixed mode, where a step runs up to three FP32 cycles
before it is judged."""
import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu

D, N, INF = 1, 2, 3
P3 = ((1, 1, 1), (0, 0, 0), (0, 0, 0))
CHANNEL = ((0, 0, 0), (INF, N, N), (D, N, N))


@pytest.fixture(scope="module")
def ctx():
    from incflo_amd import mgx
    c = mgx.Context(0)
    yield c
    c.close()


def _sigma(n, kind):
    if kind == "smooth":
        return 0.5 + np.random.default_rng(1).random(n[::-1])
    z, y, x = np.meshgrid(*[(np.arange(m) + 0.5) / m for m in n[::-1]], indexing="ij")
    return np.where((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.4) ** 2 < 0.09, 1000.0, 1.0)


CASES = [  # kind of solve, cells, sides, coefficients, cell shape
    ("mac", (40, 24, 32), CHANNEL, "smooth", (2, 1, 1)),
    ("mac", (40, 24, 32), P3, "smooth", (2, 1, 1)),
    ("mac", (36, 20, 12), P3, "smooth", (1, 1, 3)),
    ("mac", (96, 16, 24), CHANNEL, "smooth", (2, 1, 1)),
    ("nodal", (24, 200, 128), CHANNEL, "bubble", (1, 1, 1)),
    ("nodal", (40, 24, 32), ((1, 0, 1), (0, D, 0), (0, N, 0)), "bubble", (1, 1, 1)),
    ("nodal", (36, 20, 12), P3, "bubble", (1, 1, 1)),
]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("what,n,sides,kind,shape", CASES)
def test_no_worse_than_without_the_deep_levels(ctx, what, n, sides, kind, shape, mixed):
    from incflo_amd import mgx
    print(f"case level choice {what} {n} {kind} {shape} mixed {mixed}", flush=True)
    per, lo, hi = sides
    ph = tuple(m * s / n[1] for m, s in zip(n, shape))
    bxs = B.chop_domain(n, 64)
    lev = mgx.make_level(n, bxs, periodic=per, prob_hi=ph)
    nodal = what == "nodal"
    sig = _sigma(n, kind)
    rng = np.random.default_rng(3)
    b = rng.standard_normal(tuple(n[a] + (1 if nodal and not per[a] else 0) for a in (2, 1, 0)))
    b -= b.mean()
    rhs = ctx.array(B.to_boxed(b, bxs, 0, nodal=nodal, periodic=per))
    mode = mgx.MODE_MIXED if mixed else mgx.MODE_FP64

    def solve(**opts):
        if nodal:
            P = mgx.NodalProjector(ctx, lev)
            P.setDomainBC(lo, hi)
        else:
            P = mgx.MacProjector(ctx, lev)
            P.setDomainBC([N if v == INF else v for v in lo], hi)
        P.set_options(mgx.default_opts(maxiter=150, **opts))
        if nodal:
            P.set_sigma(ctx.array(B.to_boxed(sig, bxs, 0)), 0)
        else:
            P.set_beta_from_density(ctx.array(B.to_boxed(1.0 / sig, bxs, 0)), 0, 1.0)
        info = P.solve(ctx.array(B.field_size(bxs, 0, 1, nodal)), 0, rhs, 0, 1e-10, mode=mode)
        P.close()
        return info

    full = solve()
    few = solve(max_coarsening_level=full.nlevels - 2)
    assert few.nlevels == full.nlevels - 1
    print(f"  cycles {full.vcycles}, {few.vcycles} without the last level")
    assert full.vcycles <= (2 if mixed else 1.15) * few.vcycles + 2


DEEP = [  # cells, sides, levels: the last ones 2 or 3 cells wide
    ((128, 16, 8), P3, 3),                                      # 32 x 4 x 2
    ((128, 16, 8), CHANNEL, 3),
    ((256, 16, 8), ((0, 1, 1), (N, 0, 0), (D, 0, 0)), 3),       # 64 x 4 x 2
    ((8, 8, 96), ((1, 1, 0), (0, 0, N), (0, 0, N)), 3),         # 2 x 2 x 24
    ((64, 12, 24), ((1, 0, 1), (0, D, 0), (0, N, 0)), 3),       # 16 x 3 x 6
    ((24, 24, 12), P3, 3),                                      # 6 x 6 x 3
]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("what", ["nodal", "mac"])
@pytest.mark.parametrize("n,sides,levels", DEEP)
def test_levels_of_two_and_three_cells(ctx, orc, n, sides, levels, what, mixed):
    """Smooth coefficients on cubes through all levels: the cycles of any other
    hierarchy (8 to 11 to 1e-10) and the oracle's residual (within 2 rtol, the two
    operators round differently by a few eps per row)."""
    from incflo_amd import mgx
    print(f"case deep levels {what} {n} mixed {mixed}", flush=True)
    per, lo, hi = sides
    nodal = what == "nodal"
    if not nodal:
        lo = [N if v == INF else v for v in lo]
    ph = tuple(m / n[1] for m in n)
    g = orc.Geom.make(n, periodic=per, bclo=lo, bchi=hi, prob_hi=ph)
    bxs = B.chop_domain(n, 64)
    lev = mgx.make_level(n, bxs, periodic=per, prob_hi=ph)
    rng = np.random.default_rng(sum(n))
    sig = 0.5 + rng.random(n[::-1])
    b = rng.standard_normal(g.node_shape() if nodal else g.cell_shape())
    if all(per[d] or (lo[d] != D and hi[d] != D) for d in range(3)):
        b -= b.mean()
    rhs = ctx.array(B.to_boxed(b, bxs, 0, nodal=nodal, periodic=per))
    xd = ctx.array(B.field_size(bxs, 0, 1, nodal))
    P = mgx.NodalProjector(ctx, lev) if nodal else mgx.MacProjector(ctx, lev)
    P.setDomainBC(lo, hi)
    if nodal:
        P.set_sigma(ctx.array(B.to_boxed(sig, bxs, 0)), 0)
    else:
        beta = [0.5 + rng.random(orc.face_shape(g, d)) for d in range(3)]
        for d in range(3):
            if per[d]:
                first, last = [slice(None)] * 3, [slice(None)] * 3
                first[2 - d], last[2 - d] = 0, -1
                beta[d][tuple(last)] = beta[d][tuple(first)]
        P.set_beta(*[ctx.array(B.faces_to_boxed(beta[d], bxs, 0, d)) for d in range(3)], ng=0)
    info = P.solve(xd, 0, rhs, 0, 1e-10, mode=mgx.MODE_MIXED if mixed else mgx.MODE_FP64)
    x = B.from_boxed(xd.download(), bxs, 0, b.shape, nodal=nodal)
    P.close()
    assert info.nlevels == levels and info.vcycles <= 14
    r = orc.nodal_residual(g, sig, b, x) if nodal else orc.mac_residual(g, beta, b, x)
    assert np.max(np.abs(r)) <= 2e-10 * np.max(np.abs(b))
