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
