"""GPU tests of the bottom solve's exits: whole levels solved as the bottom
(max_coarsening_level 0), where one outer iteration shows which exit was taken."""
import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu

D, N = 1, 2


@pytest.fixture(scope="module")
def ctx():
    from incflo_amd import mgx
    c = mgx.Context(0)
    yield c
    c.close()


def _solve(ctx, n, beta, b, rtol, **opts):
    """one MAC solve, Dirichlet at x = 0 and walls elsewhere, unit cells"""
    from incflo_amd import mgx
    bxs = B.chop_domain(n, 64)
    P = mgx.MacProjector(ctx, mgx.make_level(n, bxs, periodic=(0, 0, 0), prob_hi=n))
    P.setDomainBC((D, N, N), (N, N, N))
    P.set_options(mgx.default_opts(max_coarsening_level=0, **opts))
    P.set_beta(*[ctx.array(np.ascontiguousarray(f).ravel()) for f in beta], ng=0)
    x = ctx.array(B.field_size(bxs, 0, 1))
    info = P.solve(x, 0, ctx.array(np.ascontiguousarray(b).ravel()), 0, rtol)
    P.close()
    return info, x.download()


# A right-hand side of 1e-161 whose first BiCGStab iteration leaves a residual
# below bottom_rtol and a rho below the smallest double: that is convergence,
# not the breakdown that rho = 0 otherwise is.  Taken for a breakdown, the answer
# gives way to smoothing sweeps from zero and the solve takes 5 to 8 iterations.
UNDERFLOW = [  # right-hand side * 4096, bottom_rtol, exponent
    ((-279.5, 1486.0, 1034.0, 2125.0, 1952.5), 0.012, 531),
    ((-479.5, -330.0, -1216.5, -1089.5, -1768.0, -1683.0, -2050.5, -2020.5), 0.323, 534),
    ((-500.0, -1102.0, -2026.0, -2536.0, -3243.0, -3584.0, -3967.0, -4087.0), 0.178, 535),
    ((-410.0, -1189.0, -1946.0, -2606.0, -3186.0, -3627.0, -3940.0, -4095.0), 0.466, 535),
]


@pytest.mark.parametrize("b,rtol,k", UNDERFLOW)
def test_rho_underflow_after_convergence(ctx, b, rtol, k):
    n = (len(b), 1, 1)
    print(f"case bottom exit, rho underflow, {n} 2^-{k}", flush=True)
    beta = [np.ones([n[2 - a] + (2 - a == d) for a in range(3)]) for d in range(3)]
    info, _ = _solve(ctx, n, beta, np.array(b) / 4096 * 2.0 ** -k, rtol, bottom_solver="bicgstab",
                     bottom_rtol=rtol, maxiter=20)
    assert info.iters == 1


def _dense(n, beta):
    """-L of the solve above as a matrix (unit cells)"""
    m = int(np.prod(n))
    A = np.zeros((m, m))
    at = lambda p: p[0] + n[0] * (p[1] + n[1] * p[2])
    for k in range(n[2]):
        for j in range(n[1]):
            for i in range(n[0]):
                r = at((i, j, k))
                for d in range(3):
                    for s in (0, 1):
                        q, f = [i, j, k], [k, j, i]
                        q[d] += 2 * s - 1
                        f[2 - d] += s
                        w = beta[d][tuple(f)]
                        if 0 <= q[d] < n[d]:
                            A[r, at(q)] -= w
                            A[r, r] += w
                        elif d == 0 and s == 0:
                            A[r, r] += 2 * w
    return A


@pytest.mark.parametrize("seed", range(6))
@pytest.mark.parametrize("kind", ["cg", "bicgstab"])
def test_stopping_test_is_exact(ctx, kind, seed):
    """The residual after the first step, alpha = (b S S b) / (b S A S b) along the
    scaled right-hand side, is known to round-off (about 100 eps for 60 unknowns);
    a bottom_rtol 1e-12 above it has to accept that step and one 1e-12 below it
    has to go on: smoothing sweeps (CG) or the second half of the iteration."""
    n = (5, 4, 3)
    print(f"case bottom exit, stopping test, {kind} seed {seed}", flush=True)
    rng = np.random.default_rng(seed)
    beta = [0.5 + rng.random([n[2 - a] + (2 - a == d) for a in range(3)]) for d in range(3)]
    A = _dense(n, beta)
    b = rng.standard_normal(len(A))
    s2 = 1.0 / np.diag(A)
    p = s2 * b
    step = (b @ p) / (p @ A @ p) * p
    ratio = np.max(np.abs(b - A @ step)) / np.max(np.abs(b))
    for side in (1.0 + 1e-12, 1.0 - 1e-12):
        _, x = _solve(ctx, n, beta, b, 0.999, bottom_solver=kind,
                      bottom_rtol=ratio * side, bottom_maxiter=1, maxiter=1, verbose=0)
        same = np.max(np.abs(x + step)) <= 1e-12 * np.max(np.abs(step))
        assert same == (side > 1.0)
