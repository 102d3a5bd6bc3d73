"""GPU tests of the bottom-solve kernels at the sizes where their variant
changes: nodal rows in registers up to 512 nodes, columns of 4 or 8 nodes where
512 threads hold the level, rows in global memory for others up to 4096, then
segments of columns (the multiplied vector in LDS or global memory); EB and
cell-centred rows in registers up to 1024 and 2048 unknowns, in global memory
above, and their vectors from 4096 on.

max_coarsening_level 0 makes the whole level the bottom, so each size runs one
variant.  The check is the answer's residual under the oracle's FP64 operator:
the solve stops at rtol in the library's operator, the two operators round
differently by a few eps per row (below 1e-13 of ||b|| at these sizes), so 2 rtol
bounds it."""
import sys

import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu

D, N, INF = 1, 2, 3
RTOL = 1e-11


@pytest.fixture(scope="module")
def ctx():
    from incflo_amd import mgx
    c = mgx.Context(0)
    yield c
    c.close()


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


NODAL = [  # cells, periodicity, lo, hi, kind, overset mask
    ((7, 9, 5), (1, 1, 1), (0, 0, 0), (0, 0, 0), "bicgcg", False),         # 315 nodes
    ((7, 7, 7), (0, 0, 0), (N, N, N), (N, N, N), "cg", False),             # 512, singular walls
    ((8, 8, 7), (1, 0, 1), (0, D, 0), (0, N, 0), "bicgcg", False),         # 504
    ((8, 6, 8), (0, 0, 0), (INF, N, N), (D, N, N), "bicgcg", False),       # 567: 4 per thread
    ((3, 60, 5), (1, 0, 0), (0, N, N), (0, D, N), "cg", True),             # 1098, columns along y
    ((15, 9, 7), (0, 0, 0), (INF, N, N), (D, N, N), "bicgcg", False),      # 1280
    ((17, 15, 13), (1, 1, 1), (0, 0, 0), (0, 0, 0), "bicgcg", False),      # 3315: 8 per thread
    ((15, 15, 15), (0, 0, 0), (D, N, N), (N, N, N), "cg", True),           # 4096
    ((12, 25, 9), (0, 0, 0), (INF, N, N), (D, N, N), "bicgcg", False),     # 3380: rows in memory
    ((10, 19, 18), (1, 0, 1), (0, N, 0), (0, D, 0), "cg", True),           # 3600
    ((10, 18, 17), (0, 0, 0), (N, N, N), (N, N, N), "bicgcg", False),      # 3762
    ((21, 19, 17), (0, 1, 0), (N, 0, D), (D, 0, N), "bicgcg", False),      # 7480: segments
    ((20, 4, 60), (0, 0, 1), (D, N, 0), (N, N, 0), "cg", True),            # 6300, columns along y
    ((30, 27, 25), (1, 1, 1), (0, 0, 0), (0, 0, 0), "bicgcg", False),      # 20250: beyond LDS
    ((32, 29, 23), (0, 0, 0), (INF, N, N), (D, N, N), "cg", True),         # 23760
    ((3, 130, 45), (1, 0, 0), (0, N, N), (0, D, N), "bicgcg", False),      # 18078, in LDS
]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,per,bclo,bchi,kind,masked", NODAL)
def test_nodal_bottom_of_every_size(ctx, orc, n, per, bclo, bchi, kind, masked, mixed):
    from incflo_amd import mgx
    _say(f"case nodal bottom {n} {kind} mask {masked} mixed {mixed}")
    ph = (1.0, 1.3, 0.9)
    g = orc.Geom.make(n, periodic=per, bclo=bclo, bchi=bchi, prob_hi=ph)
    rng = np.random.default_rng(sum(n))
    sigma = 1.0 + 0.5 * np.tanh(rng.standard_normal(g.cell_shape()))
    b = rng.standard_normal(g.node_shape())
    bxs = B.chop_domain(n, 64)
    P = mgx.NodalProjector(ctx, mgx.make_level(n, bxs, periodic=per, prob_hi=ph))
    P.setDomainBC(bclo, bchi)
    P.set_options(mgx.default_opts(bottom_solver=kind, max_coarsening_level=0, bottom_maxiter=400))
    P.set_sigma(ctx.array(B.to_boxed(sigma, bxs, 0)), 0)
    mask = np.ones(g.node_shape(), np.int32)
    if masked:
        mask[1, 1:3, 1:4] = 0
        flat = B.to_boxed(mask.astype(float), bxs, 0, nodal=True, periodic=per).astype(np.int32)
        P.setOversetMask(ctx.array(flat, np.int32))
    singular = not masked and all(per[d] or (bclo[d] != D and bchi[d] != D) for d in range(3))
    if singular:
        b -= b.mean()
    rd = ctx.array(B.to_boxed(b, bxs, 0, nodal=True, periodic=per))
    xd = ctx.array(B.field_size(bxs, 0, 1, True))
    info = P.solve(xd, 0, rd, 0, RTOL, mode=mgx.MODE_MIXED if mixed else mgx.MODE_FP64)
    x = B.from_boxed(xd.download(), bxs, 0, g.node_shape(), nodal=True)
    P.close()
    assert info.converged and info.nlevels == 1
    r = orc.nodal_residual(g, sigma, b, x) * mask
    assert np.max(np.abs(x[mask == 0]), initial=0.0) == 0.0
    assert np.max(np.abs(r)) <= 2 * RTOL * np.max(np.abs(b))
    if singular:
        assert abs(x.mean()) <= 1e-12 * np.max(np.abs(x))


MAC = [
    ((7, 9, 5), (1, 1, 1), (0, 0, 0), (0, 0, 0), "bicgcg"),     # 315 cells
    ((8, 8, 8), (1, 0, 1), (0, N, 0), (0, D, 0), "cg"),          # 512
    ((9, 19, 3), (0, 0, 0), (N, N, N), (D, N, N), "bicgcg"),     # 513: 2 per thread
    ((13, 11, 9), (0, 0, 0), (N, N, N), (N, N, N), "bicgcg"),    # 1287: 4 per thread
    ((17, 15, 13), (1, 1, 1), (0, 0, 0), (0, 0, 0), "cg"),       # 3315: rows in global memory
    ((21, 19, 17), (0, 1, 0), (N, 0, D), (D, 0, N), "bicgcg"),   # 6783: vectors too
    ((30, 27, 25), (1, 1, 1), (0, 0, 0), (0, 0, 0), "cg"),       # 20250: beyond LDS
]


@pytest.mark.parametrize("n,per,bclo,bchi,kind", MAC)
def test_mac_bottom_of_every_size(ctx, orc, n, per, bclo, bchi, kind):
    from incflo_amd import mgx
    _say(f"case mac bottom {n} {kind}")
    ph = (1.0, 1.3, 0.9)
    g = orc.Geom.make(n, periodic=per, bclo=bclo, bchi=bchi, prob_hi=ph)
    rng = np.random.default_rng(sum(n))
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
    P.set_options(mgx.default_opts(bottom_solver=kind, max_coarsening_level=0, bottom_maxiter=400))
    P.set_beta(*[ctx.array(B.faces_to_boxed(beta[d], bxs, 0, d)) for d in range(3)], ng=0)
    rd = ctx.array(B.to_boxed(b, bxs, 0, periodic=per))
    xd = ctx.array(B.field_size(bxs, 0, 1))
    info = P.solve(xd, 0, rd, 0, RTOL)
    x = B.from_boxed(xd.download(), bxs, 0, g.cell_shape())
    P.close()
    assert info.converged and info.nlevels == 1
    r = orc.mac_residual(g, beta, b, x)
    assert np.max(np.abs(r)) <= 2 * RTOL * np.max(np.abs(b))


EB = [((32, 16, 16), 0),  # 8976 nodes: rows and vectors in global memory
      ((32, 16, 16), 1),  # 1224: rows in global memory
      ((32, 16, 16), 2),  # 180
      ((16, 8, 6), 0),    # 918: rows of two nodes per thread in registers
      ((24, 12, 10), 0),  # 3250: rows in global memory, four nodes per thread
      ((50, 25, 15), 0)]  # 19890: beyond LDS


@pytest.mark.parametrize("n,levels", EB)
def test_eb_bottom_of_every_size(ctx, orc, n, levels):
    from incflo_amd import mgx
    _say(f"case eb bottom {n}, max_coarsening_level {levels}")
    ph, per, bclo, bchi = (2.0, 1.0, n[2] / n[1]), (0, 0, 1), (INF, N, 0), (D, N, 0)
    g = orc.Geom.make(n, periodic=per, bclo=bclo, bchi=bchi, prob_hi=ph)
    bxs = B.chop_domain(n, 16)
    P = mgx.NodalProjector(ctx, mgx.make_level(n, bxs, periodic=per, prob_hi=ph))
    P.setDomainBC(bclo, bchi)
    P.set_options(mgx.default_opts(max_coarsening_level=levels, bottom_maxiter=400))
    P.set_eb_cylinder(0.5, 0.5, 0.2)
    ct, mom = orc.eb_cylinder(g, 0.5, 0.5, 0.2)
    rng = np.random.default_rng(4)
    sigma = 0.5 + rng.random(g.cell_shape())
    mask = orc.eb_node_mask(g, ct).astype(bool)
    b = np.where(mask, rng.standard_normal(g.node_shape()), 0.0)
    P.set_sigma(ctx.array(B.to_boxed(sigma, bxs, 0)), 0)
    rd = ctx.array(B.to_boxed(b, bxs, 0, nodal=True, periodic=per))
    xd = ctx.array(B.field_size(bxs, 0, 1, True))
    info = P.solve(xd, 0, rd, 0, RTOL, 0.0, mode=mgx.MODE_FP64)
    x = B.from_boxed(xd.download(), bxs, 0, g.node_shape(), nodal=True)
    P.close()
    assert info.converged and info.nlevels == levels + 1
    r = np.where(mask, b - orc.eb_nodal_apply(g, ct, mom, sigma, x), 0.0)
    assert np.max(np.abs(r)) <= 2 * RTOL * np.max(np.abs(b))


# levels of 2 and 3 cells are made only with four sweeps or more per cycle:
# with fewer the cycle did not converge through them (49 cycles without)
@pytest.mark.parametrize("nu1,nu2", [(0, 1), (1, 0), (1, 2), (2, 2)])
def test_mac_few_sweeps_converge(ctx, nu1, nu2):
    from incflo_amd import mgx
    n = (36, 20, 12)
    _say(f"case mac {n} nu {nu1},{nu2}")
    ph = tuple(m / 20 for m in n)
    rng = np.random.default_rng(7)
    beta = [0.5 + rng.random((n[2] + (d == 2), n[1] + (d == 1), n[0] + (d == 0))) for d in range(3)]
    b = rng.standard_normal((n[2], n[1], n[0]))
    bxs = B.chop_domain(n, 64)
    P = mgx.MacProjector(ctx, mgx.make_level(n, bxs, periodic=(0, 0, 0), prob_hi=ph))
    P.setDomainBC((D, N, N), (N, D, N))
    P.set_options(mgx.default_opts(nu1=nu1, nu2=nu2, maxiter=200))
    P.set_beta(*[ctx.array(B.faces_to_boxed(beta[d], bxs, 0, d)) for d in range(3)], ng=0)
    xd = ctx.array(B.field_size(bxs, 0, 1))
    info = P.solve(xd, 0, ctx.array(B.to_boxed(b, bxs, 0)), 0, RTOL)
    P.close()
    assert info.converged and info.vcycles <= 60
