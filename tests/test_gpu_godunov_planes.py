"""GPU test of the Godunov kernels' face-plane mapping and component counts:
planes that are no multiple of a 256-point run (one run only, a run and a
remainder, many), one, two and three components per launch, against the FP64
oracle at the round-off tolerance of the other Godunov tests."""
import numpy as np
import pytest

from incflo_amd import boxes as B
from test_gpu_godunov import _canon_faces, _faces_out, _field, ctx  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(8, 12, 6), (15, 17, 19), (63, 9, 10), (64, 7, 5)])
@pytest.mark.parametrize("nc", [1, 2, 3])
def test_godunov_planes(ctx, orc, n, nc):  # noqa: F811
    from incflo_amd import mgx
    print(f"case godunov planes {n} nc={nc}", flush=True)
    bxs = B.chop_domain(n, 64)
    vel = _field(n, 1)
    dt = 0.4 / max(n) / np.max(np.abs(vel))
    g = orc.Geom.make(n)
    A = mgx.Advection(ctx, mgx.make_level(n, bxs))
    um = _faces_out(ctx, bxs, n)
    A.extrap_vel_to_faces(ctx.array(B.to_boxed(vel, bxs, 3)), 3, dt, um[0], um[1], um[2], umac_ng=1)
    umac = orc.godunov_extrap_vel(g, vel, dt)
    for d in range(3):
        got, _ = _canon_faces(um[d], bxs, 1, d, n)
        assert np.max(np.abs(got - umac[d])) <= 1e-12 * np.max(np.abs(umac[d])), d
    cons = [1, 0, 1][:nc]
    sc = 1.0 + 0.3 * _field(n, 7)[:nc]
    umd = []
    for d in range(3):
        full = np.concatenate([umac[d], np.take(umac[d], [0], axis=2 - d)], axis=2 - d)
        umd.append(ctx.array(B.faces_to_boxed(full, bxs, 1, d)))
    conv = ctx.array(B.field_size(bxs, 1, nc))
    A.scalar_term(ctx.array(B.to_boxed(sc, bxs, 3)), 3, nc, umd[0], umd[1], umd[2], 1, dt, conv, 1,
                  iconserv=cons)
    st = orc.godunov_scalar_states(g, sc, umac, dt, iconserv=cons)
    cref = orc.scalar_advection(g, sc, umac, st, iconserv=cons)
    got = B.from_boxed(conv.download(), bxs, 1, (n[2], n[1], n[0]), ncomp=nc)
    A.close()
    assert np.max(np.abs(got - cref)) <= 1e-11 * np.max(np.abs(cref))
