"""GPU test of the device memory that a solver handle takes, in level-sized FP64
arrays.  A level that cannot be halved is the bottom itself, and its workspace
follows the variant that solves it: 7 vectors and the multiplied one of the nodal
segments of columns (with the 15 or so of the handle and the solve; 64 MiB for
the kernel's scratch), 7 coefficients and 7 vectors of the cell-centred rows.  On levels that the V-cycle
smooths on tiles no residual is stored (128^3 cells: 20.0 arrays with one)."""
import ctypes as C

import numpy as np
import pytest

from incflo_amd import boxes as B

pytestmark = pytest.mark.gpu


def _free(ctx):
    from incflo_amd import mgx
    ctx.sync()
    free, total = C.c_size_t(), C.c_size_t()
    assert mgx.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("what,n,arrays,mib", [("nodal", 129, 24, 64), ("mac", 129, 31.6, 0),
                                               ("mac", 128, 19.4, 0)])
def test_solver_memory(what, n, arrays, mib):
    from incflo_amd import mgx
    print(f"case solver memory {what} {n}^3", flush=True)
    ctx = mgx.Context(0)
    bxs = B.chop_domain((n, n, n), 64)
    lev = mgx.make_level((n, n, n), bxs)
    x, b = ctx.array(n ** 3), ctx.array(np.random.default_rng(0).standard_normal(n ** 3))
    before = _free(ctx)
    P = mgx.NodalProjector(ctx, lev) if what == "nodal" else mgx.MacProjector(ctx, lev)
    # one cycle of one iteration: the memory is that of any solve
    P.set_options(mgx.default_opts(maxiter=1, bottom_maxiter=1))
    if what == "nodal":
        P.set_const_sigma(1.0)
    else:
        P.updateBeta(1.0)
    try:
        P.solve(x, 0, b, 0, 1e-30)
    except mgx.MgxError:
        pass
    used = before - _free(ctx)
    P.close()
    ctx.close()
    print(f"  {used / (8 * n ** 3):.1f} arrays")
    assert used <= arrays * 8 * n ** 3 + (mib << 20)
