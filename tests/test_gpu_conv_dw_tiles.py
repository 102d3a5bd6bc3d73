"""GPU test of the convolution's weight gradient at the edges of its 4 x 4 x 4
voxel tiles and channel blocks (32, 16 or 8 input and 32 or 16 output channels
per workgroup): sizes that are no multiple of 4 and below it, wrapped and
padded, several samples and more tiles than voxel ranges.  Same bound as the
other convolution tests: FP32 sums of products of BF16 operands, 2e-5 of the
sum of the terms' magnitudes."""
import numpy as np
import pytest

from incflo_amd import boxes as B  # noqa: F401  (the package under test)

pytestmark = pytest.mark.gpu

CASES = [  # cin, cout, (batch, nz, ny, nx), periodic
    (8, 16, (1, 1, 2, 3), (1, 1, 1)),
    (8, 32, (2, 4, 4, 4), (0, 1, 0)),
    (16, 16, (3, 12, 10, 9), (1, 0, 1)),
    (24, 16, (1, 5, 4, 6), (1, 1, 1)),
    (48, 32, (2, 6, 8, 5), (0, 0, 0)),
    (32, 16, (1, 8, 7, 8), (1, 1, 1)),
    (96, 96, (1, 4, 2, 4), (1, 1, 1)),
    (16, 16, (1, 40, 40, 40), (1, 1, 1)),  # 1000 tiles over 768 ranges
]


@pytest.mark.parametrize("cin,cout,shape,per", CASES)
def test_weight_gradient_tiles(orc, cin, cout, shape, per):
    from incflo_amd import mgx
    print(f"case conv dw cin={cin} cout={cout} shape={shape} per={per}", flush=True)
    ctx = mgx.Context(0)
    rng = np.random.default_rng(cin + cout + sum(shape))
    x = rng.standard_normal(shape + (cin,)).astype(np.float32)
    w = np.zeros((cout, 27 * cin), np.float32)
    g = rng.standard_normal(shape + (cout,)).astype(np.float32)
    dwd = ctx.array(cout * 27 * cin, np.float32)
    dbd = ctx.array(cout, np.float32)
    mgx.conv3d_backward(ctx, ctx.array(x.ravel(), np.float32), ctx.array(w.ravel(), np.float32),
                        ctx.array(g.ravel(), np.float32), None, dwd, dbd, shape, cin, cout, periodic=per)
    x64, g64, w64 = x.astype(np.float64), g.astype(np.float64), w.astype(np.float64)
    _, dw, db = orc.conv3d_backward(x64, w64, g64, periodic=per, bf16=True)
    _, mag, mdb = orc.conv3d_backward(np.abs(x64), w64, np.abs(g64), periodic=per, bf16=True)
    got = dwd.download().reshape(dw.shape)
    gb = dbd.download()
    ctx.close()
    assert np.all(np.abs(got - dw) <= 2e-5 * mag + 1e-30)
    assert np.all(np.abs(gb - db) <= 1e-5 * mdb + 1e-30)
