"""GPU: the convolutions over many tiles (weights resident in registers) and few (output channels split).

A launch with at least two 16 x 8 tiles for every CU walks them with persistent workgroups, one form
for each number of 16-channel output groups (1-6) and of 32-channel input groups (1-3); the
others split their output channels over workgroups.  The batches here are copies of a few small
images, so that level 0 (and in the last shape level 1) has tiles enough while the reference
needs those images alone: the loss is a mean, so 2^k copies leave every gradient as it is (a
power of two scales BF16 values exactly) and every output repeats.  Widths give every group count in
both directions, shapes end inside a tile in x or y or have tiles that lie inside.
The networks and the tolerance for gradients are those of the weight-gradient test: sums that no
order of additions changes, 1e-3 per layer.  Outputs: the values of the last layer are FP32 sums of
equal BF16 operands, so 1e-5 relative to the largest.
"""
import numpy as np
import pytest

from test_gpu_wgrad import U, _case, _rel
from vtrace_amd import denoise as DN
from vtrace_amd import renderer as R

pytestmark = pytest.mark.gpu

NETS = [((16, 32, 48, 64, 96), (96, 16, 32, 64)), ((96, 64, 32, 16, 16), (16, 96, 48, 80)),
        ((48, 32, 32, 16, 32), (80, 48, 32, 32)), ((64, 48, 32, 32, 16), (64, 32, 32, 16)),
        ((80, 16, 32, 32, 16), (48, 16, 16, 16)), (DN.ENC, DN.DEC)]


@pytest.mark.parametrize("enc,dec", NETS)
@pytest.mark.parametrize("n,h,w,copies", [(2, 16, 16, 256), (1, 48, 80, 32)])
def test_convolutions_over_many_tiles(enc, dec, n, h, w, copies):
    d = DN.Denoiser(R.get_renderer(), enc=enc, dec=dec, seed=None)
    try:
        p, x, t = _case(d.layers, d.nparam, n, h, w)
        d.set_params(p)
        print(f"case: convolutions {copies} x {n}x{h}x{w} widths {enc} {dec}", flush=True)
        y, g, _ = d.grad(np.tile(x, (copies, 1, 1, 1)), np.tile(t, (copies, 1, 1, 1)))
        y = y.reshape(copies, n, h, w, 3)
        assert np.array_equal(y, np.broadcast_to(y[:1], y.shape))
        ref_y, _, ref = U.UNetRef(d.layers, enc, dec).loss_and_grads(p.astype(np.float64), x.astype(np.float64),
                                                                     t.astype(np.float64), bf16=True)
        assert np.abs(y[0] - ref_y).max() <= 1e-5 * np.abs(ref_y).max()
        for i, (cin, cout, wo, bo) in enumerate(d.layers):
            for a, b, what in ((wo, bo, "weights"), (bo, bo + cout, "biases")):
                err = _rel(g[a:b], ref[a:b])
                assert err < 1e-3, (i, cin, cout, what, err)
    finally:
        d.close()
