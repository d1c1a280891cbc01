"""GPU: every form of the convolution with resident weights on images of several tiles that end inside a tile.

128 copies of a 48 x 80 image: its level 1, 24 x 40 pixels, has 3 x 3 tiles of 16 x 8 (up to 64 output
channels) or 3 x 2 of 16 x 16 (80 and 96) and ends inside a tile in x, the latter in y too; with 256 CUs
both are tiles enough.  Halos there lie in neighbouring tiles on every side.  The networks' level-1
widths give every pair of output and input groups that the form takes, forward and backward, with and
without the mask of the layer below (level 0 ends with a tile, its last layer is the one that
writes FP32).  Networks and tolerances are those of test_gpu_conv_tiles.py, where the reasons stand: values that no order of
sums changes, 1e-3 per layer for gradients, 1e-5 of the largest output.
"""
import numpy as np
import pytest

from test_gpu_wgrad import U, _case, _rel
from vtrace_amd import denoise as DN
from vtrace_amd import renderer as R

pytestmark = pytest.mark.gpu

# encoder widths of levels 0-2, decoder widths of levels 0-2; 16 below
NETS = [((64, 32, 16), (16, 48, 64)), ((80, 16, 32), (64, 16, 32)), ((80, 64, 16), (64, 48, 16)),
        ((16, 48, 16), (64, 32, 48)), ((80, 32, 32), (80, 16, 64)), ((64, 48, 32), (80, 64, 48)),
        ((96, 16, 16), (64, 96, 48)), ((32, 96, 16), (80, 64, 96)), ((48, 80, 16), (96, 48, 80)),
        ((16, 96, 32), (96, 48, 80)), ((96, 32, 16), (80, 96, 16)), ((16, 64, 32), (64, 64, 16)),
        ((32, 48, 16), (32, 80, 16)), ((32, 80, 16), (48, 80, 64)), ((16, 80, 16), (48, 80, 32)),
        ((32, 64, 16), (96, 16, 16)), ((48, 48, 32), (96, 32, 16)), ((80, 48, 32), (64, 16, 16)),
        ((48, 64, 16), (64, 32, 16)), ((96, 48, 32), (96, 48, 16)), ((64, 96, 32), (64, 96, 80)),
        ((48, 96, 16), (64, 32, 16)), ((64, 80, 32), (16, 64, 32)), ((96, 64, 32), (48, 48, 32)),
        ((64, 64, 32), (96, 16, 80))]
COPIES, H, W = 128, 48, 80


@pytest.mark.parametrize("enc,dec", NETS)
def test_images_that_end_inside_a_tile(enc, dec):
    enc, dec = enc + (16, 16), dec + (16,)
    d = DN.Denoiser(R.get_renderer(), enc=enc, dec=dec, seed=None)
    try:
        p, x, t = _case(d.layers, d.nparam, 1, H, W)
        d.set_params(p)
        print(f"case: convolutions {COPIES} x {H}x{W} widths {enc} {dec}", flush=True)
        y, g, _ = d.grad(np.tile(x, (COPIES, 1, 1, 1)), np.tile(t, (COPIES, 1, 1, 1)))
        assert np.array_equal(y, np.broadcast_to(y[:1], y.shape))
        ref_y, _, ref = U.UNetRef(d.layers, enc, dec).loss_and_grads(p.astype(np.float64), x.astype(np.float64),
                                                                     t.astype(np.float64), bf16=True)
        assert np.abs(y[0] - ref_y[0]).max() <= 1e-5 * np.abs(ref_y).max()
        for i, (cin, cout, wo, bo) in enumerate(d.layers):
            for a, b, what in ((wo, bo, "weights"), (bo, bo + cout, "biases")):
                err = _rel(g[a:b], ref[a:b])
                assert err < 1e-3, (i, cin, cout, what, err)
    finally:
        d.close()
