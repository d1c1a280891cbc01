"""GPU: weight and bias gradients of every layer at the edges of the weight-gradient kernel's tiles.

The kernel walks 16 x 4 pixel tiles per image with a one-pixel halo, in blocks of 16 or 32 input
channels and 1-6 blocks of 16 output channels.  The shapes give images smaller than a tile (down to
one pixel at the lowest level), widths and heights that end inside a tile, one and several images,
and networks whose layers have every block count and input channels that end inside a block.
Every output channel of the networks here is half the sum of two input values, so a rounding to BF16
never depends on a summation order and no cascade of roundings runs through the layers (as random
weights have it, where two correct references come to differ by up to 10 %).  What is left is the
loss gradient, FP32 on the GPU and FP64 in the reference, which can round to the BF16 neighbour
(2^-8 of the value) on a few pixels in 10^4: two references that accumulate in FP64 and FP32 agree
to 2e-7 here.  Tolerance 1e-3 per layer; a wrong tile, tap or channel is off by more than 1e-2.
"""
import os
import sys

import numpy as np
import pytest

from vtrace_amd import denoise as DN
from vtrace_amd import renderer as R

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import unet_ref as U  # noqa: E402

pytestmark = pytest.mark.gpu

WIDE = ((16, 48, 80, 96, 96), (96, 80, 16, 64))


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def _case(layers, nparam, n, h, w):
    rng = np.random.default_rng(100 * n + h + w)
    p = np.zeros(nparam, np.float32)
    for cin, cout, wo, bo in layers:
        k = p[wo:wo + cout * 9 * cin].reshape(cout, 9, cin)
        for co in range(cout):   # two distinct taps, inputs spread over the channels that carry values
            taps = rng.choice(9, 2, replace=False)
            k[co, taps[0], (7 * co + 3) % min(cin, 11 if cin == 16 else cin)] = 0.5
            k[co, taps[1], (5 * co + 1) % min(cin, 11 if cin == 16 else cin)] = 0.5
        p[bo:bo + cout] = 0.125
    x = rng.normal(size=(n, h, w, 16)).astype(np.float32)
    x[..., 11:] = 0.0
    x[..., 0:3] *= 0.25
    t = np.abs(rng.normal(size=(n, h, w, 3))).astype(np.float32)
    return p, x, t


@pytest.mark.parametrize("n,h,w,widths", [(1, 16, 16, (DN.ENC, DN.DEC)), (3, 48, 80, (DN.ENC, DN.DEC)),
                                          (2, 16, 144, (DN.ENC, DN.DEC)), (1, 80, 32, WIDE), (5, 16, 48, WIDE)])
def test_weight_gradients_at_tile_edges(n, h, w, widths):
    enc, dec = widths
    d = DN.Denoiser(R.get_renderer(), enc=enc, dec=dec, seed=None)
    try:
        p, x, t = _case(d.layers, d.nparam, n, h, w)
        d.set_params(p)
        print(f"case: weight gradients {n}x{h}x{w} widths {enc} {dec}", flush=True)
        _, g, _ = d.grad(x, t)
        _, g2, _ = d.grad(x, t)
        assert np.array_equal(g.view(np.uint32), g2.view(np.uint32))   # a fixed order of sums
        _, _, ref = U.UNetRef(d.layers, enc, dec).loss_and_grads(p.astype(np.float64), x.astype(np.float64),
                                                                 t.astype(np.float64), bf16=True)
        for i, (cin, cout, wo, bo) in enumerate(d.layers):
            for a, b, what in ((wo, bo, "weights"), (bo, bo + cout, "biases")):
                assert np.linalg.norm(ref[a:b]) > 0.0
                err = _rel(g[a:b], ref[a:b])
                assert err < 1e-3, (i, cin, cout, what, err)
    finally:
        d.close()
