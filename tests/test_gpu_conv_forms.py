"""GPU: the output layer's gradient has the same bits in both forms of the convolution.

Its 8 channels fill a quarter of a K step: a step holds four taps in the form with the output channels
split (few tiles: one image), one tap and zeros in the one with the weights in registers (many: 512
images).  The weights let taps cancel: a large one, its negative and a small one, in places of their
own for every input channel, so that sums of other groups of taps round elsewhere (were the four taps
of a step added as one exact sum, about one channel in eight would differ).  The gradient reaches
the layer below in two rows of one image only; everywhere else the predicted irradiance is at its clamp
and passes none.  512 is a power of two, so the two gradients differ by exactly that factor, and all that
is not zero lies in one tile of the weight gradient, so its sum has one order.
"""
import numpy as np
import pytest

from vtrace_amd import denoise as DN
from vtrace_amd import renderer as R

pytestmark = pytest.mark.gpu

COPIES = 512


@pytest.mark.parametrize("width", [16, 32, 48, 64, 80, 96])   # outputs of the launch: 1 to 6 groups of 16
def test_gradient_of_eight_channels_in_both_forms(width):
    d = DN.Denoiser(R.get_renderer(), enc=(16, 16, 16, 16, 16), dec=(width, 16, 16, 16), seed=None)
    try:
        rng = np.random.default_rng(width)
        p = np.zeros(d.nparam, np.float32)
        for cin, cout, wo, bo in d.layers:
            p[bo:bo + cout] = 0.125   # activations: 0.125 everywhere
        cin, cout, wo, bo = d.layers[18]
        p[bo:bo + cout] = 0.0
        k = p[wo:wo + cout * 9 * cin].reshape(cout, 9, cin)
        for ci in range(cin):
            big, minus, small = rng.choice(9, 3, replace=False)
            k[0, big, ci], k[0, minus, ci] = 1024.0, -1024.0
            k[0, small, ci] = 2.0 ** -rng.integers(6, 12) * (1 + rng.integers(0, 128) / 128)
        d.set_params(p)
        x = np.zeros((1, 16, 16, 16), np.float32)
        x[..., 0:3] = 2000.0               # past the clamp, whatever the network adds
        x[0, 5:7, 1:15, 0:3] = 0.5         # but here
        x[..., 3:6] = 0.7
        t = np.full((1, 16, 16, 3), 1.3, np.float32)
        rest = np.full((COPIES - 1, 16, 16, 16), 2000.0, np.float32)
        print(f"case: gradient of 8 channels to {width}", flush=True)
        y1, g1, _ = d.grad(x, t)
        y2, g2, _ = d.grad(np.concatenate([x, rest]), np.broadcast_to(t, (COPIES, 16, 16, 3)))
        assert np.array_equal(y1[0].view(np.uint32), y2[0].view(np.uint32))
        for i in (17, 18):
            cin, cout, wo, bo = d.layers[i]
            a, b = g1[wo:bo + cout], g2[wo:bo + cout] * np.float32(COPIES)
            assert np.count_nonzero(a) > a.size // (4 if i == 17 else 60)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (i, np.abs(a - b).max(), np.abs(a).max())
    finally:
        d.close()
