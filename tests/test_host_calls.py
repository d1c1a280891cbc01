"""CPU: the order of the library's HIP calls and what is left undone when one of them fails.

The library runs against a stand-in runtime (fake_hip.py): launches do nothing but are written down, and a
chosen call fails.
"""
import numpy as np
import pytest

import fake_hip


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fakehip"))


def _count(hip, what):
    return sum(what in line for line in hip.lines())


# ---- training: no update on gradients that are not there -----------------------------------
def train_with_a_failed_launch(hip, what, nth):
    from vtrace_amd import denoise, renderer
    net = denoise.Denoiser(renderer.get_renderer(), seed=1)
    rad, gbuf = np.ones((64, 64, 4), np.float32), np.ones((64, 64, 8), np.float32)
    net.add_frame(rad, gbuf, rad, 1)
    net.train(1, batch=1, crop=64)
    hip.clear()
    hip.fail(what, nth)
    with pytest.raises(renderer.RendererError):
        net.train(1, batch=1, crop=64)
    assert _count(hip, "FAILED") == 1
    assert _count(hip, "k_wgrad_reduce") == 0, hip.lines()
    hip.clear()
    net.train(1, batch=1, crop=64)   # the next step is a whole one again
    assert _count(hip, "k_wgrad_reduce") == 1


# a convolution's: the 20th and later are the backward pass's
@pytest.mark.parametrize("what,nth", [("k_lossE", 1), ("k_loss_sum", 1), ("k_pool_bwd", 1), ("k_pool_bwd", 4),
                                      ("k_conv3x3_split", 20), ("k_conv3x3_split", 37), ("k_conv3x3_wgrad", 1)])
def test_no_update_after_a_failed_launch(fake, what, nth):
    fake_hip.child(fake, "test_host_calls", "train_with_a_failed_launch", what, nth)
