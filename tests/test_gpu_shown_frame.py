"""GPU: the shown frame's bytes at the sizes where their way to the host changes.

Frames of up to 4 MB (2^20 pixels) are encoded straight into page-locked memory, four pixels a thread,
larger ones on the device and copied.  Widths and heights leave 0-3 pixels for the last thread, one
pixel alone, and sit at and above the limit.  The bytes are those the radiance encodes to: the
smallest code whose upper sRGB threshold lies above the value, alpha rounded.
"""
import copy

import numpy as np
import pytest

from vtrace_amd import renderer as R
from vtrace_amd import scenes

pytestmark = pytest.mark.gpu


def _encode(rad):
    v = (np.arange(255) + 0.5) / 255.0
    thr = np.where(v <= 0.04045, v / 12.92, ((v + 0.055) / 1.055) ** 2.4).astype(np.float32)
    code = [np.searchsorted(thr, rad[..., k], side="right").astype(np.uint32) for k in (2, 1, 0)]
    a = np.clip(rad[..., 3] * np.float32(255.0) + np.float32(0.5), 0.0, 255.0).astype(np.uint32)
    return code[0] | code[1] << 8 | code[2] << 16 | a << 24


@pytest.mark.parametrize("width,height", [(1, 1), (2, 1), (3, 1), (5, 1), (67, 31), (320, 240), (1024, 1023), (1024, 1024),
                                          (1025, 1024)])
def test_shown_frame_bytes(width, height):
    sc = scenes.multi_volume_scene(count=3, n=32, world=160, seed=7, width=width, height=height, spp=1, max_bounces=0)
    p = copy.copy(sc.params)
    p.mode = 0
    sc.params = p
    print(f"case: shown frame {width}x{height}", flush=True)
    r = R.reset_renderer()
    R.load_scene(r, sc)
    for _ in range(2):
        r.render(sc.P, sc.C)
        assert np.array_equal(r.bgra8(), _encode(r.radiance()))
    small = np.zeros(width * height - 1, np.uint32)
    assert r.lib.vt_read_bgra8(small.ctypes.data, small.nbytes) != 0   # too small a buffer stays refused


@pytest.mark.parametrize("width,height", [(3, 1), (67, 31), (1024, 1024), (1025, 1024)])
def test_shown_frame_into_page_locked_memory(width, height):
    """The same bytes as into ordinary memory, the memory behind them untouched."""
    import torch

    sc = scenes.multi_volume_scene(count=3, n=32, world=160, seed=8, width=width, height=height, spp=1, max_bounces=0)
    r = R.reset_renderer()
    R.load_scene(r, sc)
    r.render(sc.P, sc.C)
    n = width * height
    mem = torch.full((n + 8,), -1, dtype=torch.int32, pin_memory=True).numpy()
    print(f"case: shown frame {width}x{height} into page-locked memory", flush=True)
    assert r.lib.vt_read_bgra8(mem.ctypes.data, 4 * n) == 0
    assert np.array_equal(mem[:n].view(np.uint32).reshape(height, width), r.bgra8()) and np.all(mem[n:] == -1)


@pytest.mark.parametrize("sky", [(float("nan"), float("inf"), -1.0), (0.0, -0.0, 1e30), (1.0, 0.99999994, float("-inf"))])
def test_shown_frame_of_extreme_radiance(sky):
    """NaN and what lies below the first threshold show as 0, what lies above the last as 255."""
    r = R.reset_renderer()
    r.set_params(scenes.RenderParams(6, 3, viewport_square=0, mode=1, sky=sky))
    r.render(scenes.perspective(scenes.FOV, 2.0), scenes.look_at((0.0, 0.0, 9.0), (0.0, 0.0, 0.0)))
    want = [0 if not v > 0.0 else 255 for v in sky]
    print(f"case: shown frame, sky {sky}", flush=True)
    got = r.bgra8()
    assert np.all(got == np.uint32(want[2] | want[1] << 8 | want[0] << 16 | 0xFF000000)), hex(int(got[0, 0]))
