"""GPU: frames of every mode one after another on the same wavefront block.

Work and queue counters are zeroed by the launch that ends a frame (mode 0: one of two counter slots
by the next mode-0 frame), so a frame may depend on the one before it: modes in every order, sizes
that outgrow the block (a new one is zeroed first), one stream and several chunks, with the serving
loop's sub-batches between them.  Every frame equals the one a fresh library renders, bit for bit.
"""
import copy

import numpy as np
import pytest

from vtrace_amd import renderer as R
from vtrace_amd import scenes, serving

pytestmark = pytest.mark.gpu

#: mode, width, height, samples, bounces, chunks (0: the default)
FRAMES = [(0, 64, 48, 1, 0, 0), (2, 64, 48, 2, 3, 0), (0, 320, 240, 1, 0, 0), (0, 64, 48, 1, 0, 0), (1, 320, 240, 1, 0, 0),
          (2, 200, 160, 3, 2, 3), (2, 64, 48, 2, 3, 0), (1, 64, 48, 1, 0, 0), (0, 320, 240, 1, 0, 0),
          (2, 333, 250, 2, 4, 2), (2, 200, 160, 3, 2, 3), (0, 64, 48, 1, 0, 0)]


def _scene():
    return scenes.multi_volume_scene(count=3, n=32, world=160, seed=7, width=64, height=48, spp=1, max_bounces=1)


def _frame(r, sc, f):
    mode, w, h, spp, bounces, chunks = f
    p = copy.copy(sc.params)
    p.mode, p.width, p.height, p.spp, p.max_bounces = mode, w, h, spp, bounces
    r.set_params(p)
    assert r.lib.vt_set_frame_split(chunks) == 0
    r.render(sc.P, sc.C)
    return r.hits().copy(), r.radiance().copy()


@pytest.mark.parametrize("blocks", [0, 5])   # 5 workgroups: most tiles come from the counters
def test_frames_after_each_other(blocks):
    sc = _scene()
    want = []
    for f in dict.fromkeys(FRAMES):
        r = R.reset_renderer()
        R.load_scene(r, sc)
        want.append(_frame(r, sc, f))
    want = dict(zip(dict.fromkeys(FRAMES), want))
    r = R.reset_renderer()
    R.load_scene(r, sc)
    loop = serving.ServingLoop(r, max_slots=4, max_work=1 << 20)
    loop.add_scene(sc.records)
    try:
        assert r.lib.vt_set_persistent_blocks(blocks) == 0
        served = None
        for k, f in enumerate(FRAMES + FRAMES[::-1]):
            print(f"case: frame {k} {f} blocks={blocks}", flush=True)
            hits, rad = _frame(r, sc, f)
            assert np.array_equal(hits.view(np.uint8), want[f][0].view(np.uint8))
            assert np.array_equal(rad.view(np.uint32), want[f][1].view(np.uint32))
            q = serving.Request(0, 96, 64, 2, sc.P, sc.C, seed=3, max_bounces=4)
            rid, done = loop.submit(q), []
            while rid not in done:
                done += list(loop.step())
            img = loop.read(rid, 96, 64)
            assert served is None or np.array_equal(img, served)
            served = img
    finally:
        loop.close()
        r.lib.vt_set_persistent_blocks(0)
        r.lib.vt_set_frame_split(0)
