"""GPU: the split of a launch's work between tiles kept for its waves and tiles fetched from counters.

A one-stream launch keeps one 64-item tile for each of its waves (4 per workgroup) and hands out
the rest by per-part counters, so the sizes that matter are tile counts just below, at and above
the waves of a part, workgroup counts that leave parts empty (fewer than 8), and a launch that is
smaller than the persistent grid.  Hits, mode-0 colour and radiance against the oracle.
"""
import copy
import sys

import numpy as np
import pytest

import oracle_ffi as O
from parity_util import assert_hits_equal, radiance_error
from vtrace_amd import renderer as R
from vtrace_amd import scenes

pytestmark = pytest.mark.gpu

REL_TOL = 1e-5   # FP32 radiance against the FP64 replay, as the other parity tests


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("width,height,blocks", [
    (5, 3, 0),        # one tile, most of it outside the frame
    (64, 32, 1),      # 32 tiles, one workgroup: parts 1-7 have no waves
    (64, 32, 7),      # part 7 has none
    (64, 64, 8),      # 64 tiles: 8 a part, 4 waves a part
    (72, 64, 9),      # 72 tiles, a second workgroup in part 0 only
    (64, 32, 8),      # 4 tiles a part: exactly its waves
    (67, 45, 0),      # ragged, far below the persistent grid
])
def test_kept_and_fetched_tiles(width, height, blocks, mode):
    sc = scenes.multi_volume_scene(count=3, n=32, world=160, seed=7, width=width, height=height,
                                   spp=3 if mode == 2 else 1, max_bounces=2)
    p = copy.copy(sc.params)
    p.mode = mode
    sc.params = p
    print(f"case: {width}x{height} blocks={blocks} mode={mode}", flush=True)
    sys.stdout.flush()
    r = R.reset_renderer()
    R.load_scene(r, sc)
    try:
        assert r.lib.vt_set_persistent_blocks(blocks) == 0
        r.render(sc.P, sc.C)
        hits, rad = r.hits(), r.radiance()
    finally:
        r.lib.vt_set_persistent_blocks(0)
    o_hits, o_rad, _ = O.render(sc)
    assert_hits_equal(hits, o_hits, f"{width}x{height} blocks={blocks} mode={mode}")
    if mode == 0:
        assert np.array_equal(rad.view(np.uint32), o_rad.view(np.uint32))
    else:
        assert radiance_error(rad, o_rad)[0] <= REL_TOL
