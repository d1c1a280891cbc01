"""GPU: nearer subtrees first against the fixed order.

A counted launch visits the tree in the fixed order its counters are defined by, the others visit
nearer subtrees first and enter no instance behind a hit.  Which instance wins does not depend on the
order, so both give the same bits, and the oracle's hits.  The scenes make order matter: boxes that
overlap and contain each other, equal boxes (ties go to the lower index), an eye inside some of them,
trees on both sides of the 127 nodes kept in LDS, a single leaf, and one deeper than the stack in LDS.
"""
import copy

import numpy as np
import pytest

import oracle_ffi as O
from parity_util import assert_hits_equal, gpu_render, radiance_error
from test_gpu_parity import _deep_chain_scene
from vtrace_amd import scenes

pytestmark = pytest.mark.gpu

REL_TOL = 1e-5   # FP32 radiance against the FP64 replay, as the other parity tests


def _overlapping(count, seed):
    rng = scenes.Rng(seed)
    vols = [scenes.Volume(scenes.gen_volume((16, 16, 16), 10 * seed + k, 0.05 + 0.1 * k), scenes.gen_palette(seed + k))
            for k in range(3)]
    side = 12.0 * count ** (1.0 / 3.0)   # about as much box as space
    recs = []
    for i in range(count):
        if i % 5 == 4:
            recs.append(recs[-1].copy())   # an equal box: a tie
        else:
            c = tuple(rng.uniform(-side, side) / 2.0 for _ in range(3))
            recs.append(scenes.instance_record(scenes.model_matrix(c, rng.uniform(8.0, 32.0)), i % 3))
    p = scenes.RenderParams(150, 110, viewport_square=0, mode=2, spp=2, max_bounces=2, jitter=1, seed=seed)
    return scenes.Scene(vols, np.stack(recs).astype(np.float32), scenes.perspective(scenes.FOV, 150 / 110),
                        scenes.look_at((-0.7 * side - 20.0, 0.3 * side, -0.6 * side), (0.0, 0.0, 0.0)), p,
                        name=f"overlapping_{count}")


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("count", [1, 2, 17, 64, 65, 300, 0])
def test_nearer_first_equals_fixed_order(count, mode):
    sc = _overlapping(count, 3 + count) if count else _deep_chain_scene()
    if mode != 2:
        p = copy.copy(sc.params)
        p.mode, p.spp, p.max_bounces = mode, 1, 0
        sc.params = p
    print(f"case: {sc.name} mode={mode}", flush=True)
    hits, rad, _ = gpu_render(sc)
    f_hits, f_rad, _ = gpu_render(sc, stats=True)
    assert np.array_equal(hits.view(np.uint8), f_hits.view(np.uint8))
    assert np.array_equal(rad.view(np.uint32), f_rad.view(np.uint32))
    o_hits, o_rad, _ = O.render(sc, use_bvh=True)
    assert_hits_equal(hits, o_hits, sc.name)
    assert (hits["inst"] != 0xFFFFFFFF).any()
    if mode == 0:
        assert np.array_equal(rad.view(np.uint32), o_rad.view(np.uint32))
    else:
        assert radiance_error(rad, o_rad)[0] <= REL_TOL
