"""GPU: requests of different bounce counts in one serving loop.

A batch is launched as deep as its longest paths, and a replayed graph as deep as the loop's
max_bounces; every request still ends after its own count: its image equals a render by itself bit
for bit, also after other requests have left their path state behind.
"""
import numpy as np
import pytest

from test_gpu_serving import _plain, _setup
from vtrace_amd import renderer as R
from vtrace_amd import scenes, serving

pytestmark = pytest.mark.gpu


def _requests(bounces, size):
    rng = scenes.Rng(31)
    out = []
    for i, b in enumerate(bounces):
        sc = i % 3
        n = (32, 64, 48)[sc]
        w, h = size[0] + 13 * i, size[1] - 7 * i
        eye, target = scenes.orbit_camera(rng, (0.0, 0.0, 0.0), 1.3 * n, 2.0)
        out.append(serving.Request(sc, w, h, 2 + i % 3, scenes.perspective(scenes.FOV, w / h),
                                   scenes.look_at(eye, target), seed=40 + i, max_bounces=b,
                                   sun_dir=scenes.sun_direction(rng)))
    return out


# one stream, several, and a request alone in its batch
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("bounces,size,streams", [((4, 0, 2, 1, 3), (96, 80), 1), ((1, 4, 0, 2), (330, 250), 4),
                                                  ((1,), (64, 64), 1), ((0, 0), (40, 40), 1)])
def test_each_request_ends_after_its_own_bounces(graph, bounces, size, streams):
    r = R.reset_renderer()
    _, recs = _setup(r)
    reqs = _requests(bounces, size)
    print(f"case: serving bounces {bounces} {size} graph {graph} streams {streams}", flush=True)
    loop = serving.ServingLoop(r, max_slots=8, spp_chunk=2, memory_budget=128 << 20, max_work=1 << 20, max_bounces=4,
                               use_graph=graph, policy=serving.ROUND_ROBIN, pipeline=2, streams=streams)
    for rc in recs:
        loop.add_scene(rc)
    loop.run_all(_requests((4,) * len(bounces), size))   # deeper paths before
    got = loop.run_all(reqs)
    loop.close()
    for i, q in enumerate(reqs):
        want, _ = _plain(r, recs, q)
        assert np.array_equal(got[i].view(np.uint32), want.view(np.uint32)), f"request {i}, {q.max_bounces} bounces"
