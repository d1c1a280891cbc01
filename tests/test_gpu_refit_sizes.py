"""GPU: refits with moved instances at the sizes where the build that they go on from changes form.

A refit takes the leaves' order and the parents as the build left them (one workgroup up to 512 instances, boxes
joined in one workgroup up to 4096, codes sorted by counting up to 10240) and its counters from a launch of
its own.  After it the topology is the build's, a leaf's box is the oracle's for its moved instance,
and every inner box the union of its children's.  Two refits follow each other, the second one back to
where the build was: the tree is then the build's bit for bit.
"""
import numpy as np
import pytest

import oracle_ffi as O
from test_gpu_lbvh_sizes import _records
from vtrace_amd import renderer as R
from vtrace_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [("scattered", n) for n in (2, 63, 64, 65, 511, 512, 513, 4095, 4096, 4097, 8192, 8193,
                                                              10240, 10241, 16383, 16384, 16385)] +
                                   [("equal", 300), ("equal", 3000), ("chain", 31), ("chain", 512), ("chain", 2000)])
def test_refit_of_moved_instances(kind, n):
    print(f"case: refit {kind} n={n}", flush=True)
    r = R.get_renderer()
    ids = [r.upload(scenes.Volume(scenes.gen_volume((8, 8, 8), k, 0.5), scenes.gen_palette(k))) for k in range(3)]
    recs = _records(n, kind)

    def sent(a):
        b = a.copy()
        b.view(np.uint32)[:, 15] = np.array(ids, np.uint32)[np.arange(n) % 3]
        return b

    r.set_instances(sent(recs))
    before, _ = r.lbvh()
    moved = recs.copy()
    moved[:, 12:15] += np.random.default_rng(n).uniform(-400.0, 400.0, (n, 3)).astype(np.float32)
    r.refit_instances(sent(moved))
    after, inst = r.lbvh()
    assert np.array_equal(after["left"], before["left"]) and np.array_equal(after["right"], before["right"])
    inv, aabb, _, _ = O.instance_prep(moved, 3)
    leaf = after[n - 1:]
    assert np.array_equal(np.sort(leaf["left"]), np.arange(n))
    assert np.array_equal(leaf["lo"], aabb[leaf["left"], :3]) and np.array_equal(leaf["hi"], aabb[leaf["left"], 3:])
    assert not np.array_equal(leaf["lo"], before["lo"][n - 1:])
    inner, lft, rgt = after[:n - 1], after[after["left"][:n - 1]], after[after["right"][:n - 1]]
    assert np.array_equal(inner["lo"], np.minimum(lft["lo"], rgt["lo"]))
    assert np.array_equal(inner["hi"], np.maximum(lft["hi"], rgt["hi"]))
    assert np.array_equal(inst["inv"].view(np.uint32), inv.reshape(n, 4, 4)[:, :, :3].reshape(n, 12).view(np.uint32))
    r.refit_instances(sent(recs))
    assert np.array_equal(r.lbvh()[0].view(np.uint32), before.view(np.uint32))
