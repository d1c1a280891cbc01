"""GPU: the LBVH at the sizes where its build changes form, against the oracle's tree bit for bit.

Up to 512 instances one workgroup builds it (P = the power of two >= n threads), up to 4096 its boxes
are joined in one workgroup, up to 16384 its codes are sorted by counting; the sizes are one below,
at and above each line and around a wave.  Besides scattered instances, many at one place (equal
codes, told apart by index) and a power-of-two chain (a tree as deep as its codes are long).
"""
import numpy as np
import pytest

import oracle_ffi as O
from vtrace_amd import renderer as R
from vtrace_amd import scenes

pytestmark = pytest.mark.gpu


def _records(n, kind):
    rng = np.random.default_rng(n)
    size = rng.uniform(4.0, 90.0, (n, 3)).astype(np.float32)
    pos = rng.uniform(-3000.0, 3000.0, (n, 3)).astype(np.float32)
    if kind == "equal":
        pos[rng.random(n) < 0.8] = pos[0]
        size[:] = size[0]
    elif kind == "chain":
        pos[:] = 0.0
        size[:] = 6.0
        for i in range(n):
            pos[i, i % 3] = 8.0 * 2.0 ** ((i // 3) % 10)
    recs = np.zeros((n, 16), np.float32)
    recs[:, 0], recs[:, 5], recs[:, 10] = size[:, 0], size[:, 1], size[:, 2]
    recs[:, 12:15] = pos
    recs.view(np.uint32)[:, 15] = np.arange(n) % 3
    return recs


@pytest.mark.parametrize("kind,n", [("scattered", n) for n in (2, 4, 17, 63, 64, 65, 128, 129, 511, 512, 513, 1024, 4095,
                                                              4097, 16384, 16385)] +
                                   [("equal", n) for n in (5, 64, 300, 512, 3000, 5000)] +
                                   [("chain", n) for n in (7, 31, 512, 2000)])
def test_lbvh_at_the_edges_of_its_forms(kind, n):
    print(f"case: lbvh {kind} n={n}", flush=True)
    r = R.get_renderer()
    ids = [r.upload(scenes.Volume(scenes.gen_volume((8, 8, 8), k, 0.5), scenes.gen_palette(k))) for k in range(3)]
    recs = _records(n, kind)
    sent = recs.copy()
    sent.view(np.uint32)[:, 15] = np.array(ids, np.uint32)[np.arange(n) % 3]
    r.set_instances(sent)
    nodes, inst = r.lbvh()
    o_nodes, _, _ = O.lbvh(recs, 3)
    assert np.array_equal(nodes.view(np.uint32).reshape(-1, 8), o_nodes)
    # a refit with the same records keeps every box (it uses the build's order and parents)
    r.refit_instances(sent)
    again, _ = r.lbvh()
    assert np.array_equal(again.view(np.uint32).reshape(-1, 8), o_nodes)


@pytest.mark.parametrize("kind,n", [("scattered", 10239), ("scattered", 10240), ("scattered", 10241), ("equal", 10240),
                                    ("equal", 10241)])
def test_lbvh_where_counting_ends(kind, n):
    """The codes of up to 10240 instances are sorted by counting, of more by the radix sort."""
    test_lbvh_at_the_edges_of_its_forms(kind, n)
