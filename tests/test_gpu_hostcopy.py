"""GPU: copies to and from ordinary host memory, at the sizes where they change form (4 MB out, 24 MB in,
chunks of 512 KB to 2 MB over several threads): the bytes equal those of a copy through page-locked
memory, also when two threads read at once and after the renderer was reset."""
import threading

import numpy as np
import pytest
import torch

from vtrace_amd import renderer as R
from vtrace_amd import scenes

pytestmark = pytest.mark.gpu


def _frame(r, w, h):
    sc = scenes.multi_volume_scene(count=2, n=32, world=128, seed=w + h, width=w, height=h, spp=1, max_bounces=1)
    R.load_scene(r, sc)
    r.render(sc.P, sc.C)
    return r.radiance(out=torch.empty((h, w, 4), pin_memory=True).numpy()).copy()


# 16 B a pixel: just under 4 MB, 4 MB, a little more, an odd size of many chunks
@pytest.mark.parametrize("w,h", [(512, 511), (512, 512), (13799, 19), (1237, 1021)])
def test_radiance_read_into_ordinary_memory(w, h):
    r = R.reset_renderer()
    print(f"case: radiance {w}x{h} = {16 * w * h} bytes", flush=True)
    want = _frame(r, w, h)
    assert np.array_equal(r.radiance().view(np.uint32), want.view(np.uint32))
    raw = np.full(16 * w * h + 17, 0xA5, np.uint8)   # a destination at an odd address, ends untouched
    off = 4 - raw.ctypes.data % 4
    out = raw[off:off + 16 * w * h].view(np.float32).reshape(h, w, 4)
    r.radiance(out=out)
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    assert np.all(raw[:off] == 0xA5) and np.all(raw[off + 16 * w * h:] == 0xA5)


def test_two_threads_read_at_once():
    r = R.reset_renderer()
    want = _frame(r, 1000, 700)
    got = [None] * 2

    def read(k):
        for _ in range(5):
            got[k] = r.radiance()

    ts = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert all(np.array_equal(g.view(np.uint32), want.view(np.uint32)) for g in got)


@pytest.mark.parametrize("d", [191, 192, 211, 383, 384, 421])   # 256 x 256 x d bytes around 12 and 24 MB
def test_volume_round_trip(d):
    r = R.reset_renderer()
    idx = scenes.gen_volume((256, 256, d), 3, 0.3)
    tid = r.upload(scenes.Volume(idx, scenes.gen_palette(3)))
    dense = r.volume_dense(tid)
    ax = [np.floor((np.arange(n, dtype=np.float32) / np.float32(n)) * np.float32(n)).astype(np.int64).clip(0, n - 1)
          for n in idx.shape]
    want = idx[np.ix_(*ax)]   # the texel a voxel samples (nearest)
    occ = want != 0
    assert dense.shape == idx.shape and np.array_equal(dense[occ], want[occ]) and not np.any(dense[~occ])


# sizes whose last chunk, and whose last 64 bytes, are not whole
@pytest.mark.parametrize("w,h,d", [(301, 293, 289), (5, 65535, 77), (4097, 4099, 3)])
def test_volume_of_an_odd_size_round_trip(w, h, d):
    r = R.reset_renderer()
    rng = np.random.default_rng(w)
    idx = rng.integers(0, 3, (d, h, w), dtype=np.uint8)
    tid = r.upload(scenes.Volume(idx, scenes.gen_palette(3)))
    dense = r.volume_dense(tid)
    ax = [np.floor((np.arange(n, dtype=np.float32) / np.float32(n)) * np.float32(n)).astype(np.int64).clip(0, n - 1)
          for n in idx.shape]
    want = idx[np.ix_(*ax)]
    occ = want != 0
    assert dense.shape == idx.shape and np.array_equal(dense[occ], want[occ]) and not np.any(dense[~occ])
