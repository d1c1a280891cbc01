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


# ---- instance records: the GPU reads the caller's buffer in place, so it is handed out again when that is over ----
def commit_and_reopen(hip, n, refit, fail):
    from vtrace_amd import renderer
    r = renderer.get_renderer()
    recs = np.zeros((n, 16), np.float32)
    r.set_instances(recs)
    hip.clear()
    if fail:
        hip.fail(fail)
    recs[:, 12] = 1 + np.arange(n)
    if fail:
        with pytest.raises(renderer.RendererError):
            (r.refit_instances if refit else r.set_instances)(recs)
        assert _count(hip, "FAILED") == 1
    else:
        (r.refit_instances if refit else r.set_instances)(recs)
    calls = [c for c in hip.lines() if c.startswith(("launch", "record", "attribute"))]
    hip.clear()
    assert r.lib.start_update_instances(n)
    waits = [c.split()[2] for c in hip.lines() if c.startswith("sync event")]
    reads = [k for k, c in enumerate(calls) if "k_instance_prep" in c or "k_lbvh_one" in c]
    assert len(reads) == 1 and len(waits) == 1
    # behind the launch that reads them, right behind it where much follows
    marks = [k for k, c in enumerate(calls) if f"record event {waits[0]}" in c]
    assert len(marks) == 1 and marks[0] > reads[0], calls
    assert marks[0] == reads[0] + 1 or (refit and n <= 8192), calls


@pytest.mark.parametrize("n,refit,fail", [(1, False, None), (300, False, None), (3000, False, None), (9000, False, None),
                                          (40000, False, None), (5, True, None), (3000, True, None), (9000, True, None),
                                          # a later launch, or the permission for its LDS, fails
                                          (3000, False, "k_karras"), (4000, False, "attribute"), (40000, False, "k_sort_hist"),
                                          (3000, True, "k_refit"), (9000, True, "k_refit")])
def test_records_are_free_once_they_are_read(fake, n, refit, fail):
    fake_hip.child(fake, "test_host_calls", "commit_and_reopen", n, refit, fail)


# ---- a tree that could not be built is not traced ----------------------------------------------
def commit_fails(hip, n, fail):
    from vtrace_amd import renderer
    r = renderer.get_renderer()
    r.set_instances(np.ones((3, 16), np.float32))
    assert r.lib.vt_instance_count() == 3
    r.lib.start_update_instances(n)
    hip.fail(fail)
    assert r.lib.end_update_instances(n) == -1 and _count(hip, "FAILED") == 1
    assert r.lib.vt_instance_count() == 0
    assert r.lib.vt_read_lbvh(None, 0, None, 0) == -1
    r.set_instances(np.ones((n, 16), np.float32))
    assert r.lib.vt_instance_count() == n


# memory for the larger tree, a launch in the middle of a build, the copy of the tree's depth behind it
@pytest.mark.parametrize("n,fail", [(2000, "malloc"), (2000, "copy out"), (2000, "k_karras"), (40000, "k_sort_scan"), (2, "k_lbvh_one")])
def test_no_instances_after_a_failed_build(fake, n, fail):
    fake_hip.child(fake, "test_host_calls", "commit_fails", n, fail)


# ---- reading the shown frame: into any memory that a copy takes, and every failure has a text ------
def read_shown(hip, kind, width, height, fail=None):
    import ctypes

    from vtrace_amd import renderer, scenes
    r = renderer.get_renderer()
    r.set_params(scenes.RenderParams(width, height, mode=0))
    r.render(scenes.perspective(1.0, 1.0), scenes.look_at((0.0, 0.0, 9.0), (0.0, 0.0, 0.0)))
    n = width * height * 4
    mem = np.zeros(n, np.uint8)
    dst = {"ordinary": lambda: mem.ctypes.data, "page_locked": lambda: hip.page_locked(n),
           "device": lambda: hip.device(n)}[kind]()
    r.lib.vt_read_bgra8(dst, n)   # (what is allocated on first use)
    hip.clear()
    if fail:
        r.lib.vt_read_bgra8(None, n)
        before = r.error()
        hip.fail(fail)
        assert r.lib.vt_read_bgra8(dst, n) == -1 and _count(hip, "FAILED") == 1
        assert r.error() != before and r.error().startswith("read-back")
        return
    assert r.lib.vt_read_bgra8(dst, n) == 0
    copies = [c for c in hip.lines() if c.startswith("copy")]
    if kind == "ordinary" and n <= 4 << 20:
        assert copies == [], copies
    elif kind != "ordinary":   # by the copy engine, into the caller's memory
        assert len(copies) == 1 and ctypes.c_void_p(dst).value == int(copies[0].split()[2], 16), copies


@pytest.mark.parametrize("kind", ["ordinary", "page_locked", "device"])
@pytest.mark.parametrize("width,height", [(64, 48), (1024, 1024), (1025, 1024)])
def test_shown_frame_into_any_memory(fake, kind, width, height):
    fake_hip.child(fake, "test_host_calls", "read_shown", kind, width, height)


@pytest.mark.parametrize("kind,fail", [("ordinary", "k_encode_srgb8"), ("ordinary", "sync stream"),
                                       ("page_locked", "k_encode_srgb8"), ("page_locked", "copy out")])
def test_failed_read_of_the_shown_frame_says_so(fake, kind, fail):
    fake_hip.child(fake, "test_host_calls", "read_shown", kind, 64, 48, fail)


# ---- a captured launch sequence: nothing has run, so nothing counts as zeroed by it --------------------------
def serve_from_a_graph(hip):
    from vtrace_amd import renderer, scenes, serving
    loop = serving.ServingLoop(renderer.get_renderer(), memory_budget=1 << 22, max_work=1 << 14, streams=1, pipeline=1)
    loop.add_scene(np.ones((1, 16), np.float32))
    q = serving.Request(0, 32, 32, 1, scenes.perspective(1.0, 1.0), scenes.look_at((0.0, 0.0, 9.0), (0.0, 0.0, 0.0)), seed=1)
    for k in range(3):
        loop.submit(q)
        if k == 2:
            hip.fail("graph ")   # a replay that could not be queued leaves the counters in doubt
        hip.clear()
        try:
            loop.step()
        except renderer.RendererError:
            assert k == 2
        calls = [c.split(" grid")[0] for c in hip.lines() if c.startswith(("launch", "capture", "graph"))]
        names = ["graph" if c.startswith("graph") else c for c in calls]
        assert not any("capture" in c and ("k_accumulate" in c or "k_zero_counters" in c) for c in names), names
        run = [c for c in names if not c.startswith("capture")]
        if k == 0:   # new counters are zeroed, then the sequence runs and ends with the accumulation
            assert len(run) == 3 and "k_zero_counters" in run[0] and run[1] == "graph" and "k_accumulate" in run[2], run
            assert sum(c.startswith("capture") for c in names) == 6
        elif k == 1:
            assert len(run) == 2 and run[0] == "graph" and "k_accumulate" in run[1], run
    hip.lib.hipGetLastError()
    loop.submit(q)
    hip.clear()
    loop.step()
    assert _count(hip, "k_zero_counters") == 1


def test_captured_sequences_leave_the_counters_to_the_launches(fake):
    fake_hip.child(fake, "test_host_calls", "serve_from_a_graph")


# ---- the BF16 weights are made anew until that has succeeded ------------------------------------------
def prepared_weights_fail(hip):
    from vtrace_amd import denoise, renderer
    net = denoise.Denoiser(renderer.get_renderer(), seed=1)
    rad, gbuf = np.ones((32, 32, 4), np.float32), np.ones((32, 32, 8), np.float32)
    net.denoise(rad, gbuf, 1)
    net.set_params(net.get_params())
    hip.clear()
    hip.fail("k_prep_weights")
    with pytest.raises(renderer.RendererError):
        net.denoise(rad, gbuf, 1)
    assert _count(hip, "k_conv3x3") == 0
    hip.clear()
    net.denoise(rad, gbuf, 1)
    assert _count(hip, "k_prep_weights") == 1 and _count(hip, "k_conv3x3") == 19
    hip.clear()
    net.denoise(rad, gbuf, 1)
    assert _count(hip, "k_prep_weights") == 0


def test_weights_are_prepared_again_after_a_failure(fake):
    fake_hip.child(fake, "test_host_calls", "prepared_weights_fail")
