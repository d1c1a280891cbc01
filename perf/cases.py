"""The workloads this framework's speed is judged on, through its public entry points.

A case is a dict of plain values; ``prepare`` builds what a program holds before the call (volumes
uploaded, matrices, host arrays, a serving loop), ``run`` makes one pass and returns its whole
outputs.  The library keeps one scene, one parameter set and one network per process, like the
reference's globals, so a pass sets its own: the host loop re-sends the instance list and the
parameters before every frame (src/main.rs: update_instances, then render_tick).

Frames, hit records and serving results are fixed by the library's own FP32 rules and compared bit
for bit; they have no 64-bit counterpart (a path takes another voxel when a last bit differs), so
``exact`` has values for the network's cases only.
"""
from __future__ import annotations

import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from vtrace_amd import denoise, renderer, scenes, serving, world

MAX_TEXTURES = 65536
ENC, DEC, IN_CH = denoise.ENC, denoise.DEC, 16


def listed() -> list:
    return [
        # the reference's own picture (one primary ray per pixel, colour of the voxel hit) in a small
        # window over a small model: the smallest call, what an editor's thumbnail costs
        frame("preview_320x240", 320, 240, mode=0, size=64, count=1),
        # 128^3 model with a sun shadow at 640 x 480: the smallest lit frame
        frame("shadow_640x480", 640, 480, mode=1, size=128, count=1),
        # the size of the benchmark frame: 16 volumes of 256^3, 1080p, 4 samples, up to 4 bounces
        frame("path_1080p", 1920, 1080, mode=2, spp=4, bounces=4, size=256, count=16),
        # a large sparse volume at 4K, 1 sample and 2 bounces: the largest frame
        frame("path_4k_sparse", 3840, 2160, mode=2, spp=1, bounces=2, size=512, count=1, sparse=True),
        # odd frame over RGBA textures whose sizes are no multiple of a brick, hit records read too
        # (an editor that picks what is under the cursor)
        frame("path_ragged_rgba", 853, 479, mode=2, spp=3, bounces=3, size=100, count=9, rgba=True, hits=True),
        # thousands of moving objects: the tree is built anew for every frame
        frame("moving_4096", 640, 480, mode=0, size=16, count=4096),
        # a 256^3 model is opened: upload and first frame
        {"name": "open_256", "kind": "upload", "size_x": 256, "size_y": 256, "size_z": 256, "count": 1,
         "rgba": False, "width": 640, "height": 360},
        # the camera enters a new region of the streamed terrain: 48 chunks of 16^3 and a frame
        {"name": "stream_48_chunks", "kind": "upload", "size_x": 16, "size_y": 16, "size_z": 16, "count": 48,
         "rgba": True, "width": 1280, "height": 720},
        # twelve requests of mixed sizes through the serving loop
        {"name": "serve_12", "kind": "serve", "requests": 12, "max_width": 1280, "max_height": 720, "max_spp": 8,
         "bounces": 4},
        # an interactive frame: 1 sample traced with its G-buffer, then denoised on the device
        {"name": "frame_denoised_720p", "kind": "denoised_frame", "width": 1280, "height": 720, "spp": 1,
         "bounces": 2, "size": 128, "count": 4},
        # a saved 1080p frame denoised from host arrays
        {"name": "denoise_1080p", "kind": "denoise", "width": 1920, "height": 1080, "spp": 4},
        # the network fine-tuned on two new frames (the training defaults: batches of 8 crops of 128^2)
        {"name": "finetune_8_steps", "kind": "train", "steps": 8, "batch": 8, "crop": 128, "width": 320,
         "height": 256, "frames": 2},
    ]


def frame(name: str, width: int, height: int, mode: int, size: int, count: int, spp: int = 1, bounces: int = 0,
          rgba: bool = False, sparse: bool = False, hits: bool = False) -> dict:
    return {"name": name, "kind": "frame", "width": width, "height": height, "mode": mode, "spp": spp,
            "bounces": bounces, "size": size, "count": count, "rgba": rgba, "sparse": sparse, "hits": hits}


def draw(rng) -> dict:
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def window(lo, hi):
        w = log(lo, hi)
        return w, max(16, min(2160, int(w * rng.uniform(0.45, 1.0))))

    kind = rng.choice(("frame", "frame", "frame", "upload", "upload", "serve", "denoised_frame", "denoise", "train"))
    if kind == "frame":
        mode = rng.choice((0, 1, 2, 2))
        w, h = window(160, 2560)
        spp = 1
        if mode == 2:
            spp = rng.randint(1, max(1, min(8, 8000000 // (w * h))))
        size = rng.choice((16, 24, 33, 50, 64, 100, 128, 200, 256))
        count = log(1, 4096) if size <= 33 else rng.randint(1, 16)
        c = frame("", w, h, mode, size, count, spp, rng.randint(1, 4) if mode == 2 else 0,
                  rgba=rng.random() < 0.3, hits=rng.random() < 0.5)
    elif kind == "upload":
        w, h = window(160, 1280)
        if rng.random() < 0.5:
            c = {"kind": kind, "size_x": 16, "size_y": 16, "size_z": 16, "count": log(1, 160), "rgba": True,
                 "width": w, "height": h}
        else:
            c = {"kind": kind, "size_x": log(20, 256), "size_y": log(20, 256), "size_z": log(20, 256), "count": 1,
                 "rgba": rng.random() < 0.4, "width": w, "height": h}
    elif kind == "serve":
        c = {"kind": kind, "requests": rng.randint(1, 16), "max_width": log(200, 1280), "max_height": log(160, 720),
             "max_spp": rng.randint(1, 8), "bounces": rng.randint(1, 4)}
    elif kind == "denoised_frame":
        w, h = window(160, 1920)
        c = {"kind": kind, "width": w, "height": min(h, 1080), "spp": rng.randint(1, 2), "bounces": rng.randint(1, 4),
             "size": rng.choice((64, 100, 128, 200)), "count": rng.randint(1, 8)}
    elif kind == "denoise":
        w, h = window(100, 1920)
        c = {"kind": kind, "width": w, "height": min(h, 1080), "spp": 1 << rng.randint(0, 8)}
    else:
        crop = 16 * rng.randint(3, 10)
        c = {"kind": kind, "steps": rng.randint(2, 8), "batch": rng.randint(2, 8 if crop <= 128 else 5), "crop": crop,
             "width": crop + rng.randint(0, 150), "height": crop + rng.randint(0, 150), "frames": rng.randint(1, 3)}
    c.pop("name", None)
    return c


# ---- what the process keeps -------------------------------------------------------------------
class Session:
    """The library's globals as one program holds them: the renderer, the volumes uploaded so far,
    the serving loop and the network."""

    def __init__(self):
        self.r = renderer.get_renderer()
        self.volumes: dict = {}
        self.used = 0
        self.loop = None
        self.net = None

    def ids(self, specs: list) -> list:
        """Texture ids of the volumes `specs` = [(size, seed, fill, rgba)], uploaded on first use."""
        new = [s for s in dict.fromkeys(specs) if s not in self.volumes]
        with ThreadPoolExecutor(8) as pool:   # the generator is native and leaves the interpreter
            for s, v in zip(new, pool.map(_volume, new)):
                self.volumes[s] = self.r.upload(v)
                self.used += 1
        return [self.volumes[s] for s in specs]

    def room(self, count: int) -> None:
        """Ids are never given back, so a program that streams for hours starts over now and then."""
        if self.used + count > MAX_TEXTURES:
            self.r = renderer.reset_renderer()
            self.volumes, self.used, self.loop, self.net = {}, 0, None, None
        self.used += count


_session: Session | None = None


def session() -> Session:
    global _session
    if _session is None:
        _session = Session()
    return _session


def _volume(spec) -> scenes.Volume:
    size, seed, fill, rgba = spec
    idx, pal = scenes.gen_volume((size, size, size), seed, fill), scenes.gen_palette(seed)
    return scenes.Volume(scenes.expand_palette(idx, pal) if rgba else idx, None if rgba else pal)


def _pinned(shape, dtype=torch.float32) -> np.ndarray:
    return torch.empty(shape, dtype=dtype, pin_memory=True).numpy()


# ---- frames -------------------------------------------------------------------------------------
def _place(rng: scenes.Rng, count: int, size: float):
    """Centres of `count` boxes on a jittered lattice about two and a half boxes apart, and the
    radius of the whole."""
    side = max(1, math.ceil(count ** (1.0 / 3.0)))
    step = 2.5 * size
    cells = [(x, y, z) for x in range(side) for y in range(side) for z in range(side)]
    for i in range(count):   # the first `count` of a shuffle
        j = rng.randint(i, len(cells) - 1)
        cells[i], cells[j] = cells[j], cells[i]
    mid = (side - 1) / 2.0
    centres = [tuple((c - mid) * step + rng.uniform(-0.4, 0.4) * size for c in cell) for cell in cells[:count]]
    return centres, 0.5 * step * side


def _view(rng: scenes.Rng, radius: float, width: int, height: int):
    eye, target = scenes.orbit_camera(rng, (0.0, 0.0, 0.0), radius, 0.05 * radius)
    return scenes.perspective(scenes.FOV, width / height), scenes.look_at(eye, target)


def _prepare_frame(c: dict, seed: int) -> dict:
    s, rng, n = session(), scenes.Rng(seed), c["size"]
    distinct = 16 if c["count"] > 16 else c["count"]
    fill = 0.05 if c.get("sparse") else 0.3
    ids = s.ids([(n, 100 * n + k, fill if c.get("sparse") else 0.1 + 0.02 * k, c.get("rgba", False))
                 for k in range(distinct)])
    centres, radius = _place(rng, c["count"], n)
    records = np.stack([scenes.instance_record(scenes.model_matrix(p, float(n)), ids[i % distinct])
                        for i, p in enumerate(centres)])
    P, C = _view(rng, 0.6 * radius + 0.7 * n, c["width"], c["height"])
    mode = c.get("mode", 2)
    params = scenes.RenderParams(c["width"], c["height"], viewport_square=0, mode=mode, spp=c.get("spp", 1),
                                 max_bounces=c.get("bounces", 0), jitter=1 if mode == 2 else 0, seed=seed,
                                 sun_dir=scenes.sun_direction(rng))
    out = _pinned((c["height"], c["width"], 4)) if mode else None
    return {"r": s.r, "records": records, "params": params, "P": P, "C": C, "out": out, "mode": mode,
            "hits": c.get("hits", False)}


def _run_frame(st: dict) -> dict:
    r = st["r"]
    r.set_instances(st["records"])
    r.set_params(st["params"])
    r.render(st["P"], st["C"])
    # mode 0 is shown (the swapchain's BGRA8); lit frames go on as radiance
    got = {"radiance": r.radiance(out=st["out"])} if st["mode"] else {"bgra8": r.bgra8().view(np.uint8)}
    if st["hits"]:
        got["hits"] = r.hits().view(np.uint8)
    return got


# ---- uploads ------------------------------------------------------------------------------------
_terrain: list | None = None


def _terrain_chunks() -> list:
    """The occupied chunks around the terrain's origin (what the pager queues there)."""
    global _terrain
    if _terrain is None:
        gen = world.TerrainGenerator(0)
        got = gen.gen_chunks(world.load_positions((0.0, 0.0, 0.0)))
        _terrain = [v.data for v in got if v is not None]
    return _terrain


_noise: dict = {}


def _prepare_upload(c: dict, seed: int) -> dict:
    rng = scenes.Rng(seed)
    dims = (c["size_x"], c["size_y"], c["size_z"])
    if c["count"] > 1 or dims == (16, 16, 16):   # streamed chunks: terrain tinted by the seed
        chunks = _terrain_chunks()
        tint = np.uint32(rng.u32() & 0x000F0F0F)
        first = rng.randint(0, len(chunks) - 1)
        vols = []
        for k in range(c["count"]):
            d = chunks[(first + k) % len(chunks)]
            vols.append(scenes.Volume(np.where(d != 0, d ^ tint, d).astype(np.uint32), None))
    else:
        if dims not in _noise:
            _noise[dims] = scenes.gen_volume(dims, sum(dims), 0.25)
        shift = [rng.randint(0, d - 1) for d in reversed(dims)]
        idx, pal = np.ascontiguousarray(np.roll(_noise[dims], shift, (0, 1, 2))), scenes.gen_palette(seed)
        vols = [scenes.Volume(scenes.expand_palette(idx, pal) if c["rgba"] else idx, None if c["rgba"] else pal)]
    size = float(max(dims))
    centres, radius = _place(rng, c["count"], size)
    models = [scenes.model_matrix(p, tuple(float(d) for d in dims)) for p in centres]
    P, C = _view(rng, 0.6 * radius + 0.7 * size, c["width"], c["height"])
    return {"volumes": vols, "models": models, "P": P, "C": C,
            "params": scenes.RenderParams(c["width"], c["height"], viewport_square=0, mode=0)}


def _run_upload(st: dict) -> dict:
    s = session()
    s.room(len(st["volumes"]))
    r = s.r
    ids = r.upload_many(st["volumes"])
    r.set_instances(np.stack([scenes.instance_record(m, i) for m, i in zip(st["models"], ids)]))
    r.set_params(st["params"])
    r.render(st["P"], st["C"])
    return {"bgra8": r.bgra8().view(np.uint8), "brick_map": r.brick_map(ids[0]).view(np.uint8)}


# ---- serving ------------------------------------------------------------------------------------
SERVED = [(64, 1, 0.3, False), (128, 2, 0.2, False), (128, 3, 0.35, False), (256, 4, 0.15, False)]


def _prepare_serve(c: dict, seed: int) -> dict:
    s, rng = session(), scenes.Rng(seed)
    if s.loop is None:
        recs = serving.scene_records(s.ids(SERVED), [v[0] for v in SERVED])
        s.loop = serving.ServingLoop(s.r)
        for rec in recs:
            s.loop.add_scene(rec)
    requests, outs = [], []
    for i in range(c["requests"]):
        # sizes from the whole down to a fifth, the same for every seed; cameras are the seed's
        f = 0.2 + 0.8 * ((i * 7 + 3) % c["requests"] + 1) / c["requests"]
        w, h = max(16, int(c["max_width"] * f)), max(16, int(c["max_height"] * f))
        k = i % len(SERVED)
        eye, target = scenes.orbit_camera(rng, (0.0, 0.0, 0.0), rng.uniform(1.2, 2.0) * SERVED[k][0],
                                          0.1 * SERVED[k][0])
        requests.append(serving.Request(k, w, h, 1 + (i * 5 + c["max_spp"] - 1) % c["max_spp"],
                                        scenes.perspective(scenes.FOV, w / h), scenes.look_at(eye, target),
                                        seed=seed + i, max_bounces=c["bounces"], sun_dir=scenes.sun_direction(rng)))
        outs.append(_pinned((h, w, 4)))
    return {"loop": s.loop, "requests": requests, "outs": outs}


def _run_serve(st: dict) -> list:
    loop = st["loop"]
    where = {loop.submit(q): i for i, q in enumerate(st["requests"])}
    left = len(where)
    while left:
        for rid in loop.step():
            q, i = st["requests"][where[rid]], where[rid]
            loop.read(rid, q.width, q.height, out=st["outs"][i])
            left -= 1
    return list(st["outs"])


# ---- network ------------------------------------------------------------------------------------
def _layers() -> list:
    """(inputs, outputs) of the 19 convolutions, in the parameter vector's order."""
    shapes, c = [], IN_CH
    for e in ENC:
        shapes += [(c, e), (e, e)]
        c = e
    up = ENC[4]
    for lvl in (3, 2, 1, 0):
        shapes += [(up + ENC[lvl], DEC[lvl]), (DEC[lvl], DEC[lvl])]
        up = DEC[lvl]
    return shapes + [(up, 3)]


_weights = None


def weights() -> np.ndarray:
    """The program's network: He-normal, small biases, an output layer as small as a trained one's."""
    global _weights
    if _weights is None:
        rng, parts = np.random.default_rng(11), []
        for i, (ci, co) in enumerate(_layers()):
            fan = 9 * (denoise.N_FEATURES if i == 0 else ci)
            w = rng.normal(0.0, math.sqrt((2.0 if i < 18 else 0.02) / fan), (co, 9, ci))
            if i == 0:
                w[..., denoise.N_FEATURES:] = 0.0
            parts += [w.reshape(-1), rng.normal(0.0, 0.02, co)]
        _weights = np.concatenate(parts).astype(np.float32)
    return _weights


def network() -> "denoise.Denoiser":
    s = session()
    if s.net is None:
        s.net = denoise.Denoiser(s.r, seed=None)
    s.net.set_params(weights())
    return s.net


def _traced(width: int, height: int, spp: int, seed: int):
    """(radiance, G-buffer, clean radiance) as a traced frame has them: flat faces of one albedo and
    an axis-aligned normal, sky between them, and the noise of `spp` paths."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape):
        return torch.rand(*shape, device="cuda", generator=g)

    cell = 8
    gh, gw = -(-height // cell), -(-width // cell)

    def grow(a):
        return a.repeat_interleave(cell, 0).repeat_interleave(cell, 1)[:height, :width]

    hit = grow((rand(gh, gw) > 0.2).float())[..., None]
    albedo = grow(0.05 + 0.9 * rand(gh, gw, 3) ** 2)
    axis = grow((rand(gh, gw) * 6).long().clamp(max=5))
    normal = torch.tensor([[-1, 0, 0], [1, 0, 0], [0, -1, 0], [0, 1, 0], [0, 0, -1], [0, 0, 1]], device="cuda",
                          dtype=torch.float32)[axis]
    dist = grow(50.0 + 900.0 * rand(gh, gw))[..., None]
    light = grow(0.1 + 1.5 * rand(gh, gw, 1) ** 2) * torch.tensor([1.0, 0.95, 0.85], device="cuda")
    noise = (-torch.log1p(-rand(height, width, 1) * 0.999) - 1.0) / math.sqrt(spp) + 1.0
    sky = torch.tensor(scenes.SKY, device="cuda")
    clean = hit * albedo * light + (1 - hit) * sky
    noisy = hit * (albedo * light * noise.clamp(min=0.0)) + (1 - hit) * sky
    one = torch.ones(height, width, 1, device="cuda")
    gbuf = torch.cat([hit * albedo + (1 - hit) * sky, hit * dist, hit * normal, hit], -1)
    return torch.cat([noisy, one], -1), gbuf, torch.cat([clean, one], -1)


def _prepare_denoise(c: dict, seed: int) -> dict:
    rad, gbuf, _ = _traced(c["width"], c["height"], c["spp"], seed)
    return {"net": network(), "rad": rad.cpu().numpy(), "gbuf": gbuf.cpu().numpy(), "spp": c["spp"]}


def _run_denoise(st: dict) -> dict:
    return {"image": st["net"].denoise(st["rad"], st["gbuf"], st["spp"])[0]}


def _run_denoised_frame(st: dict) -> dict:
    r = st["r"]
    r.set_instances(st["records"])
    r.enable_gbuffer(True)
    r.set_params(st["params"])
    r.render(st["P"], st["C"])
    image = st["net"].denoise_frame()[0]
    r.enable_gbuffer(False)
    return {"image": image}


#: a fine-tuning rate: a trained network is adapted, not trained anew
RATE = 4e-6


def _frames(c: dict, seed: int) -> list:
    return [(*_traced(c["width"], c["height"], 1 << (2 * k), 1000 * seed + k), 1 << (2 * k))
            for k in range(c["frames"])]


def _prepare_train(c: dict, seed: int) -> dict:
    return {"net": network(), "frames": [tuple(t.cpu().numpy() for t in f[:3]) + (f[3],) for f in _frames(c, seed)],
            "steps": c["steps"], "batch": c["batch"], "crop": c["crop"], "seed": seed & 0xFFFF, "start": weights()}


def _run_train(st: dict) -> dict:
    net = st["net"]
    net.set_params(st["start"])
    net.clear_frames()
    for rad, gbuf, target, spp in st["frames"]:
        net.add_frame(rad, gbuf, target, spp)
    losses = net.train(st["steps"], batch=st["batch"], crop=st["crop"], lr=RATE, seed=st["seed"])
    return {"losses": losses, "params": net.get_params()}


# ---- the network in 64 bits, from torch alone ------------------------------------------------------
def _conv(x, w, b, relu):
    """3x3, zero border; x (n, h, w, ci), w (co, 9, ci)."""
    n, h, wd, ci = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(n * h * wd, -1)
    for t in range(9):
        y = y + p[:, t // 3:t // 3 + h, t % 3:t % 3 + wd].reshape(-1, ci) @ w[:, t].t()
    return (y.clamp(min=0) if relu else y).reshape(n, h, wd, -1)


def _unet(x, params):
    layers, at = [], 0
    for ci, co in _layers():
        layers.append((params[at:at + 9 * ci * co].view(co, 9, ci), params[at + 9 * ci * co:at + 9 * ci * co + co]))
        at += 9 * ci * co + co
    skips = []
    for lvl in range(5):
        x = _conv(_conv(x, *layers[2 * lvl], True), *layers[2 * lvl + 1], True)
        if lvl < 4:
            skips.append(x)
            n, h, w, ch = x.shape
            x = x.view(n, h // 2, 2, w // 2, 2, ch).mean((2, 4))
    for k, lvl in enumerate((3, 2, 1, 0)):
        x = torch.cat([x.repeat_interleave(2, 1).repeat_interleave(2, 2), skips[lvl]], -1)
        x = _conv(_conv(x, *layers[10 + 2 * k], True), *layers[11 + 2 * k], True)
    return _conv(x, *layers[18], False)


def _features(rad, gbuf, spp):
    rad, gbuf = rad.double(), gbuf.double()
    x = torch.zeros(*rad.shape[:-1], IN_CH, dtype=torch.float64, device=rad.device)
    x[..., 0:3] = torch.log1p(rad[..., :3].clamp(min=0) / (gbuf[..., 0:3] + 0.01))
    x[..., 3:6] = gbuf[..., 0:3]
    x[..., 6:9] = gbuf[..., 4:7]
    x[..., 9] = torch.log1p(gbuf[..., 3].clamp(min=0)) / 8
    x[..., 10] = math.log2(spp) / 8
    return x


def _radiance(x, y):
    return (x[..., 3:6] + 0.01) * torch.expm1((x[..., 0:3] + y).clamp(max=16.0))


def _pcg(v: int) -> int:
    """PCG-RXS-M-XS 32 (O'Neill 2014) as Jarzynski and Olano (2020) hash with it."""
    s = (v * 747796405 + 2891336453) & 0xFFFFFFFF
    w = (((s >> ((s >> 28) + 4)) ^ s) * 277803737) & 0xFFFFFFFF
    return (w >> 22) ^ w


def _exact_denoise(c: dict, seed: int) -> dict:
    rad, gbuf, _ = _traced(c["width"], c["height"], c["spp"], seed)
    h, w = rad.shape[:2]
    x = _features(rad, gbuf, c["spp"]).permute(2, 0, 1)[None]
    x = torch.nn.functional.pad(x, (0, -w % 16, 0, -h % 16), mode="replicate").permute(0, 2, 3, 1).contiguous()
    with torch.no_grad():
        y = _unet(x, torch.from_numpy(weights()).cuda().double())
        image = torch.ones(h, w, 4, dtype=torch.float64, device="cuda")
        image[..., :3] = _radiance(x, y)[0, :h, :w].clamp(min=0)
    return {"image": image}


def _exact_train(c: dict, seed: int) -> dict:
    frames = [(_features(rad, gbuf, spp), target[..., :3].double()) for rad, gbuf, target, spp in _frames(c, seed)]
    st, crops, crop = _pcg((seed & 0xFFFF) ^ 0x9E3779B9), [], c["crop"]
    for _ in range(c["steps"] * c["batch"]):
        got = []
        for n in (len(frames), c["height"] - crop + 1, c["width"] - crop + 1):
            st = _pcg(st)
            got.append(st % n)
        crops.append(got)
    p = torch.from_numpy(weights()).cuda().double().requires_grad_()
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    warm = min(100, c["steps"] // 10 + 1)
    for it in range(c["steps"]):
        mine = crops[it * c["batch"]:(it + 1) * c["batch"]]
        x, t = (torch.stack([frames[k][i][a:a + crop, b:b + crop] for k, a, b in mine]) for i in (0, 1))
        loss = ((_radiance(x, _unet(x, p)) - t) ** 2 / (t * t + 0.01)).mean()
        grad, = torch.autograd.grad(loss, p)
        losses.append(loss.detach())
        rate = RATE * (0.05 + 0.475 * (1.0 + math.cos(math.pi * it / c["steps"]))) * min(1.0, (it + 1) / warm)
        m = 0.9 * m + 0.1 * grad
        v = 0.999 * v + 0.001 * grad * grad
        with torch.no_grad():
            p -= rate * (m / (1 - 0.9 ** (it + 1))) / ((v / (1 - 0.999 ** (it + 1))).sqrt() + 1e-8)
    return {"losses": torch.stack(losses), "params": p.detach()}


# ---- the five functions ----------------------------------------------------------------------------
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("frame", "denoised_frame"):
        st = _prepare_frame(case, seed)
        if kind == "denoised_frame":
            st["net"] = network()
    else:
        st = {"upload": _prepare_upload, "serve": _prepare_serve, "denoise": _prepare_denoise,
              "train": _prepare_train}[kind](case, seed)
    st["kind"] = kind
    return st


def run(state: dict):
    return {"frame": _run_frame, "upload": _run_upload, "serve": _run_serve, "denoised_frame": _run_denoised_frame,
            "denoise": _run_denoise, "train": _run_train}[state["kind"]](state)


def exact(case: dict, seed: int):
    if case["kind"] == "denoise":
        return _exact_denoise(case, seed)
    return _exact_train(case, seed) if case["kind"] == "train" else None


def _conv_flops(pixels: float) -> float:
    """Multiply-adds of one forward pass over `pixels` level-0 pixels, as operations."""
    lvl = [l for l in range(5) for _ in (0, 1)] + [3, 3, 2, 2, 1, 1, 0, 0, 0]
    return sum(2.0 * 9 * ci * co * pixels / 4 ** l for (ci, co), l in zip(_layers(), lvl))


def work(case: dict) -> dict:
    """Bytes: what crosses the entry points, once.  Operations: the network's multiply-adds; for rays
    the camera ray, one box test and one entry of a volume (about 120 each), whatever walks follow."""
    kind = case["kind"]
    ray = 120.0
    if kind == "serve":
        px = [(max(16, int(case["max_width"] * f)) * max(16, int(case["max_height"] * f)),
               1 + (i * 5 + case["max_spp"] - 1) % case["max_spp"])
              for i in range(case["requests"])
              for f in (0.2 + 0.8 * ((i * 7 + 3) % case["requests"] + 1) / case["requests"],)]
        return {"bytes": 16.0 * sum(p for p, _ in px), "flops": ray * sum(p * s for p, s in px)}
    if kind == "train":
        px = case["steps"] * case["batch"] * case["crop"] ** 2
        n = len(weights())
        return {"bytes": 64.0 * case["frames"] * case["width"] * case["height"] + 8.0 * n,
                "flops": 3.0 * _conv_flops(px)}
    px = case["width"] * case["height"]
    if kind == "denoise":
        return {"bytes": 64.0 * px, "flops": _conv_flops(px)}
    if kind == "denoised_frame":
        return {"bytes": 16.0 * px + 64.0 * case["count"], "flops": _conv_flops(px) + ray * px * case["spp"]}
    if kind == "upload":
        vox = case["size_x"] * case["size_y"] * case["size_z"] * case["count"]
        return {"bytes": (4.0 if case["rgba"] else 1.0) * vox + 64.0 * case["count"] + 4.0 * px, "flops": ray * px}
    out = 4.0 if case["mode"] == 0 else 16.0
    return {"bytes": px * (out + (16.0 if case["hits"] else 0.0)) + 64.0 * case["count"],
            "flops": ray * px * case["spp"]}
