"""What is timed of the photon mapper: the work its callers have it do.

Every case goes through the C ABI the way a host program does: a context (or a
batch) is kept, output buffers belong to the caller, and a pass is the calls of
one frame or one request.  Scenes are the library's presets and its batch
generator; `seed` drives the photon and camera streams, the density field, the
batch's sphere layouts and every caller-given array.

Kinds of case:
  frame    emit + build + render: the scene changes every frame (animation)
  view     render of a crop from photon maps that are kept (a moving window, a
           serving loop), with the medium or with the surface estimate alone
  voxel    emit + render with the voxel-grid estimate
  cache    emit + build + render through the learned radiance cache
  knn      kd-tree build over caller-given points + k-NN lists of queries
  predict  radiance of caller-given rows by the cache's network
  grad     loss gradient of the cache's network on caller-given rows
  batch    one frame of many scenes through the captured graph
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "cuda-photon-mapper_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import pmamd  # noqa: E402

# Radiance queries per eye sample: the march crosses the room at 0.01 a step
# (about 60 points a sample over the presets' views), and most samples end on a
# diffuse surface.
_STEPS, _HITS = 60.0, 0.94


def listed():
    return [
        # A small window of the unit room from kept maps, without allocation: a
        # tight serving loop, or the tile a user drags over.
        {"name": "view_room_64x48", "kind": "view", "preset": 1, "w": 64, "h": 48, "spp": 1, "cone": True,
         "media": True, "noalloc": True},
        # The interactive program's frame: 100k photons, 256 x 256, new photons each frame.
        {"name": "room_256", "kind": "frame", "preset": 1, "n_emit": 100000, "n_volume": 0, "w": 256, "h": 256,
         "spp": 1, "cone": False},
        # The precision variant: BF16 photon power and direction, FP64 transmittance.
        {"name": "room_bf16_480x270", "kind": "frame", "preset": 3, "n_emit": 100000, "n_volume": 0, "w": 480,
         "h": 270, "spp": 1, "cone": False},
        # A ragged crop of the full fog scene from kept maps: progressive or tiled rendering.
        {"name": "view_fog_477x271x4", "kind": "view", "preset": 2, "w": 477, "h": 271, "spp": 4, "cone": False,
         "media": True, "noalloc": False},
        # The headline frame: 1M surface + 2M volume records, 1920 x 1080 x 4, k = 64.
        {"name": "fog_1080x4", "kind": "frame", "preset": 2, "n_emit": 1000000, "n_volume": 2000000, "w": 1920,
         "h": 1080, "spp": 4, "cone": False},
        # The same maps without the march: surface estimates only.
        {"name": "surfaces_1080x4", "kind": "view", "preset": 2, "w": 1920, "h": 1080, "spp": 4, "cone": False,
         "media": False, "noalloc": False},
        # The voxel-grid estimate, grids rebuilt for new photons each frame.
        {"name": "voxel_1080x4", "kind": "voxel", "preset": 2, "n_emit": 1000000, "n_volume": 2000000, "w": 1920,
         "h": 1080, "spp": 4, "blend": True},
        # The learned cache's frame in its BF16 form, a few frames into its training.
        {"name": "cache_1080x4", "kind": "cache", "n_emit": 1000000, "n_volume": 2000000, "w": 1920, "h": 1080,
         "spp": 4, "stride": 4, "threshold": 0.12},
        # Neighbour lists over a caller's points on the room's walls.
        {"name": "knn_walls_1m", "kind": "knn", "n": 1000000, "nq": 65536, "k": 64, "walls": True},
        # The network alone, half surface and half volume rows.
        {"name": "predict_2m", "kind": "predict", "n": (1 << 21) + 137},
        # One gradient of the network's loss.
        {"name": "grad_64k", "kind": "grad", "n": 1 << 16},
        # Sixteen scenes of uneven photon counts and image sizes, tuned once by the library.
        {"name": "batch_16", "kind": "batch", "scenes": 16, "photons_low": 10000, "photons_high": 2000000,
         "side_low": 128, "side_high": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "view", "view", "voxel", "cache", "knn", "predict", "grad", "batch"])
    if kind in ("frame", "view"):
        preset = rng.choice([1, 2, 3])
        c = {"kind": kind, "preset": preset, "w": _log_int(rng, 40, 900), "h": _log_int(rng, 30, 600),
             "spp": rng.choice([1, 2, 3, 4]), "cone": rng.random() < 0.25}
        if kind == "frame":
            c["n_emit"] = _log_int(rng, 10000, 400000) if preset != 2 else _log_int(rng, 200000, 1000000)
            c["n_volume"] = 0 if preset != 2 else 2 * c["n_emit"]
        else:
            c["media"], c["noalloc"] = rng.random() < 0.75, rng.random() < 0.5
        return c
    if kind == "voxel":
        n = _log_int(rng, 50000, 1000000)
        return {"kind": kind, "preset": 2, "n_emit": n, "n_volume": 2 * n, "w": _log_int(rng, 200, 1920),
                "h": _log_int(rng, 120, 1080), "spp": rng.choice([1, 2, 4]), "blend": rng.random() < 0.5}
    if kind == "cache":
        n = _log_int(rng, 200000, 1000000)
        return {"kind": kind, "n_emit": n, "n_volume": 2 * n, "w": _log_int(rng, 240, 1920),
                "h": _log_int(rng, 160, 1080), "spp": rng.choice([1, 2, 4]), "stride": rng.choice([2, 4, 5]),
                "threshold": rng.choice([0.05, 0.12])}
    if kind == "knn":
        return {"kind": kind, "n": _log_int(rng, 5000, 2000000), "nq": _log_int(rng, 500, 65536),
                "k": rng.randint(1, 64), "walls": rng.random() < 0.5}
    if kind == "predict":
        return {"kind": kind, "n": _log_int(rng, 1000, 4000000)}
    if kind == "grad":
        return {"kind": kind, "n": _log_int(rng, 1000, 1 << 19)}
    lo = _log_int(rng, 10000, 100000)
    return {"kind": kind, "scenes": rng.randint(2, 16), "photons_low": lo,
            "photons_high": lo + _log_int(rng, 1000, 1500000), "side_low": rng.randint(64, 200),
            "side_high": rng.randint(256, 800)}


# ------------------------------------------------------------------ inputs
def _config(case, seed):
    c = pmamd.preset(case.get("preset", 2))
    c.seed = 1 + seed % 0x7FFFFFFF
    if case.get("n_volume"):
        c.n_emit, c.cap_surface, c.cap_volume = 0, case["n_emit"], case["n_volume"]
    elif case.get("n_emit"):
        c.n_emit = case["n_emit"]
    if case.get("cone"):
        c.estimator = pmamd.PM_EST_CONE
    if case["kind"] != "view":
        c.width, c.height = case["w"], case["h"]
    c.spp = case["spp"]
    if case["kind"] == "cache":
        c.storage, c.fp64_transmittance = pmamd.PM_STORE_BF16, 1
    return c


def _emit_build(g):
    g.emit()
    g.build()


def _rows(n, seed):
    """Input rows (position, direction, normal) and radiance targets, as the cache's own records hold them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.zeros((n, 9), device="cuda")
    x[:, :3] = torch.rand((n, 3), device="cuda", generator=gen)
    d = torch.randn((n, 3), device="cuda", generator=gen)
    x[:, 3:6] = d / d.norm(dim=1, keepdim=True)
    walls = torch.tensor([[-1.0, 0, 0], [0, 1, 0], [1, 0, 0], [0, -1, 0], [0, 0, -1]], device="cuda")
    pick = torch.randint(0, 5, (n // 2,), device="cuda", generator=gen)
    x[: n // 2, 6:9] = walls[pick]  # half surface rows; a volume row's normal is zero
    return x, torch.exp(torch.randn((n, 3), device="cuda", generator=gen))


_SHAPES = [(128, 224), (128, 128), (128, 128), (128, 128), (16, 128)]


def _params(seed):
    """Weights in the library's flat layout (W row-major, then b, per layer; padding zero)."""
    rng = np.random.default_rng(seed)
    parts = []
    for i, (o, k) in enumerate(_SHAPES):
        rows, cols = (3 if i == 4 else o), (216 if i == 0 else k)
        s = math.sqrt(6.0 / (cols + (rows if i == 4 else 0)))
        w, b = np.zeros((o, k), np.float32), np.zeros(o, np.float32)
        w[:rows, :cols] = rng.uniform(-s, s, (rows, cols))
        b[:rows] = rng.uniform(-0.1, 0.1, rows)
        parts += [w.ravel(), b]
    return np.concatenate(parts)


def _points(case, seed):
    """Points on the room's walls, or spread through its volume, and queries near them."""
    rng = np.random.default_rng(seed)
    n, nq = case["n"], case["nq"]
    pos = rng.random((n, 3), dtype=np.float32)
    q = rng.random((nq, 3), dtype=np.float32)
    if case["walls"]:
        for p in (pos, q):
            w = rng.integers(0, 5, len(p))
            axis, side = np.array([0, 0, 1, 1, 2])[w], np.array([0, 1, 0, 1, 1], np.float32)[w]
            p[np.arange(len(p)), axis] = side
    # a cap that holds about three times k points on average
    share = 3.0 * case["k"] / n
    r = math.sqrt(share * 5 / math.pi) if case["walls"] else (share * 0.75 / math.pi) ** (1.0 / 3.0)
    return pos, q, float(np.float32(min(0.5, r)))


def _batch_configs(case, seed):
    out, n = [], case["scenes"]
    for i in range(n):
        c = pmamd.batch_scene(1 + seed % 0x7FFFFFFF, i)
        a = ((7 * i) % n) / max(1, n - 1)  # photon counts over their logarithm, in no order of the sizes
        c.n_emit = int(case["photons_low"] * (case["photons_high"] / case["photons_low"]) ** a)
        c.width = int(case["side_low"] * (case["side_high"] / case["side_low"]) ** (i / max(1, n - 1)))
        c.height = c.width - i % 3
        c.medium, c.sigma_s, c.sigma_a = pmamd.PM_MEDIUM_HOMOGENEOUS, 0.3 * (i + 1) / n, 0.03 * (i + 1) / n
        out.append(c)
    return out


def _image(h, w):
    return torch.empty((h, w, 3), dtype=torch.float32, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "lib": pmamd.load()}
    if kind == "batch":
        cfgs = _batch_configs(case, seed)
        s["b"] = pmamd.Batch(cfgs)
        s["b"].autotune(16)
        s["img"] = [_image(c.height, c.width) for c in cfgs]
        return s
    if kind in ("predict", "grad"):
        s["g"] = pmamd.PhotonMapper(pmamd.preset(5))
        s["g"].cache_reset(1)
        s["g"].cache_params(_params(seed))
        s["n"] = case["n"]
        s["x"], s["t"] = _rows(case["n"], seed)
        s["out"] = torch.empty((case["n"], 3), device="cuda")
        torch.cuda.synchronize()
        return s
    if kind == "knn":
        c = pmamd.preset(1)
        g = s["g"] = pmamd.PhotonMapper(c)
        pos, q, s["rcap"] = _points(case, seed)
        s["map"] = pmamd.PM_MAP_SURFACE if case["walls"] else pmamd.PM_MAP_VOLUME
        g.set_records(s["map"], pos, np.ones_like(pos), np.tile(np.float32([0, 0, 1]), (len(pos), 1)), len(pos))
        s["k"], s["nq"] = case["k"], case["nq"]
        s["q"] = torch.from_numpy(q).cuda()
        s["idx"] = torch.empty((case["nq"], case["k"]), dtype=torch.int32, device="cuda")
        s["d2"] = torch.empty((case["nq"], case["k"]), device="cuda")
        s["count"] = torch.empty(case["nq"], dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return s
    c = _config(case, seed)
    g = s["g"] = pmamd.PhotonMapper(c)
    s["w"], s["h"] = case["w"], case["h"]
    s["img"] = _image(case["h"], case["w"])
    if kind == "view":
        # the window: towards the middle of the configured frame, inside it
        c0 = (max(c.width, case["w"]), max(c.height, case["h"]))
        g.set_render(c0[0], c0[1], case["spp"], c.k_surface, c.k_volume, c.rcap_surface, c.rcap_volume)
        s["x0"], s["y0"] = (c0[0] - case["w"]) * 2 // 5, (c0[1] - case["h"]) * 3 // 7
        if not case["media"]:
            g.set_option(pmamd.PM_OPT_RENDER_MEDIA, 0)
        s["noalloc"] = case["noalloc"]
        _emit_build(g)
    elif kind == "voxel":
        g.set_option(pmamd.PM_OPT_VOXEL_GRID, 2 if case["blend"] else 1)
    elif kind == "cache":
        g.cache_reset(1)
        g.cache_configure(threshold=case["threshold"], batch=8192, march_stride=case["stride"])
        for _ in range(3):
            _emit_build(g)
            pmamd.check(s["lib"].pm_render_cache_crop(g.h, 0, 0, s["w"], s["h"], s["img"].data_ptr(), None), "cache")
    return s


def run(s):
    kind, lib = s["kind"], s["lib"]
    if kind == "batch":
        s["b"].submit()
        for i, img in enumerate(s["img"]):
            pmamd.check(lib.pm_batch_image(s["b"].h, i, img.data_ptr(), None), "pm_batch_image")
        return s["img"]
    g = s["g"]
    if kind == "predict":
        pmamd.check(lib.pm_cache_predict(g.h, s["x"].data_ptr(), s["n"], s["out"].data_ptr()), "pm_cache_predict")
        return s["out"]
    if kind == "grad":
        grad, loss = np.empty(lib.pm_cache_param_count(), np.float32), ctypes.c_double()
        pmamd.check(lib.pm_cache_grad(g.h, s["x"].data_ptr(), s["t"].data_ptr(), s["n"], grad.ctypes.data, grad.size,
                                      ctypes.byref(loss)), "pm_cache_grad")
        return {"grad": grad, "loss": loss.value}
    if kind == "knn":
        g.build()
        pmamd.check(lib.pm_knn(g.h, s["map"], s["q"].data_ptr(), s["nq"], s["k"], s["rcap"], s["idx"].data_ptr(),
                               s["d2"].data_ptr(), s["count"].data_ptr()), "pm_knn")
        return {"idx": s["idx"], "d2": s["d2"], "count": s["count"]}
    rgb = s["img"].data_ptr()
    if kind == "view":
        call = lib.pm_render_crop_noalloc if s["noalloc"] else lib.pm_render_crop
        pmamd.check(call(g.h, s["x0"], s["y0"], s["w"], s["h"], rgb, None), "render")
        return s["img"]
    g.emit()
    if kind == "voxel":
        pmamd.check(lib.pm_render(g.h, rgb, None), "pm_render")
        return s["img"]
    g.build()
    if kind == "cache":
        pmamd.check(lib.pm_render_cache_crop(g.h, 0, 0, s["w"], s["h"], rgb, None), "pm_render_cache_crop")
    else:
        pmamd.check(lib.pm_render(g.h, rgb, None), "pm_render")
    return s["img"]


# ------------------------------------------------------------------ the work of a pass
def _frame_work(samples, pixels, records, k, steps=_STEPS, per_neighbour=34.0):
    """Records written and read once, the image once; per neighbour of a query its squared distance (8) and its
    phase function and sum (26)."""
    return {"bytes": 12.0 * pixels + 2.0 * 44.0 * records, "flops": samples * (steps + _HITS) * k * per_neighbour}


def work(case):
    kind = case["kind"]
    row = 2.0 * (216 * 128 + 3 * 128 * 128 + 128 * 3)
    if kind == "predict":
        return {"bytes": 48.0 * case["n"], "flops": row * case["n"]}
    if kind == "grad":
        return {"bytes": 48.0 * case["n"], "flops": 3.0 * row * case["n"]}
    if kind == "knn":
        return {"bytes": 28.0 * case["n"] + (16.0 + 8.0 * case["k"]) * case["nq"],
                "flops": 8.0 * case["k"] * case["nq"] + case["n"] * math.log2(max(2, case["n"]))}
    if kind == "batch":
        w = {"bytes": 0.0, "flops": 0.0}
        n = case["scenes"]
        for i in range(n):
            photons = case["photons_low"] * (case["photons_high"] / case["photons_low"]) ** (i / max(1, n - 1))
            side = case["side_low"] * (case["side_high"] / case["side_low"]) ** (i / max(1, n - 1))
            one = _frame_work(side * side, side * side, 2.0 * photons, 8, 40.0)  # sparse maps: few within the cap
            w = {k: w[k] + one[k] for k in w}
        return w
    pixels = float(case["w"] * case["h"])
    samples = pixels * case["spp"]
    preset = case.get("preset", 2)
    k = 64 if preset == 2 else 8  # the room's volume map is sparse: most points find a few photons within the cap
    if kind == "view":
        records = {1: 2.5e5, 2: 3e6, 3: 2.5e5}[preset]
        w = _frame_work(samples, pixels, 0.0, k, _STEPS if case["media"] else 0.0)
        w["bytes"] += 44.0 * records * min(1.0, pixels / 1e5)
        return w
    records = case["n_emit"] + case["n_volume"] if case["n_volume"] else 2.5 * case["n_emit"]
    if kind == "voxel":  # a table lookup of a window (8 corners x 3 channels, 4 windows blended) a query
        return _frame_work(samples, pixels, records, 1, _STEPS, 24.0 * (4 if case["blend"] else 1))
    if kind == "cache":  # one network row per `stride` march points, the training's rows, exact surface estimates
        rows = samples * _STEPS / case["stride"]
        w = _frame_work(samples, pixels, records, 64, 0.0)
        w["flops"] += 2.0 * (144 * 128 + 3 * 128 * 128 + 128 * 3) * rows + 3.0 * row * (1 << 18)
        return w
    return _frame_work(samples, pixels, records, k)


# ------------------------------------------------------------------ values in 64 bits
def _forward64(flat, x):
    acts, layers, p = [], [], 0
    for o, k in _SHAPES:
        layers.append((flat[p:p + o * k].view(o, k), flat[p + o * k:p + o * k + o]))
        p += o * k + o
    turn = x[:, :, None] * (2.0 ** (torch.arange(12, device=x.device, dtype=torch.float64) - 1.0))
    turn = 2.0 * math.pi * (turn - torch.floor(turn))
    h = torch.stack([torch.sin(turn), torch.cos(turn)], dim=3).reshape(len(x), 216)
    h = torch.cat([h, torch.zeros((len(x), 8), device=x.device, dtype=torch.float64)], dim=1)
    acts.append(h)
    for w, b in layers[:4]:
        h = torch.relu(h @ w.t() + b)
        acts.append(h)
    return acts, layers, h @ layers[4][0].t() + layers[4][1]


def _exact_network(case, seed):
    x, t = _rows(case["n"], seed)
    flat = torch.from_numpy(_params(seed)).cuda().double()
    if case["kind"] == "predict":
        out = torch.empty((case["n"], 3), dtype=torch.float64, device="cuda")
        for a in range(0, case["n"], 1 << 17):
            _, _, y = _forward64(flat, x[a:a + (1 << 17)].double())
            out[a:a + (1 << 17)] = torch.clamp(torch.expm1(y[:, :3]), min=0.0)
        return out
    n, loss = case["n"], 0.0
    grads = [torch.zeros((o, k + 1), dtype=torch.float64, device="cuda") for o, k in _SHAPES]
    for a in range(0, n, 1 << 17):
        acts, layers, y = _forward64(flat, x[a:a + (1 << 17)].double())
        d = y[:, :3] - torch.log1p(torch.clamp(t[a:a + (1 << 17)].double(), min=0.0))
        loss += float((d * d).sum()) / (3 * n)
        delta = torch.zeros_like(y)
        delta[:, :3] = 2.0 * d / (3 * n)
        for i in range(4, -1, -1):
            grads[i][:, :-1] += delta.t() @ acts[i]
            grads[i][:, -1] += delta.sum(0)
            if i:
                delta = (delta @ layers[i][0]) * (acts[i] > 0)
    return {"grad": torch.cat([torch.cat([g[:, :-1].reshape(-1), g[:, -1]]) for g in grads]), "loss": loss}


def _exact_knn(case, seed):
    pos, q, rcap = _points(case, seed)
    p = torch.from_numpy(pos).cuda().double()
    d2 = torch.full((case["nq"], case["k"]), math.inf, dtype=torch.float64, device="cuda")
    kk, step = min(case["k"], case["n"]), max(1, (1 << 27) // case["n"])
    for a in range(0, case["nq"], step):
        c = torch.from_numpy(q[a:a + step]).cuda().double()
        d = torch.zeros((len(c), case["n"]), dtype=torch.float64, device="cuda")
        for axis in range(3):
            d += (c[:, axis, None] - p[None, :, axis]) ** 2
        best = torch.topk(d, kk, dim=1, largest=False, sorted=True).values
        d2[a:a + step, :kk] = torch.where(best <= rcap * rcap, best, torch.full_like(best, math.inf))
    return {"idx": None, "d2": d2, "count": None}


def exact(case, seed):
    """64-bit values of the network's outputs and of the neighbour distances.

    A frame has none that could be compared: photon paths, hits and the set of
    the k nearest photons are decisions taken in 32 bits, and where 64 bits
    decide otherwise the pixel is another estimate, not a better-rounded one."""
    if case["kind"] in ("predict", "grad"):
        return _exact_network(case, seed)
    if case["kind"] == "knn" and case["n"] * case["nq"] <= 1.5e11:
        return _exact_knn(case, seed)
    return None
