"""What the engine is timed on: the work that a program using it hands to the GPU.

Six kinds of call, each through the public entry points:

- "frame": one turn of the engine loop (DN_draw, DN_sync_gpu, DN_update_lighting), lit either where
  the camera looked or, with `relight`, on every exposed chunk of the map;
- "rays": one DNX_cast_rays batch (picking, visibility and collision queries);
- "edits": a frame that first applies sphere edits (DNX_shape_spheres) and so re-uploads chunks;
- "batch": one DNX_batch_update_lighting over many uneven volumes;
- "train" / "grad" / "predict": the learned radiance cache, online training with the prediction of
  every lit voxel, gradients of rows the program brings itself, and predictions of such rows.

The maps are seeded fBm terrains with boxes, in the sizes the benchmark and the tests use and odd
ones between them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from doonengine_amd import _lib, scenes
from doonengine_amd.volume import RC_NPARAM, Batch, RadianceCache, Volume

DEV = "cuda"


def _frame(name, chunks, image, direct, spec, bounces, samples, relight, glass=False):
    return {"name": name, "kind": "frame", "cx": chunks[0], "cy": chunks[1], "cz": chunks[2], "width": image[0],
            "height": image[1], "direct": direct, "spec": spec, "bounces": bounces, "samples": samples,
            "relight": relight, "glass": glass}


def listed():
    return [
        # the smallest loop: a few chunks in a thumbnail, all latency and launches
        _frame("frame_tiny", (4, 3, 4), (48, 40), 0, 15, 5, 1, False),
        # an ordinary small world in a small window, fixed shadow rays
        _frame("frame_256", (16, 16, 16), (256, 256), 16, 16, 5, 1, False),
        # a large world at full HD with the engine's default lighting, lit where the camera looks
        _frame("frame_1080p", (64, 32, 64), (1920, 1080), 0, 15, 5, 1, False),
        # the benchmark's frame: everything that can be seen from somewhere is lit, 32 shadow rays a voxel
        _frame("relight_1080p", (64, 32, 64), (1920, 1080), 32, 32, 4, 1, True),
        # mirrors, gloss and glass on a map of odd size, an odd window, two samples a voxel
        _frame("frame_glass", (37, 13, 29), (1023, 577), 0, 15, 5, 2, True, glass=True),
        # a large query batch of rays that have nothing in common
        {"name": "rays_2m", "kind": "rays", "cx": 32, "cy": 16, "cz": 32, "n": 2000003, "first": True},
        # 256 sphere edits a frame on a 128^3 map: edit, draw, re-upload, light
        {"name": "edits_256", "kind": "edits", "chunks": 16, "n": 256, "image": 256, "direct": 16},
        # many small worlds of uneven size lit by one launch
        {"name": "batch_24", "kind": "batch", "n": 24, "grid": 24, "direct": 16, "bounces": 4},
        # the radiance cache's online training at the benchmark's schedule: 8 steps, then every voxel predicted
        {"name": "cache_train", "kind": "train", "chunks": 16, "log2": 19, "rows": 131072, "steps": 8, "direct": 16},
        # gradients of rows that the program brings, read back for an optimiser of its own
        {"name": "cache_grad", "kind": "grad", "log2": 14, "rows": 65552},
        # a handful of predictions inside a serving loop, without allocations
        {"name": "predict_1k", "kind": "predict", "log2": 19, "rows": 1008, "noalloc": True},
        # predictions of a whole map's surface
        {"name": "predict_1m", "kind": "predict", "log2": 19, "rows": 1000016, "noalloc": False},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "rays", "edits", "batch", "train", "grad", "predict", "predict"])
    if kind == "frame":
        while True:
            cx, cy, cz = _log(rng, 3, 64), _log(rng, 3, 32), _log(rng, 3, 64)
            if cx * cy * cz <= 65536:
                break
        c = _frame("", (cx, cy, cz), (_log(rng, 33, 1920), _log(rng, 33, 1080)), rng.choice([0, 0, 1, 5, 16, 24, 32]),
                   rng.choice([15, 16, 32]), rng.randint(1, 5), rng.choice([1, 1, 2]), rng.random() < 0.5,
                   rng.random() < 0.25)
        del c["name"]
        return c
    if kind == "rays":
        return {"kind": kind, "cx": rng.randint(4, 40), "cy": rng.randint(3, 20), "cz": rng.randint(4, 40),
                "n": _log(rng, 64, 2000000), "first": rng.random() < 0.5}
    if kind == "edits":
        return {"kind": kind, "chunks": rng.randint(6, 16), "n": _log(rng, 1, 256), "image": rng.randint(64, 256),
                "direct": rng.choice([0, 16])}
    if kind == "batch":
        return {"kind": kind, "n": rng.randint(2, 24), "grid": rng.randint(8, 24), "direct": rng.choice([0, 7, 16]),
                "bounces": rng.randint(1, 4)}
    if kind == "train":
        return {"kind": kind, "chunks": rng.randint(6, 16), "log2": rng.randint(15, 19), "rows": 16 * _log(rng, 512, 8192),
                "steps": rng.randint(1, 8), "direct": rng.choice([0, 16])}
    if kind == "grad":
        return {"kind": kind, "log2": rng.randint(10, 16), "rows": 16 * _log(rng, 1, 4096)}
    rows = 16 * _log(rng, 1, 62500)
    return {"kind": kind, "log2": rng.randint(14, 19), "rows": rows, "noalloc": rows <= 262144 and rng.random() < 0.5}


# ---------------------------------------------------------------------------
# device memory of the engine and of torch, each as the other takes it


class _Out:
    """A tensor where the engine takes a device buffer."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


class _Dev:
    def __init__(self, vol, ptr, shape):
        self.vol = vol
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<i4", "data": (ptr, False), "version": 2}


def _view(vol, ptr, shape):
    """An int32 tensor over device memory of a volume, which lives at least as long as the tensor."""
    t = torch.as_tensor(_Dev(vol, ptr, shape), device=DEV)
    t.volume = vol
    return t


def _volume_state(s, vol):
    """Tile flags, chunk records and the voxel pool where they lie on the device."""
    v = vol.v
    key = (v.gpuMap, v.gpuChunks, v.gpuVoxels, v.voxelCap)
    if s.get("key") != key:          # the pool moves when it grows
        s["key"] = key
        s["views"] = (_view(vol, v.gpuMap, (vol.tiles,)), _view(vol, v.gpuChunks, (vol.tiles, 32)),
                      _view(vol, v.gpuVoxels, (int(v.voxelCap), 4)))
    return s["views"]


# ---------------------------------------------------------------------------
# maps


def _terrain(chunks, seed, glass=False):
    """Normal and albedo words (Z, Y, X) of a terrain with boxes, and its materials."""
    X, Y, Z = (8 * c for c in chunks)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    r = np.random.default_rng(seed)
    gx, gz = np.meshgrid(np.arange(X, dtype=np.float64), np.arange(Z, dtype=np.float64))
    f = scenes.fbm(gx / 64.0, gz / 64.0, seed)
    h = Y * 0.25 + min(0.3 * Y, 64.0) * f
    hz, hx = np.gradient(h)
    nrm = np.stack([-hx, np.ones_like(h), -hz], axis=-1)
    nrm /= np.linalg.norm(nrm, axis=-1, keepdims=True)
    mats = [scenes.Material(albedo=tuple(int(v) for v in r.integers(50, 230, 3))) for _ in range(4)]
    mats[3].emissive, mats[3].emission = True, 4.0
    if glass:
        mats[1].specular, mats[1].shininess, mats[1].reflect_type = 0.9, 60, 1
        mats[2].specular, mats[2].shininess = 0.3, 4
        mats.append(scenes.Material(albedo=(180, 220, 240), opacity=0.3))
    solid_mats = [0, 1, 2]
    q = np.quantile(h, [1 / 3, 2 / 3])
    band = (h >= q[0]).astype(np.uint32) + (h >= q[1])

    def words(m, n):
        return (scenes.pack_normal_word(np.asarray(m, np.uint32), np.asarray(n, np.float32))).astype(np.uint32)

    alb = np.array([(m.albedo[0] << 24) | (m.albedo[1] << 16) | (m.albedo[2] << 8) for m in mats], np.uint32)

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a, np.uint32).view(np.int32)).to(DEV)

    solid = torch.arange(Y, device=DEV)[None, :, None] < torch.from_numpy(h).to(DEV)[:, None, :]
    nw = torch.where(solid, dev(words(band, nrm))[:, None, :], -1)
    aw = torch.where(solid, dev(alb[band])[:, None, :], 0)
    boxes = max(2, min(2000, X * Z // 132))
    size = r.integers(2, max(3, min(40, X // 4, Y // 2, Z // 4)) + 1, (boxes, 3))
    at = r.random((boxes, 2))
    kind = r.integers(0, len(solid_mats) + (1 if glass else 0), boxes)
    up = words(np.arange(len(mats)), np.tile([0.0, 1.0, 0.0], (len(mats), 1))).view(np.int32)
    alb_i = alb.view(np.int32)
    for b in range(boxes):
        sx, sy, sz = (int(v) for v in size[b])
        ox, oz = int(at[b, 0] * max(1, X - sx)), int(at[b, 1] * max(1, Z - sz))
        oy = int(np.clip(h[oz + sz // 2, ox + sx // 2] - 0.3 * sy, 0, max(0, Y - sy)))
        m = 4 if kind[b] == 3 else solid_mats[kind[b]]
        nw[oz:oz + sz, oy:oy + sy, ox:ox + sx] = int(up[m])
        aw[oz:oz + sz, oy:oy + sy, ox:ox + sx] = int(alb_i[m])
    glow = torch.rand(nw.shape, device=DEV, generator=g) < 0.005
    glow &= nw != -1
    nw[glow] = (nw[glow] & 0x00FFFFFF) | (3 << 24)
    aw[glow] = int(alb_i[3])
    return nw.cpu().numpy().view(np.uint32), aw.cpu().numpy().view(np.uint32), mats


def _load(chunks, seed, glass=False, params=None):
    """A volume with its map resident on the GPU and the camera above one corner."""
    nw, aw, mats = _terrain(chunks, seed, glass)
    vol = Volume(chunks, min_chunks=chunks[0] * chunks[1] * chunks[2])
    for i, m in enumerate(mats):
        vol.set_material(i, emissive=m.emissive, emission=m.emission, specular=m.specular, shininess=m.shininess,
                         reflect_type=m.reflect_type, opacity=m.opacity, refract=1.3 if m.opacity < 1.0 else 1.0)
    vol.set_dense(nw, aw)
    vol.set_vec("camPos", (0.06 * chunks[0], 0.7 * chunks[1], 0.06 * chunks[2]))
    vol.set_vec("camOrient", (30.0, 45.0, 0.0))
    vol.set_vec("sunDir", (-1.0, 1.0, -1.0))
    for k, v in (params or {}).items():
        setattr(vol.v, k, v)
    vol.request_all()
    vol.sync()
    vol.mats_in = mats
    return vol


def _time(s):
    """The program's clock: a sixtieth of a second a frame."""
    s["t"] += 1.0 / 60.0
    return s["t"]


# ---------------------------------------------------------------------------
# rows of the radiance cache


def _rows(n, seed, extent=128.0):
    """Rows of the surface of a map, in runs of 32 neighbouring voxels as the lit chunks hold them."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    runs = (n + 31) // 32
    k = torch.arange(32, device=DEV)
    base = torch.randint(0, int(extent) // 8, (runs, 3), device=DEV, generator=g).double() * 8
    slope = torch.rand(runs, 1, device=DEV, generator=g) * 2 - 1
    half = torch.randint(0, 2, (runs, 1), device=DEV, generator=g) * 4
    x = (k % 8)[None, :].expand(runs, 32).double()
    z = (k // 8)[None, :] + half
    y = torch.clamp(torch.floor(3.5 + slope * (x - 3.5)), 0, 7)
    pos = torch.stack([base[:, 0:1] + x, base[:, 1:2] + y, base[:, 2:3] + z], -1) + 0.5
    nrm = torch.nn.functional.normalize(torch.stack([-slope, torch.ones_like(slope), 0 * slope], -1), dim=-1)
    alb = torch.rand(runs, 1, 3, device=DEV, generator=g) * 0.8 + 0.1
    s = torch.zeros(runs * 32, 16, device=DEV)
    s[:, 0:3] = pos.reshape(-1, 3)
    s[:, 3:6] = nrm.expand(runs, 32, 3).reshape(-1, 3)
    s[:, 6:9] = alb.expand(runs, 32, 3).reshape(-1, 3)
    s[:, 9:12] = torch.rand(runs * 32, 3, device=DEV, generator=g)
    s[:, 12] = (torch.rand(runs * 32, device=DEV, generator=g) > 0.02).float()
    s[:, 13:16] = torch.rand(runs * 32, 3, device=DEV, generator=g) * 0.2
    return s[:n].contiguous()


def _params(log2, seed):
    """Weights and table at the scale that training gives them: host arrays as DNX_rc_set_params takes them."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 77)
    w = torch.zeros(RC_NPARAM, device=DEV)
    for off, rows, ld, used_rows, used in ((0, 64, 48, 64, 38), (3072, 64, 64, 64, 64), (7168, 64, 64, 64, 64),
                                           (11264, 16, 64, 3, 64)):
        a = math.sqrt(6.0 / (used_rows + used))
        w[off:off + rows * ld].view(rows, ld)[:used_rows, :used] = \
            (torch.rand(used_rows, used, device=DEV, generator=g) * 2 - 1) * a
    t = torch.randn(32 << log2, device=DEV, generator=g) * 0.05
    return w.cpu().numpy(), t.cpu().numpy()


RES = [int(math.floor(16 * math.exp((math.log(256) - math.log(16)) / 15) ** l)) for l in range(16)]


def _exact_net(log2, seed, extent=128.0):
    """The cache's network in 64 bits: a function from rows to outputs, its four matrices and its table."""
    w, t = _params(log2, seed)
    w = torch.from_numpy(w).to(DEV).double()
    table = torch.from_numpy(t).to(DEV).double().view(16, 1 << log2, 2).requires_grad_()
    mats = [w[o:o + r * c].view(r, c).clone().requires_grad_()
            for o, r, c in ((0, 64, 48), (3072, 64, 64), (7168, 64, 64), (11264, 16, 64))]

    def forward(rows):
        rows = rows.double()
        x = torch.clamp(rows[:, 0:3] / extent, 0.0, 1.0)
        feats = []
        for l, n in enumerate(RES):
            p = x * n + 0.5
            c = torch.floor(p)
            f, c, S = p - c, c.long(), n + 2
            acc = 0
            for k in range(8):
                o = [(k >> a) & 1 for a in range(3)]
                q = [c[:, a] + o[a] for a in range(3)]
                if S ** 3 <= 1 << log2:
                    i = q[0] + S * (q[1] + S * q[2])
                else:
                    i = (q[0] ^ (q[1] * 2654435761) ^ (q[2] * 805459861)) & ((1 << log2) - 1)
                wt = 1
                for a in range(3):
                    wt = wt * (f[:, a] if o[a] else 1 - f[:, a])
                acc = acc + wt[:, None] * table[l][i]
            feats.append(acc)
        h = torch.cat(feats + [rows[:, 3:9], torch.zeros(rows.shape[0], 10, device=DEV, dtype=torch.float64)], 1)
        for m in mats[:3]:
            h = torch.relu(h @ m.t())
        return (h @ mats[3].t())[:, :3]

    return forward, mats, table


# ---------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "t": 100.0 + (seed % 997)}
    if kind == "frame":
        chunks = (case["cx"], case["cy"], case["cz"])
        vol = _load(chunks, seed, case["glass"], {"numSpecularRays": case["spec"], "numDirectRays": case["direct"],
                                                  "diffuseBounceLimit": case["bounces"]})
        w, h = case["width"], case["height"]
        s["vol"], s["image"] = vol, torch.zeros(h, w, 4, device=DEV)
        s["out"] = _Out(s["image"])
        s["view"] = vol.view_projection(h / w)
    elif kind == "rays":
        chunks = (case["cx"], case["cy"], case["cz"])
        s["vol"] = _load(chunks, seed)
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        n = case["n"]
        box = torch.tensor(chunks, device=DEV, dtype=torch.float32)
        s["from"] = (torch.rand(n, 3, device=DEV, generator=g) * torch.tensor([1.0, 0.6, 1.0], device=DEV) +
                     torch.tensor([0.0, 0.3, 0.0], device=DEV)) * box
        d = torch.nn.functional.normalize(torch.randn(n, 3, device=DEV, generator=g), dim=1)
        # no component is zero (the walk's rule for such a direction has no end), as the engine's own
        # rays see to with their 1e-4
        s["dir"] = torch.where(d.abs() < 1e-4, torch.full_like(d, 1e-4), d).contiguous()
        s["hits"] = torch.zeros(n, 10, device=DEV, dtype=torch.int32)
    elif kind == "edits":
        c = case["chunks"]
        vol = _load((c, c, c), seed, params={"numSpecularRays": 16, "numDirectRays": case["direct"]})
        scene = scenes.Scene("", (c, c, c), None, None, vol.mats_in, (0, 0, 0), (0, 0, 0))
        s["edits"] = [vol.sphere_edits(scenes.sphere_edits(scene, (seed * 16 + k) % (1 << 30), case["n"]))
                      for k in range(16)]
        s["at"] = 0
        w = case["image"]
        s["vol"], s["image"] = vol, torch.zeros(w, w, 4, device=DEV)
        s["out"] = _Out(s["image"])
        s["view"] = vol.view_projection(1.0)
    elif kind == "batch":
        vols, s["mark"], s["of"] = [], [], []
        span = case["grid"] - 3
        for k in range(case["n"]):
            chunks = tuple(4 + int(span * float(scenes.uniform01(k, a, seed=977))) for a in range(3))
            vols.append(_load(chunks, seed * 64 + k, params={"numSpecularRays": 16, "numDirectRays": case["direct"],
                                                             "diffuseBounceLimit": case["bounces"]}))
            s["mark"].append(int(10 * 4000 ** float(scenes.uniform01(k, 5, seed=977))))
            s["of"].append({})
        s["vols"], s["batch"] = vols, Batch(vols)
    elif kind == "train":
        c = case["chunks"]
        vol = _load((c, c, c), seed, params={"numSpecularRays": 16, "numDirectRays": case["direct"]})
        vol.mark_visible(32768)
        vol.sync()
        s["vol"] = vol
        s["slots"] = 40 * c * c              # requests the prediction buffer holds: more than such a map has
        s["rc"] = RadianceCache(vol, log2Table=case["log2"], samplesPerFrame=case["rows"], seed=seed % 65536,
                                lrDecaySteps=256.0, lrDecayPower=1.0, emaDecay=0.9994)
        s["pred"] = torch.zeros(s["slots"] * 32, 4, device=DEV)
        s["w"] = torch.zeros(RC_NPARAM, pin_memory=True)
    else:
        s["vol"] = Volume((4, 3, 4), min_chunks=48)
        s["rc"] = RadianceCache(s["vol"], log2Table=case["log2"], extent=128.0)
        s["rc"].set_params(*_params(case["log2"], seed))
        s["rows"] = _rows(case["rows"], seed)
        if kind == "grad":
            s["dw"] = torch.zeros(RC_NPARAM, pin_memory=True)
            s["dt"] = torch.zeros(32 << case["log2"], pin_memory=True)
        else:
            s["pred"] = torch.zeros(case["rows"], 4, device=DEV)
            s["out"], s["in"] = _Out(s["pred"]), _Out(s["rows"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("frame", "edits"):
        vol = s["vol"]
        if kind == "edits":
            vol.shape_spheres(s["edits"][s["at"] % len(s["edits"])])
            s["at"] += 1
        h, w = s["image"].shape[:2]
        vol.draw(s["out"], w, h, *s["view"])
        if case.get("relight"):
            vol.mark_visible(32768)
        vol.sync()
        vol.update_lighting(case.get("samples", 1), 1000, _time(s))
        return (s["image"],) + _volume_state(s, vol)
    if kind == "rays":
        vol = s["vol"]
        vol.lib.DNX_cast_rays(vol.ptr, case["n"], s["from"].data_ptr(), s["dir"].data_ptr(), case["first"],
                              s["hits"].data_ptr())
        return s["hits"]
    if kind == "batch":
        for v, m in zip(s["vols"], s["mark"]):
            v.mark_visible(m)
            v.sync()
        s["batch"].update_lighting(1, 1000, _time(s))
        return [_volume_state(o, v)[2] for o, v in zip(s["of"], s["vols"])]
    rc = s["rc"]
    if kind == "train":
        rc.train_frame(_time(s), case["steps"])
        rc.lib.DNX_rc_predict_requests(rc.ptr, s["pred"].data_ptr(), s["slots"])
        rc.lib.DNX_rc_get_params(rc.ptr, s["w"].data_ptr(), None, None, None)
        return {"prediction": s["pred"], "weights": s["w"]}
    if kind == "grad":
        rc.lib.DNX_rc_train_samples(rc.ptr, s["rows"].data_ptr(), case["rows"], False)
        rc.lib.DNX_rc_get_params(rc.ptr, None, None, s["dw"].data_ptr(), s["dt"].data_ptr())
        return {"weights": s["dw"], "table": s["dt"]}
    if case["noalloc"]:
        rc.predict_samples_noalloc(s["in"], case["rows"], s["out"])
    else:
        rc.predict_samples(s["in"], case["rows"], s["out"])
    return s["pred"]


def exact(case, seed):
    """The cache's outputs in 64 bits. Frames, rays, edits and batches give packed words, which have no value
    beside their own (a frame's picture shows what its passes lit: a path tracer's time in 64 bits), and a
    training frame draws its own rows."""
    kind = case["kind"]
    if kind not in ("grad", "predict"):
        return None
    forward, mats, table = _exact_net(case["log2"], seed)
    rows = _rows(case["rows"], seed)
    if kind == "predict":
        out = torch.zeros(case["rows"], 4, device=DEV, dtype=torch.float64)
        with torch.no_grad():
            for i in range(0, case["rows"], 65536):
                r = rows[i:i + 65536]
                out[i:i + 65536, :3] = forward(r) + r[:, 13:16].double()
        out[:, 3] = rows[:, 12].double()
        return out
    y = forward(rows)
    loss = (0.5 * (y - rows[:, 9:12].double()) ** 2 * rows[:, 12:13].double()).sum() / case["rows"]
    loss.backward()
    return {"weights": torch.cat([m.grad.reshape(-1) for m in mats]).cpu(), "table": table.grad.reshape(-1).cpu()}


def work(case):
    """Bytes a pass reads and writes at the least, and its floating operations: about 24 per step of a ray
    (a step of either grid: three compares, selects and adds), with the steps that terrains like these take."""
    kind = case["kind"]
    if kind in ("frame", "edits"):
        if kind == "edits":
            c = case["chunks"]
            cols, px, tiles = 64 * c * c, case["image"] ** 2, c ** 3
            lit, rays = min(px / 4, 14.0 * cols), case["direct"] or 1
        else:
            cols, px, tiles = 64 * case["cx"] * case["cz"], case["width"] * case["height"], case["cx"] * case["cy"] * case["cz"]
            lit = 14.0 * cols if case["relight"] else min(px / 16, 14.0 * cols)
            rays = (case["direct"] or 1) * case["samples"]
        rays += 2.5 * case.get("samples", 1)
        return {"bytes": 16.0 * px + 32.0 * lit + 12.0 * tiles, "flops": 24.0 * (6.0 * lit * rays + 40.0 * px)}
    if kind == "rays":
        return {"bytes": 64.0 * case["n"], "flops": 24.0 * 30.0 * case["n"]}
    if kind == "batch":
        lit = case["n"] * 14.0 * 64.0 * (case["grid"] / 2) ** 2
        return {"bytes": 32.0 * lit, "flops": 24.0 * 6.0 * lit * (case["direct"] or 1) + 24.0 * 15.0 * lit}
    n, forward = case["rows"], 2.0 * (38 * 64 + 64 * 64 * 2 + 64 * 3) + 16 * 8 * 6
    if kind == "predict":
        return {"bytes": n * 80.0, "flops": forward * n}
    if kind == "grad":
        return {"bytes": n * 64.0 + 4.0 * (32 << case["log2"]) + 4.0 * RC_NPARAM, "flops": 3.0 * forward * n}
    # a training step sweeps the parameters and moments of the table's entries once
    return {"bytes": case["steps"] * (n * 128.0 + 40.0 * (32 << case["log2"])), "flops": case["steps"] * 3.0 * forward * n}
