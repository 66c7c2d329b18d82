"""Workloads of the voxel ray tracer, as a program that uses it runs them.

A case is a dict of plain values; its `kind` says which calls one pass makes:

  visibility  primary visibility of `cams` cameras into a device buffer
  frame       one plain frame: visibility, then one-bounce GI at `spp`
  cache       one neural-cache frame of a cache that has trained on the view
  batch       one captured frame of `cams` cameras (plain GI)
  cache_batch one captured frame of `cams` cameras with the cache, trained
              jointly on every camera
  build       SVO build of a loaded scene and its first SVO view
  edit        an object moves (destroy, create, SVO update), then a frame
  rays        host rays through the SVO (tgx_svo_trace)
  shade       the shading pass over a visibility buffer
  fit         one Adam step of the cache on host samples, then inference on
              held-out samples

Scenes are the library's own generators: one 32^3 Bernoulli object, or
`objects` noise-filled objects of up to `extent` clusters per axis in a
`world`^3 volume. `seed` picks the scene, the cameras, the sun and the rays.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tg_amd as T

SUN_RANGE = 1024.0          # range of bounce and shadow rays
HIDDEN = 64
FORWARD_FLOPS = 2 * (78 * HIDDEN + 3 * HIDDEN * HIDDEN + HIDDEN * 3)


# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------

def _noise(objects: int, extent: int, world: int, luts: int = 1) -> dict:
    return {"scene": "noise", "objects": objects, "extent": extent, "world": world, "luts": luts}


_OBJECT = {"scene": "object", "objects": 1, "extent": 4, "world": 64, "luts": 1}
_HALL = _noise(512, 8, 512)            # the 512-object scene of the 1080p frame
_WORLD = _noise(4096, 32, 4096, 64)    # the 4096-object world of the batched frame


def listed() -> list[dict]:
    return [
        # a model viewer: one small object in a thumbnail, the smallest call
        {"name": "visibility_object_256", "kind": "visibility", **_OBJECT, "w": 256, "h": 256, "cams": 1},
        # the visibility buffer of a full-HD view, read by a renderer of the caller's own
        {"name": "visibility_1080p", "kind": "visibility", **_HALL, "w": 1920, "h": 1080, "cams": 1},
        # a preview window of odd size over a lighter scene, few samples
        {"name": "frame_853x479", "kind": "frame", **_noise(200, 8, 384), "depth": 10, "w": 853, "h": 479, "spp": 2},
        # the plain full-HD frame: visibility and 4 bounce samples per pixel
        {"name": "frame_1080p", "kind": "frame", **_HALL, "depth": 11, "w": 1920, "h": 1080, "spp": 4},
        # the same view rendered through the irradiance cache while it keeps training
        {"name": "cache_1080p", "kind": "cache", **_HALL, "depth": 11, "w": 1920, "h": 1080, "spp": 4,
         "train_batch": 16384, "frames": 160},
        # sixteen cameras of a large world as one captured frame, plain GI: the largest call
        {"name": "batch_16x1080p", "kind": "batch", **_WORLD, "depth": 12, "w": 1920, "h": 1080, "spp": 4, "cams": 16},
        # the same sixteen cameras through a jointly trained cache
        {"name": "cache_batch_16x1080p", "kind": "cache_batch", **_WORLD, "depth": 12, "w": 1920, "h": 1080,
         "spp": 4, "cams": 16, "train_batch": 4096, "frames": 60},
        # a level has been loaded: its SVO is built and shown once
        {"name": "build_512_objects", "kind": "build", **_HALL, "depth": 11, "w": 1920, "h": 1080},
        # an editor or a game moves one object per frame in a 540p window
        {"name": "edit_960x540", "kind": "edit", **_noise(128, 6, 320), "depth": 10, "w": 960, "h": 540, "spp": 1},
        # line-of-sight or physics queries from host code
        {"name": "rays_100003", "kind": "rays", **_HALL, "depth": 11, "rays": 100003},
        # deferred shading of a full-HD visibility buffer
        {"name": "shade_1080p", "kind": "shade", **_HALL, "w": 1920, "h": 1080},
        # offline fitting of a cache to sampled irradiance, a batch of odd length
        {"name": "fit_10000", "kind": "fit", "samples": 10000},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _hall(rng) -> dict:
    extent = rng.randint(3, 10)
    objects = min(_log(rng, 24, 900), 300000 // extent ** 3)
    return _noise(objects, extent, rng.randint(160, 640), rng.choice((1, 1, 4)))


def draw(rng) -> dict:
    kind = rng.choice(("visibility", "visibility", "frame", "frame", "frame", "cache", "cache", "batch", "cache_batch",
                       "build", "edit", "rays", "shade", "fit"))
    if kind == "fit":
        return {"kind": kind, "samples": _log(rng, 300, 70000)}
    w = _log(rng, 160, 2600)
    h = max(90, int(w * rng.uniform(0.45, 0.8)))
    depth = rng.choice((10, 11))
    c = {"kind": kind, **_hall(rng), "w": w, "h": h}
    if kind == "visibility":
        if rng.random() < 0.3:
            c.update(_OBJECT)
        c["cams"] = rng.choice((1, 1, 2, 5))
    elif kind == "frame":
        c.update(depth=depth, spp=rng.choice((1, 2, 3, 4, 8)))
    elif kind == "cache":
        c.update(depth=depth, spp=4, train_batch=rng.choice((4096, 8192, 16384)), frames=rng.randint(60, 160))
    elif kind in ("batch", "cache_batch"):
        c.update(_noise(_log(rng, 300, 3000), rng.randint(8, 24), rng.randint(1000, 4000), rng.choice((1, 16, 64))))
        c.update(depth=12, w=min(w, 1600), h=min(h, 900), spp=4, cams=rng.randint(2, 12))
        if kind == "cache_batch":
            c.update(train_batch=rng.choice((4096, 8192)), frames=rng.randint(20, 60))
    elif kind == "build":
        c.update(depth=depth)
    elif kind == "edit":
        c.update(depth=depth, spp=1, objects=min(c["objects"], 256))
    elif kind == "rays":
        del c["w"], c["h"]
        c.update(depth=depth, rays=_log(rng, 1000, 1000000))
    return c


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

class State(dict):
    """What the caller's program holds: a context, its buffers and, for
    batched frames, the captured graph."""

    def __del__(self):
        graph, ctx = self.get("graph"), self.get("ctx")
        if graph is not None:
            graph.destroy()
        if ctx is not None:
            ctx.close()


def _params(case: dict, seed: int):
    if case["scene"] == "object":
        return T.single_object_params(seed)
    return T.noise_objects_params(seed=seed, n_objects=case["objects"], max_extent=case["extent"],
                                  world=float(case["world"]), n_luts=case["luts"])


def _buffers(s: State, case: dict, cams: int = 1, gi: bool = True) -> None:
    shape = (cams, case["h"], case["w"])
    s["vis"] = torch.zeros(shape, dtype=torch.int64, device="cuda")
    if gi:
        s["radiance"] = torch.zeros((*shape, 3), dtype=torch.float32, device="cuda")
        s["irradiance"] = torch.zeros((*shape, 3), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()  # the context's stream does not wait for torch's


def _corner(case: dict, cam: np.ndarray) -> np.ndarray:
    """Min corner of a root centred on the camera."""
    return np.floor(cam[0]["camera"][:3]) - float(1 << (case["depth"] - 1))


def _nrc(case: dict, seed: int, flags: int) -> np.ndarray:
    steps = 65536 // case["train_batch"]
    return T.nrc_config(scale=1.0 / case["world"], seed=seed & 0xFFFFFFFF, train_samples=65536,
                        train_batch=case["train_batch"], train_spp=4, fallback_threshold=16.0,
                        fallback_min_samples=0, cell_size=8, flags=flags, ema_decay=0.996 if steps <= 4 else 0.999)


def prepare(case: dict, seed: int) -> State:
    kind = case["kind"]
    s = State(kind=kind, case=case)
    ctx = s["ctx"] = T.Context(0)
    if kind == "fit":
        return _prepare_fit(s, case, seed)
    params = _params(case, seed)
    if case["scene"] == "object":
        ctx.upload(T.generate_scene(params))
    else:
        ctx.generate_scene_device(params)
    w, h = case.get("w", 1920), case.get("h", 1080)
    cams = s["cams"] = np.concatenate([T.generate_camera(params, i, w, h) for i in range(case.get("cams", 1))])
    s["sun"] = T.seeded_sun(seed)
    if "spp" in case:
        s["gi"] = T.gi_params(s["sun"], spp=case["spp"], max_distance=SUN_RANGE, frame=seed & 0xFFFF)
    if kind == "visibility":
        _buffers(s, case, case["cams"], gi=False)
    elif kind == "frame":
        ctx.svo_build(_corner(case, cams), case["depth"])
        _buffers(s, case)
    elif kind == "cache":
        ctx.svo_build(_corner(case, cams), case["depth"])
        _buffers(s, case)
        ctx.nrc_create(_nrc(case, seed, T.NRC_FLAG_FALLBACK_VS_TRACER))
        for _ in range(case["frames"]):
            run(s)
    elif kind in ("batch", "cache_batch"):
        ctx.svo_build(_corner(case, cams), case["depth"])
        _buffers(s, case, case["cams"])
        flags = 0
        if kind == "cache_batch":
            flags = T.FRAME_NEURAL
            ctx.nrc_create(_nrc(case, seed, T.NRC_FLAG_FALLBACK_VS_TRACER | T.NRC_FLAG_JOINT_TRAINING))
        s["graph"] = ctx.frame_graph(cams, w, h, s["gi"], s["vis"].data_ptr(), s["radiance"].data_ptr(),
                                     s["irradiance"].data_ptr(), flags=flags)
        for _ in range(case.get("frames", 0)):
            s["graph"].launch()
    elif kind == "build":
        s["corner"] = _corner(case, cams)
        _buffers(s, case, gi=False)
    elif kind == "edit":
        _prepare_edit(s, case, params, cams)
    elif kind == "rays":
        ctx.svo_build(_corner(case, cams), case["depth"])
        rng = np.random.default_rng(seed)
        d = rng.normal(size=(case["rays"], 3))
        s["origins"] = rng.uniform(0.0, case["world"], (case["rays"], 3)).astype(np.float32)
        s["directions"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    elif kind == "shade":
        _buffers(s, case, gi=False)
        s["rgba"] = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        ctx.visibility_device(cams, w, h, s["vis"].data_ptr())
        s["shading"] = T.shade_params(light_dir=tuple(float(x) for x in s["sun"]), roughness=-1.0)
    ctx.synchronize()
    return s


def _prepare_edit(s: State, case: dict, params, cams: np.ndarray) -> None:
    """The scene as a dynamic one, object by object; the host keeps each
    object's voxels, as an editor does."""
    ctx = s["ctx"]
    scene = ctx.scene_export(params)
    ctx.scene_reserve(scene.objects.size, scene.n_clusters, scene.luts)
    bits, mats = scene.bits.reshape(-1, 16), scene.materials.reshape(-1, 512)
    s["objects"] = []
    for ob in scene.objects:
        n = int(np.prod(ob["n_cluster_pointers_per_dim"].astype(np.int64)))
        f = int(ob["first_cluster_pointer"])
        o = {"extent": ob["n_cluster_pointers_per_dim"].copy(), "translation": ob["translation"].copy(),
             "rotation": ob["rotation"].copy(), "lut": int(ob["lut_idx"]), "bits": bits[f:f + n].copy(),
             "materials": mats[f:f + n].copy()}
        o["idx"] = ctx.object_create(o["extent"], o["translation"], o["rotation"], o["lut"], o["bits"], o["materials"])
        s["objects"].append(o)
    s["turn"] = 0
    ctx.svo_build(_corner(case, cams), case["depth"])
    _buffers(s, case)


def _fit_samples(rng, n: int):
    """Surface samples (position in the unit-scaled 512^3 world, face normal,
    albedo) of a smooth irradiance field."""
    p = rng.uniform(0.0, 512.0, (n, 3)).astype(np.float32)
    nrm = np.zeros((n, 3), np.float32)
    nrm[np.arange(n), rng.integers(0, 3, n)] = rng.choice((-1.0, 1.0), n)
    albedo = rng.uniform(0.05, 0.95, (n, 3)).astype(np.float32)
    a = rng.uniform(0.5, 2.0, (3, 3))
    t = 0.2 * (1.2 + np.sin(p.astype(np.float64) @ a * (2 * np.pi / 512.0))) * (1.0 + 0.3 * nrm.sum(1, keepdims=True))
    return p, nrm, albedo, t.astype(np.float32)


def _prepare_fit(s: State, case: dict, seed: int) -> State:
    rng = np.random.default_rng(seed)
    s["train"] = _fit_samples(rng, case["samples"])
    s["held"] = _fit_samples(rng, case["samples"])[:3]
    s["ctx"].nrc_create(T.nrc_config(scale=1.0 / 512, seed=seed & 0xFFFFFFFF))
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------

def run(s: State):
    ctx, case, kind = s["ctx"], s["case"], s["kind"]
    if kind == "fit":
        loss, grad = ctx.nrc_train_batch(*s["train"], want_grad=True)
        return {"loss": loss, "grad": grad, "irradiance": ctx.nrc_infer(*s["held"])}
    if kind == "rays":
        hits = ctx.svo_trace(s["origins"], s["directions"], SUN_RANGE)
        return {k: hits[k] for k in ("hit", "distance", "block", "voxel", "normal", "steps")}
    if kind in ("batch", "cache_batch"):
        s["graph"].launch()
        return {k: s[k] for k in ("vis", "radiance", "irradiance")}
    w, h, vis = case["w"], case["h"], s["vis"].data_ptr()
    if kind == "visibility":
        ctx.visibility_device(s["cams"], w, h, vis)
        return s["vis"]
    if kind == "shade":
        ctx.shade_device(s["cams"], w, h, vis, s["shading"], s["rgba"].data_ptr())
        return s["rgba"]
    if kind == "build":
        ctx.svo_build(s["corner"], case["depth"])
        info = ctx.svo_info()
        ctx.svo_visibility_device(s["cams"], w, h, vis)
        return {"vis": s["vis"], "nodes": int(info["n_nodes"]), "leaves": int(info["n_leaves"]),
                "list_entries": int(info["n_list_entries"])}
    out = {k: s[k] for k in ("vis", "radiance", "irradiance")}
    if kind == "edit":
        s["turn"] += 1
        o = s["objects"][s["turn"] * 7 % len(s["objects"])]
        ctx.object_destroy(o["idx"])
        o["translation"][s["turn"] % 3] += np.float32(3.0 if s["turn"] % 2 else -3.0)
        o["idx"] = ctx.object_create(o["extent"], o["translation"], o["rotation"], o["lut"], o["bits"], o["materials"])
        out["reused"], out["sampled"] = ctx.svo_update()
    if kind == "cache":
        ctx.nrc_frame_device(s["cams"], w, h, s["gi"], vis, s["radiance"].data_ptr(), s["irradiance"].data_ptr())
    else:
        ctx.frame_device(s["cams"], w, h, s["gi"], vis, s["radiance"].data_ptr(), s["irradiance"].data_ptr())
    return out


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------

def work(case: dict) -> dict:
    """Bytes: the scene's object records, cluster maps (8 B) and solid bits
    (64 B per cluster) read once, each output written once. Flops: the
    cache's products (every pixel inferred, 65536 samples trained)."""
    kind = case["kind"]
    if kind == "fit":
        n = case["samples"]
        return {"bytes": n * (36 + 12 + 36 + 12) + 4 * 18624 * 4, "flops": 4 * FORWARD_FLOPS * n}
    clusters = 64 if case["scene"] == "object" else case["objects"] * ((case["extent"] + 1) / 2) ** 3
    scene = 96 * case["objects"] + 72 * clusters
    if kind == "rays":
        return {"bytes": case["rays"] * (24 + 44) + scene, "flops": 0}
    px = case["w"] * case["h"] * case.get("cams", 1)
    if kind == "visibility":
        return {"bytes": scene + 8 * px, "flops": 0}
    if kind == "shade":
        return {"bytes": 24 * px + 96 * case["objects"] + 8 * clusters, "flops": 0}
    if kind == "build":
        # materials read; bits and the materials of about 40 % solid voxels written
        return {"bytes": scene + 512 * clusters + 64 * clusters + 2 * 205 * clusters + 8 * px, "flops": 0}
    flops = 0
    if kind in ("cache", "cache_batch"):
        flops = FORWARD_FLOPS * (px + 3 * 65536 * case.get("cams", 1))
    return {"bytes": scene + 32 * px, "flops": flops}


# --------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------

def exact(case: dict, seed: int):
    """64-bit values of the shading pass and of the cache's fit step. The
    other kinds return whole words, or radiance sums over thousands of
    traversed rays, which plain numpy does not walk in seconds."""
    if case["kind"] == "fit":
        return _exact_fit(case, seed)
    if case["kind"] == "shade":
        return _exact_shade(case, seed)
    return None


def _encode(p, nrm, albedo, scale):
    x = p.astype(np.float64) * scale
    f = np.zeros((p.shape[0], 96))
    for a in range(3):
        for k in range(12):
            f[:, 24 * a + 2 * k] = np.sin(2.0 ** k * np.pi * x[:, a])
            f[:, 24 * a + 2 * k + 1] = np.cos(2.0 ** k * np.pi * x[:, a])
    f[:, 72:75], f[:, 75:78], f[:, 78] = nrm, albedo, 1.0
    return f


def _layers(flat):
    out, o = [], 0
    for shape in ((96, 64), (64, 64), (64, 64), (64, 64), (64, 3)):
        out.append(flat[o:o + shape[0] * shape[1]].reshape(shape))
        o += shape[0] * shape[1]
    return out


def _forward(ws, x):
    acts = [x]
    for w in ws[:-1]:
        acts.append(np.maximum(acts[-1] @ w, 0.0))
    return acts, acts[-1] @ ws[-1]


def _exact_fit(case: dict, seed: int):
    s = prepare(case, seed)
    flat = s["ctx"].nrc_params().astype(np.float64)
    ws = _layers(flat)
    p, nrm, albedo, t = s["train"]
    acts, y = _forward(ws, _encode(p, nrm, albedo, 1.0 / 512))
    d = y - t
    n = d.size
    loss = float((d * d).sum() / n)
    dz, grads = 2.0 * d / n, []
    for layer in range(4, -1, -1):
        grads.append(acts[layer].T @ dz)
        if layer:
            dz = (dz @ ws[layer].T) * (acts[layer] > 0.0)
    g = np.concatenate([x.ravel() for x in reversed(grads)])
    # Adam's first step: m / (1 - b1) = g, v / (1 - b2) = g^2
    stepped = _layers(flat - 1e-3 * g / (np.abs(g) + 1e-8))
    _, held = _forward(stepped, _encode(*s["held"], 1.0 / 512))
    return {"loss": loss, "grad": g, "irradiance": np.maximum(held, 0.0)}


def _unit(v):
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _exact_shade(case: dict, seed: int):
    s = prepare(case, seed)
    ctx, w, h = s["ctx"], case["w"], case["h"]
    scene = ctx.scene_arrays()
    cam = s["cams"][0]
    words = s["vis"].reshape(-1).cpu().numpy().view(np.uint64)
    prm = s["shading"][0]
    pos = cam["camera"][:3].astype(np.float64)
    corner = {k: cam["ray_" + k][:3].astype(np.float64) for k in ("bl", "br", "tl", "tr")}
    out = np.empty((w * h, 4))
    out[:] = prm["miss"].astype(np.float64)
    light = _unit(prm["light_dir"].astype(np.float64))
    radiance, ambient = float(prm["light_radiance"]), float(prm["ambient"])
    metallic = float(prm["metallic"])
    visible = np.flatnonzero((words >> np.uint64(40)).astype(np.float64) < 16777215.0)
    for i in np.array_split(visible, max(1, visible.size // 200000)):
        word = words[i]
        depth = (word >> np.uint64(40)).astype(np.float64) / 16777215.0
        cptr = ((word >> np.uint64(9)) & np.uint64(0x7FFFFFFF)).astype(np.int64)
        v = (word & np.uint64(511)).astype(np.int64)
        cidx = scene.cluster_pointers[cptr].astype(np.int64)
        ob = scene.objects[scene.cluster_idx_to_object[cidx]]
        lut = scene.luts[256 * ob["lut_idx"].astype(np.int64) + scene.materials[512 * cidx + v]]
        dims = ob["n_cluster_pointers_per_dim"].astype(np.int64)
        rel = cptr - ob["first_cluster_pointer"]
        cell = np.stack([rel % dims[:, 0], rel // dims[:, 0] % dims[:, 1], rel // (dims[:, 0] * dims[:, 1])], 1)
        rot = ob["rotation"].reshape(-1, 4, 4).transpose(0, 2, 1)[:, :3, :3].astype(np.float64)
        inv = np.linalg.inv(rot)
        fx = ((i % w) + 0.5)[:, None] / w
        fy = 1.0 - ((i // w) + 0.5)[:, None] / h
        ray = ((corner["bl"] * (1 - fy) + corner["tl"] * fy) * (1 - fx)
               + (corner["br"] * (1 - fy) + corner["tr"] * fy) * fx)
        o = (inv @ (pos - ob["translation"].astype(np.float64))[..., None])[..., 0] + 4.0 * dims - 8.0 * cell
        d = _unit((inv @ ray[..., None])[..., 0])
        lo = np.stack([v % 8, v // 8 % 8, v // 64], 1).astype(np.float64)
        with np.errstate(divide="ignore", invalid="ignore"):
            a, b = (lo - o) / d, (lo + 1.0 - o) / d
        enter, leave = np.minimum(a, b).max(1), np.maximum(a, b).min(1)
        hit = o + np.maximum(enter, 0.0)[:, None] * d
        off = hit - (lo + 0.5)
        axis = np.abs(off).argmax(1)
        n = np.zeros_like(off)
        n[np.arange(i.size), axis] = np.sign(off[np.arange(i.size), axis])
        n = _unit((rot @ n[..., None])[..., 0])
        n[~((leave > 0.0) & (enter <= leave))] = 0.0
        view = _unit(-ray * (depth * float(cam["far_plane"]))[:, None])
        albedo = lut["albedo"].astype(np.float64)
        rough = lut["roughness"].astype(np.float64) if prm["roughness"] < 0 else np.full(i.size, float(prm["roughness"]))
        half = _unit(view + light)
        hn, ln, nv = (np.clip(x, 0.0, 1.0) for x in ((half * n).sum(1), (n * light).sum(1), (n * view).sum(1)))
        a2 = rough ** 4
        dist = a2 / (np.pi * (hn * hn * (a2 - 1.0) + 1.0) ** 2)
        base = 1.0 - rough
        f = base + (1.0 - base) * (1.0 - nv) ** 5
        k = (rough + 1.0) ** 2 / 8.0
        g = nv / (nv * (1 - k) + k) * (ln / (ln * (1 - k) + k))
        spec = 0.04 * (1.0 - metallic) + albedo * metallic
        sf = dist * f * g / np.maximum(4.0 * nv * ln, 0.001)
        lit = ((((1.0 - f) * (1.0 - metallic))[:, None] * albedo / np.pi + spec * sf[:, None]) * radiance * ln[:, None])
        out[i, :3] = ambient * albedo + lit
        out[i, 3] = 1.0
    return out.reshape(h, w, 4)
