"""The performance cases of the ray-tracing library: what its users call, through the public entry points.

  closest / any   a batch of rays against one mesh (Blas.trace_closest, Blas.trace_any): picking, probes, baking,
                  camera and shadow rays over terrain
  world           PackedRay buffers against an instanced scene (World.trace_closest_packed, trace_any_packed)
  batch           many meshes, each with rays of its own, in one launch (BatchSet.trace_closest)
  frame           the path tracer: progressive frames, or one realtime frame (PathTracer.render, render_realtime)
  infer / train   the radiance cache's two directions (RadianceCache.infer, RadianceCache.train)

Every traced result is pinned bit for bit by the library's own tests, so those cases compare exactly; the radiance
cache computes in bfloat16 and has tolerances.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "atlas-engine_amd"))

import atlas_rt  # noqa: E402
from atlas_rt import _abi  # noqa: E402
from atlas_rt import workloads as W  # noqa: E402

BATCH_KERNEL = _abi.KERNEL_BVH2_PERSISTENT | _abi.KERNEL_LEAF_BATCH
TRAIN_RATE = 1e-2
EVENING_SUN = np.array([0.8, 0.3, 0.35]) / np.linalg.norm([0.8, 0.3, 0.35])  # low enough for terrain to cast shadows


def listed():
    return [
        # a click in an editor viewport: a handful of rays against one small mesh, all of it latency
        {"name": "pick", "kind": "closest", "scene": "soup", "tris": 1024, "rays": 37},
        # probe or sensor rays of one frame: too few to fill the chip
        {"name": "probes", "kind": "closest", "scene": "soup", "tris": 20011, "rays": 5003},
        # incoherent rays over a random soup, the library's headline workload
        {"name": "soup", "kind": "closest", "scene": "soup", "tris": 65536, "rays": 1048576},
        # coherent camera rays over a terrain of 1,048,352 triangles
        {"name": "terrain", "kind": "closest", "scene": "height", "grid": 725, "width": 1920, "height": 1080},
        # camera rays of a frame through a two-level scene, in the engine's PackedRay layout
        {"name": "world", "kind": "world", "any": False, "instances": 256, "width": 1280, "height": 720},
        # the shadow rays of such a frame
        {"name": "world_shadow", "kind": "world", "any": True, "instances": 256, "width": 1280, "height": 720},
        # baking many assets at once: 64 meshes of 1k to 64k triangles, 4k to 256k rays each
        {"name": "batch", "kind": "batch", "meshes": 64, "tris": 65536, "rays": 262144},
        # the interactive viewer: one progressive frame per call, then shown
        {"name": "frame", "kind": "frame", "instances": 256, "width": 1280, "height": 720, "bounces": 4, "frames": 1,
         "spf": 0},
        # offline accumulation: eight progressive frames per call
        {"name": "frames", "kind": "frame", "instances": 256, "width": 1280, "height": 720, "bounces": 4, "frames": 8,
         "spf": 0},
        # the engine's default renderer: four samples per pixel and the temporal resolve
        {"name": "realtime", "kind": "frame", "instances": 256, "width": 1280, "height": 720, "bounces": 4,
         "frames": 1, "spf": 4},
        # radiance-cache queries of a 1280 x 720 frame's second vertices (about half of its pixels)
        {"name": "infer", "kind": "infer", "queries": 460001, "log2_table": 19},
        # one online training step of the cache on a frame's training samples
        {"name": "train", "kind": "train", "queries": 65536, "log2_table": 19},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "any", "world", "batch", "frame", "infer", "train"])
    if kind in ("closest", "any"):
        if rng.random() < 0.6:
            return {"kind": kind, "scene": "soup", "tris": _log(rng, 1000, 262144), "rays": _log(rng, 32, 1048576)}
        return {"kind": kind, "scene": "height", "grid": _log(rng, 129, 725), "width": _log(rng, 61, 1920),
                "height": _log(rng, 37, 1080)}
    if kind == "world":
        return {"kind": kind, "any": rng.random() < 0.5, "instances": _log(rng, 5, 2048), "width": _log(rng, 61, 1280),
                "height": _log(rng, 37, 720)}
    if kind == "batch":
        return {"kind": kind, "meshes": rng.randint(3, 64), "tris": _log(rng, 2048, 65536), "rays": _log(rng, 8192, 262144)}
    if kind == "frame":
        realtime = rng.random() < 0.4
        return {"kind": kind, "instances": _log(rng, 16, 512), "width": _log(rng, 161, 1280),
                "height": _log(rng, 91, 720), "bounces": rng.randint(1, 4),
                "frames": 1 if realtime else rng.choice([1, 1, 3, 8]), "spf": rng.choice([1, 2, 4]) if realtime else 0}
    if kind == "infer":
        return {"kind": kind, "queries": _log(rng, 1000, 460000), "log2_table": rng.randint(15, 19)}
    return {"kind": kind, "queries": _log(rng, 1000, 65000), "log2_table": rng.randint(15, 19)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt):
    return np.random.Generator(np.random.PCG64([0x6A71A5, int(seed), salt]))


def _cuda(rays):
    return torch.from_numpy(np.ascontiguousarray(rays).view(np.float32).reshape(len(rays), -1).copy()).cuda()


def _soup(case, seed):
    g = _gen(seed, 1)
    return W.triangle_soup(case["tris"], g), W.random_rays(case["rays"], g)


def _terrain(case, seed):
    grid = case["grid"]
    verts = W.heightfield(grid=grid, seed=int(seed) % 65536 + 1)
    span = grid - 1.0
    eye = (0.5 * span, 60.0 + 0.06 * span, -0.15 * span)
    return verts, W.pinhole_rays(case["width"], case["height"], eye, 0.0, 30.0)


def _toward_light(d_rays, t, light):
    """A ray toward `light` from every hit point of d_rays (t < 1e12), pulled back a little; the rays that missed
    take the points of the ones that hit in turn, so every ray of the batch starts on a surface."""
    hit = torch.nonzero(t < 1e11).flatten()
    if not len(hit):
        hit = torch.arange(len(t), device=t.device)
        t = torch.ones_like(t)
    src = torch.where(t < 1e11, torch.arange(len(t), device=t.device), hit[torch.arange(len(t), device=t.device) % len(hit)])
    out = d_rays.clone()
    out[:, 0:3] = d_rays[src, 0:3] + d_rays[src, 4:7] * (t[src] * 0.9999 - 1e-3).clamp_min(0.0)[:, None]
    out[:, 4:7] = torch.tensor(np.asarray(light, np.float32), device=t.device)
    return out.contiguous()


def _scene(case, seed):
    """The two-level scene of the library's path-tracing workload: blob meshes, random instances."""
    g = _gen(seed, 2)
    meshes = [W.blob_mesh(g) for _ in range(8)]
    mats = {"albedo": g.uniform(0.1, 0.9, (8, 3)).astype(np.float32),
            "roughness": g.uniform(0.05, 1.0, 8).astype(np.float32), "metalness": np.zeros(8, np.float32)}
    n = case["instances"]
    xf = W.random_affine(g, n)
    which = g.integers(0, 8, n)
    blases = atlas_rt.build_many([v for v, _ in meshes])
    for k, b in enumerate(blases):
        b.set_shading(meshes[k][1], np.full(len(meshes[k][0]), k, np.int32))
    world = atlas_rt.World()
    world.update(atlas_rt.instance_descs(xf, which), blases)
    return world, blases, mats


def _sizes(k, lo, hi):
    """k uneven sizes spread evenly over the logarithm of [lo, hi], small and large ones mixed."""
    at = (np.arange(k) * 0.6180339887498949 + 0.5) % 1.0
    return np.round(lo * (hi / lo) ** at).astype(np.int64)


def _packed(d_rays):
    """PackedRay records (origin, id), (direction, 0), (0, -1, -1, 0) of (n, 8) rays."""
    n = len(d_rays)
    out = torch.zeros((n, 12), dtype=torch.float32, device="cuda")
    out[:, 0:3] = d_rays[:, 0:3]
    out[:, 4:7] = d_rays[:, 4:7]
    bits = out.view(torch.int32)
    bits[:, 3] = torch.arange(n, dtype=torch.int32, device="cuda")
    bits[:, 9:11] = -1
    return out


def _cache_inputs(case, seed):
    """Queries on the surfaces of 48 spheres inside the bounds, smooth positive targets, and the parameters of a
    network in mid-training: everything from the seed, without the library."""
    g = torch.Generator().manual_seed(int(seed))
    n, T = case["queries"], 1 << case["log2_table"]
    centre = torch.rand((48, 3), generator=g) * 1.6 - 0.8
    radius = torch.rand(48, generator=g) * 0.15 + 0.05
    which = torch.randint(0, 48, (n,), generator=g)
    normal = torch.nn.functional.normalize(torch.randn((n, 3), generator=g), dim=1)
    out = torch.nn.functional.normalize(torch.randn((n, 3), generator=g), dim=1)
    q = torch.zeros((n, 12))
    q[:, 0:3] = centre[which] + radius[which, None] * normal
    q[:, 3] = torch.rand(n, generator=g)
    q[:, 4:7] = out
    q[:, 8:11] = normal
    t = torch.zeros((n, 4))
    t[:, 0:3] = (0.6 + 0.4 * torch.sin(3.0 * q[:, 0:3] + normal)) * (0.5 + torch.rand((n, 3), generator=g))
    mlp = torch.cat([(torch.rand(k * m, generator=g) * 2 - 1) * math.sqrt(6.0 / (k + m)) for k, m in _LAYERS])
    table = ((torch.rand((12, T, 2), generator=g) * 2 - 1) * 0.5).to(torch.float16)
    return q.cuda(), t.cuda(), mlp.cuda(), table.cuda()


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("closest", "any"):
        verts, rays = (_soup if case["scene"] == "soup" else _terrain)(case, seed)
        s["blas"] = atlas_rt.Blas.build(verts)
        s["rays"] = _cuda(rays)
        n = len(s["rays"])
        s["hits"] = torch.empty((n, 4), dtype=torch.float32, device="cuda")
        if kind == "any":
            if case["scene"] == "height":
                s["blas"].trace_closest(s["rays"], s["hits"])
                s["rays"] = _toward_light(s["rays"], s["hits"][:, 0], EVENING_SUN)
            s["hits"] = torch.empty(n, dtype=torch.int32, device="cuda")
    elif kind == "world":
        s["world"], s["blases"], _ = _scene(case, seed)
        cc = W.c2_camera()
        rays = _cuda(W.pinhole_rays(case["width"], case["height"], cc["eye"], cc["yaw_deg"], cc["pitch_deg"],
                                    cc["fov_y_deg"]))
        n = len(rays)
        s["any"] = case["any"]
        if case["any"]:
            hits = torch.empty((n, 4), dtype=torch.float32, device="cuda")
            s["world"].trace_closest_rays(rays, hits)
            rays = _toward_light(rays, hits[:, 0], -W.C2_SUN_DIR)
            s["out"] = torch.empty(n, dtype=torch.int32, device="cuda")
        else:
            s["out"] = torch.empty((n, 12), dtype=torch.float32, device="cuda")
        s["in"] = _packed(rays)
        s["count"] = torch.tensor([n], dtype=torch.int32, device="cuda")
        s["n"] = n
    elif kind == "batch":
        g = _gen(seed, 3)
        k = case["meshes"]
        tris = g.permutation(_sizes(k, 1024, case["tris"]))
        counts = _sizes(k, 4096, case["rays"])
        s["blases"] = atlas_rt.build_many([W.triangle_soup(int(t), g) for t in tris])
        s["rays"] = _cuda(W.random_rays(int(counts.sum()), g))
        table = np.zeros(k, dtype=_abi.BATCH_DTYPE)
        table["blas"] = np.arange(k)
        table["ray_offset"] = np.concatenate([[0], np.cumsum(counts)[:-1]])
        table["ray_count"] = counts
        s["set"] = atlas_rt.BatchSet(s["blases"], table)
        s["hits"] = torch.empty((len(s["rays"]), 4), dtype=torch.float32, device="cuda")
    elif kind == "frame":
        s["world"], s["blases"], mats = _scene(case, seed)
        cc = W.c2_camera()
        aspect = case["width"] / case["height"]
        s["cam"] = atlas_rt.camera(cc["eye"], cc["yaw_deg"], cc["pitch_deg"], cc["fov_y_deg"], aspect)
        s["pt"] = atlas_rt.PathTracer(s["world"], case["width"], case["height"], case["bounces"], W.c2_materials(mats),
                                      W.sun_light(), env=W.C2_ENV)
        s["frames"], s["spf"] = case["frames"], case["spf"]
        if case["spf"]:
            s["pt"].set_realtime(samples_per_frame=case["spf"])
            view = atlas_rt.view_matrix(cc["eye"], cc["yaw_deg"], cc["pitch_deg"])
            proj = atlas_rt.projection_matrix(cc["fov_y_deg"], aspect)
            s["fm"] = atlas_rt.frame_matrices(view, proj, proj @ view)
        else:
            s["image"] = torch.empty((case["height"], case["width"], 4), dtype=torch.float32, device="cuda")
    else:
        s["q"], s["t"], mlp, table = _cache_inputs(case, seed)
        s["cache"] = atlas_rt.RadianceCache((-1.0, -1.0, -1.0), (1.0, 1.0, 1.0), log2_table=case["log2_table"],
                                            learning_rate=TRAIN_RATE)
        s["cache"].set_params(mlp, table.view(torch.int16).reshape(-1))
        s["out"] = torch.empty((case["queries"], 4), dtype=torch.float32, device="cuda")
        s["loss"] = torch.empty(1, dtype=torch.float32, device="cuda")
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "closest":
        s["blas"].trace_closest(s["rays"], s["hits"])
        return {"tuv": s["hits"][:, 0:3], "prim": s["hits"].view(torch.int32)[:, 3]}
    if kind == "any":
        s["blas"].trace_any(s["rays"], s["hits"])
        return {"occluded": s["hits"]}
    if kind == "world":
        if s["any"]:
            s["world"].trace_any_packed(s["in"], s["out"], s["count"], s["n"])
            return {"occluded": s["out"]}
        s["world"].trace_closest_packed(s["in"], s["out"], s["count"], s["n"])
        return {"records": s["out"].view(torch.int32)}
    if kind == "batch":
        s["set"].trace_closest(s["rays"], s["hits"], kernel=BATCH_KERNEL, block=128, refill=32)
        return {"tuv": s["hits"][:, 0:3], "prim": s["hits"].view(torch.int32)[:, 3]}
    if kind == "frame":
        if s["spf"]:
            s["pt"].render_realtime(s["cam"], s["fm"])
            return {"resolved": s["pt"].read_realtime(_abi.RT_RESOLVED)}
        s["pt"].render(s["cam"], s["frames"])
        return {"image": s["pt"].read(s["image"])}
    if kind == "infer":
        s["cache"].infer(s["q"], s["out"])
        return {"radiance": s["out"][:, 0:3]}
    s["cache"].train(s["q"], s["t"], s["loss"])
    mlp, table = s["cache"].get_params()
    return {"loss": s["loss"], "mlp": mlp, "table": table.view(torch.float16)}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
_LAYERS = [(32, 64), (64, 64), (64, 64), (64, 64), (64, 64), (64, 3)]
_MESH = 64 + 48      # bytes of a triangle and its share of the inner nodes
_BLOB = 3968         # triangles of a blob mesh


def _walk(tris):
    """Operations of one ray's way down a balanced tree: two boxes of 22 operations per level, one triangle."""
    return 44.0 * max(1.0, math.log2(max(2, tris))) + 60.0


def work(case):
    kind = case["kind"]
    if kind in ("closest", "any"):
        soup = case["scene"] == "soup"
        tris = case["tris"] if soup else 2 * (case["grid"] - 1) ** 2
        n = case["rays"] if soup else case["width"] * case["height"]
        return {"bytes": n * (32 + (16 if kind == "closest" else 4)) + min(tris, n * 64) * _MESH,
                "flops": n * _walk(tris)}
    if kind == "world":
        n = case["width"] * case["height"]
        return {"bytes": n * (48 + (4 if case["any"] else 48)) + 8 * _BLOB * _MESH + case["instances"] * 128,
                "flops": n * _walk(case["instances"])}
    if kind == "batch":
        rays, tris = int(_sizes(case["meshes"], 4096, case["rays"]).sum()), _sizes(case["meshes"], 1024, case["tris"])
        return {"bytes": rays * 48 + int(tris.sum()) * _MESH, "flops": rays * _walk(float(tris.mean()))}
    if kind == "frame":
        pixels = case["width"] * case["height"]
        return {"bytes": pixels * 32 + 8 * _BLOB * (_MESH + 96) + case["instances"] * 128,
                "flops": pixels * max(1, case["spf"]) * case["frames"] * _walk(case["instances"])}
    macs = sum(k * m for k, m in _LAYERS)
    n, touched = case["queries"], 12 * (1 << case["log2_table"]) * 4
    if kind == "infer":
        return {"bytes": n * 64 + min(touched, n * 96 * 4), "flops": n * 2.0 * (macs + 96 * 4)}
    # forward, backward and weight gradients; the table, its gradient and both moments read and written once
    return {"bytes": n * 64 + 4 * touched * 2, "flops": n * 6.0 * (macs + 96 * 4)}


def tolerance(case):
    if case["kind"] == "infer":
        return {"rel": 0.025, "max": 0.2}  # bfloat16 operands: 6.4e-3 from the 64-bit network
    if case["kind"] == "train":
        # 7.4e-3 from the 64-bit step; a gradient near zero may change the sign of Adam's first update
        return {"rel": 0.03, "max": 0.25}
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _exact_closest(case, seed):
    verts, rays = _soup(case, seed)
    tri = torch.from_numpy(verts).cuda().double().reshape(-1, 3, 3)
    r = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda().double()
    v0, e0, e1 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    n = len(r)
    tuv = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    prim = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    step = max(1, 8_000_000 // len(tri))
    for a in range(0, n, step):
        o, d, tmin, tmax = r[a:a + step, None, 0:3], r[a:a + step, None, 4:7], r[a:a + step, 3], r[a:a + step, 7]
        q = torch.linalg.cross(d.expand(-1, len(tri), 3), e1.expand(len(o), -1, 3))
        s = o - v0
        p = torch.linalg.cross(s, e0.expand(len(o), -1, 3))
        den = (q * e0).sum(-1)
        t, u, v = (p * e1).sum(-1) / den, (q * s).sum(-1) / den, (p * d).sum(-1) / den
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > tmin[:, None]) & (t < tmax[:, None])
        best, k = torch.where(ok, t, torch.inf).min(dim=1)
        hit = torch.isfinite(best)
        at = torch.arange(len(o), device="cuda")
        found = torch.stack([t[at, k], u[at, k], v[at, k]], dim=1)
        miss = torch.stack([tmax, torch.zeros_like(tmax), torch.zeros_like(tmax)], dim=1)
        tuv[a:a + step] = torch.where(hit[:, None], found, miss)
        prim[a:a + step] = torch.where(hit, k, -1).int()
    return {"tuv": tuv, "prim": prim}


def _features(q, table, log2_table):
    """The network's 32 inputs: 12 levels of trilinear table features, directions, roughness, one.  Cell indices in
    32-bit arithmetic, weights and sums in 64 bits."""
    T = 1 << log2_table
    unit = ((q[:, 0:3] + 1.0) * 0.5).clamp(0.0, 1.0)
    growth = math.exp((math.log(2048.0) - math.log(16.0)) / 11)
    cols = []
    for lev in range(12):
        res = math.floor(16.0 * growth ** lev + 1e-9)
        pos = unit * res
        cell = torch.minimum(torch.floor(pos), torch.tensor(res - 1.0, device=q.device))
        f = (pos - cell).double()
        c = cell.long()
        feat = 0.0
        for k in range(8):
            px, py, pz = c[:, 0] + (k & 1), c[:, 1] + ((k >> 1) & 1), c[:, 2] + (k >> 2)
            if (res + 1.0) ** 3 <= T:
                h = px + (res + 1) * (py + (res + 1) * pz)
            else:
                h = ((px ^ (py * 2654435761) ^ (pz * 805459861)) & 0xFFFFFFFF) & (T - 1)
            w = (f[:, 0] if k & 1 else 1 - f[:, 0]) * (f[:, 1] if k & 2 else 1 - f[:, 1]) * (f[:, 2] if k & 4 else 1 - f[:, 2])
            feat = feat + w[:, None] * table[lev][h]
        cols.append(feat)
    q64 = q.double()
    return torch.cat(cols + [q64[:, 4:7], q64[:, 8:11], q64[:, 3:4], torch.ones_like(q64[:, 3:4])], dim=1)


def _network(mlp, x):
    at = 0
    for i, (k, m) in enumerate(_LAYERS):
        x = x @ mlp[at:at + k * m].reshape(k, m)
        at += k * m
        if i < 5:
            x = x.relu()
    return x


def exact(case, seed):
    if case["kind"] == "closest" and case["scene"] == "soup" and case["tris"] * case["rays"] <= 4e8:
        return _exact_closest(case, seed)
    if case["kind"] not in ("infer", "train"):
        return None
    q, t, mlp, table = _cache_inputs(case, seed)
    mlp, table = mlp.double(), table.double()
    if case["kind"] == "infer":
        step = 1 << 17
        return {"radiance": torch.cat([_network(mlp, _features(q[a:a + step], table, case["log2_table"]))
                                       for a in range(0, len(q), step)])}
    # one step of Adam from zero moments on the relative squared error (its denominator held constant)
    mlp.requires_grad_(True)
    table.requires_grad_(True)
    y = _network(mlp, _features(q, table, case["log2_table"]))
    loss = ((y - t[:, 0:3].double()) ** 2 / (y.detach() ** 2 + 0.01)).mean()
    loss.backward()
    out = []
    for p in (mlp, table):
        m, v = 0.1 * p.grad, 0.01 * p.grad ** 2
        rate = TRAIN_RATE * math.sqrt(1 - 0.99) / (1 - 0.9)
        out.append((p - rate * m / (v.sqrt() + 1e-15)).detach().reshape(-1))
    return {"loss": loss.detach().reshape(1), "mlp": out[0], "table": out[1]}
