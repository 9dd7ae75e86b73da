"""The work that programs on this engine have it do, as cases to time.

A world is a value-noise terrain voxelised by a column fill. Programs pick voxels with rays, edit the
world (one brush dab, a list of dabs applied one by one, a batch, a tick of client requests),
collect garbage, and render frames of what is there. Every pass goes through the C ABI's Python
binding as a host program does; edits go on from the world that the pass before left, so a
case's passes form an editing session over its own pool.

What a pass returns: the roots that it left (a root pointer names the bucket that the hash of its
node picks, and so on down to the leaves: other voxels give other roots), pixels, hits, counters."""
import ctypes
import math

import numpy as np
import torch

from vkhashdag_amd import autotune, capi
from vkhashdag_amd import workloads as W

VIEW_MIN, VIEW_MAX = (640, 360), (1920, 1080)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the voxel under the cursor: one ray, host to host
        {"name": "pick_1", "kind": "pick", "res": 1024, "rays": 1},
        # a ray query over device arrays (visibility, collision, range sensing)
        {"name": "rays_1m", "kind": "rays", "res": 4096, "rays": 1000003},
        # a thumbnail or minimap of a small world, no shadows
        {"name": "frame_thumb", "kind": "frame", "res": 1024, "views": 1, "width": 255, "height": 201,
         "shadow": False, "beam": False, "lod": True},
        # the benchmark's frame: 1080p, a primary ray per pixel and a shadow ray per hit
        {"name": "frame_1080p", "kind": "frame", "res": 4096, "views": 1, "width": 1920, "height": 1080,
         "shadow": True, "beam": False, "lod": True},
        # several clients' cameras in one launch, uneven sizes, with the beam prepass
        {"name": "views_8_beam", "kind": "frame", "res": 4096, "views": 8, "width": 0, "height": 0,
         "shadow": True, "beam": True, "lod": True},
        # one dab of an interactive brush
        {"name": "dab_1", "kind": "edit", "res": 4096, "edits": 1, "batched": False, "colored": True, "rmin": 4,
         "rmax": 64, "frame": False},
        # the benchmark's step: 256 sphere adds and removes one by one, then a frame
        {"name": "step_256", "kind": "edit", "res": 4096, "edits": 256, "batched": False, "colored": True, "rmin": 4,
         "rmax": 128, "frame": True},
        # a batch of mixed edits of very uneven size, then a frame
        {"name": "batch_4096", "kind": "edit", "res": 4096, "edits": 4096, "batched": True, "colored": True, "rmin": 2,
         "rmax": 256, "frame": True},
        # a tick of a server: 64 client requests, 70% edits and 30% renders
        {"name": "serve_64", "kind": "serve", "res": 4096, "requests": 64, "rmin": 2, "rmax": 64},
        # garbage collection of an edited world, the version before the edits kept for undo; a small frame
        {"name": "gc_4096", "kind": "gc", "res": 4096, "edits": 256, "rmin": 4, "rmax": 128},
        # a frame graph: edits, garbage collection, views
        {"name": "graph_24", "kind": "graph", "res": 2048, "edits": 24, "views": 4, "rmax": 64},
        # a new heightfield generated and voxelised (uncolored, as the largest worlds are), probed by rays
        {"name": "terrain_2048", "kind": "terrain", "res": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick", "rays", "frame", "frame", "edit", "edit", "batch", "serve", "gc", "graph", "terrain"])
    res = rng.choice([512, 1024, 2048, 4096])
    rmax = _log_int(rng, 8, max(16, res // 32))
    if kind == "pick":
        return {"kind": kind, "res": res, "rays": _log_int(rng, 1, 64)}
    if kind == "rays":
        return {"kind": kind, "res": res, "rays": _log_int(rng, 64, 1 << 20)}
    if kind == "frame":
        views = rng.choice([1, 1, 2, 5])
        beam = rng.random() < 0.3
        return {"kind": kind, "res": res, "views": views, "width": _log_int(rng, 64, 1920),
                "height": _log_int(rng, 48, 1080), "shadow": rng.random() < 0.7, "beam": beam,
                "lod": beam or rng.random() < 0.7}
    if kind == "edit":
        return {"kind": kind, "res": res, "edits": _log_int(rng, 1, 256), "batched": False,
                "colored": rng.random() < 0.7, "rmin": 2, "rmax": rmax, "frame": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": "edit", "res": res, "edits": _log_int(rng, 2, 2048), "batched": True,
                "colored": rng.random() < 0.7, "rmin": 2, "rmax": rmax, "frame": rng.random() < 0.5}
    if kind == "serve":
        return {"kind": kind, "res": res, "requests": _log_int(rng, 4, 64), "rmin": 2, "rmax": min(rmax, 64)}
    if kind == "gc":
        return {"kind": kind, "res": res, "edits": _log_int(rng, 4, 256), "rmin": 2, "rmax": rmax}
    if kind == "graph":
        return {"kind": kind, "res": rng.choice([512, 1024, 2048]), "edits": _log_int(rng, 1, 24),
                "views": rng.choice([1, 2, 3, 4]), "rmax": min(rmax, 64)}
    return {"kind": "terrain", "res": rng.choice([256, 512, 1024, 2048]), "octaves": rng.randint(3, 8)}


# ---------------------------------------------------------------- worlds
def _config(res, keep_history=False):
    """The benchmark's pool geometry: 512-word pages, 4 pages a bucket, 16^3-voxel color leaves."""
    return W.config_for_resolution(res, bucket_bits=16 if res >= 1024 else 14, wbpp=9, pbpb=2, color_leaf_depth=4,
                                   keep_history=keep_history, color_node_capacity=1 << 24,
                                   color_leaf_capacity=1 << 28 if res <= 2048 else 1 << 29)


def _heights(res, seed):
    """A fractal heightfield of res x res columns in [res / 8, 3 res / 4]: six octaves of smoothed noise."""
    rng = np.random.default_rng([seed, 1])
    acc = torch.zeros((1, 1, res, res), dtype=torch.float32, device="cuda")
    for o in range(6):
        n = min(res, 4 << o)
        lattice = torch.from_numpy(rng.random((1, 1, n, n), dtype=np.float32)).cuda()
        acc += 0.5 ** o * torch.nn.functional.interpolate(lattice, size=(res, res), mode="bilinear")
    lo, hi = acc.min(), acc.max()
    acc = res / 8 + (acc - lo) / (hi - lo) * (res * 5 / 8)
    return acc.round().to(torch.int32)[0, 0]


def _world(res, seed, keep_history=False, colored=True):
    autotune.load()
    heights = _heights(res, seed).cpu().numpy().astype(np.uint32)
    pool = capi.DevicePool(_config(res, keep_history), heights=heights)
    pool.edit(W.terrain_edit(res, seed=seed % 65536, skin=8, colored=colored))
    return pool, heights


# ---------------------------------------------------------------- edits, views, requests
def _edits(case, heights, seed, count, mixed=False, invert=False):
    """count sphere adds and removes on the terrain's surface, radii log-uniform; mixed (colored worlds):
    40% adds, 40% removes and 20% box paints."""
    res, colored = case["res"], case.get("colored", True)
    rng = np.random.default_rng([seed, 2])
    e = np.zeros(count, W.EDIT_DTYPE)
    xy = rng.integers(0, res, (count, 2))
    z = heights[xy[:, 1], xy[:, 0]].astype(np.int64)
    r = np.exp(rng.uniform(math.log(case.get("rmin", 2)), math.log(case["rmax"]), count))
    u = rng.random(count)
    colors = rng.integers(0, 1 << 24, count)
    cuts = (0.4, 0.8) if mixed and colored else (0.5, 1.0)
    kind = np.where(u < cuts[0], W.SPHERE_FILL, np.where(u < cuts[1], W.SPHERE_DIG, W.AABB_PAINT))
    paint = kind == W.AABB_PAINT
    h = np.maximum(1, np.round(r)).astype(np.int64)[:, None]
    centre = np.concatenate([xy, z[:, None]], axis=1)
    e["kind"] = kind
    e["p0"] = np.where(paint[:, None], np.maximum(0, centre - h), centre)
    e["p1"] = np.where(paint[:, None], np.minimum(res, centre + h), 0)
    e["r2"] = np.where(paint, 0, (r * r).astype(np.int64))
    has = (kind != W.SPHERE_DIG) & colored
    e["colored"] = has
    e["has_value"] = has
    e["colors"] = np.where(has, colors, 0)
    return e


def _session(case, heights, seed, n, mixed):
    """An editing session's lists of n edits: fresh ones, then the same places with adds and removes
    exchanged, so that a session that goes round never stops changing the world."""
    # at most 16384 edits are drawn, and a thousand lists: what a session appends stays far below the
    # pool's capacity
    lists = max(2, min(1024, 16384 // n))
    e = _edits(case, heights, seed, lists * n, mixed)
    back = e.copy()
    add, dig = e["kind"] == W.SPHERE_FILL, e["kind"] == W.SPHERE_DIG
    back["kind"][add], back["kind"][dig] = W.SPHERE_DIG, W.SPHERE_FILL
    back["colored"][add] = back["has_value"][add] = 0
    back["colored"][dig] = back["has_value"][dig] = int(case.get("colored", True))
    back["colors"] = np.where(dig & (back["has_value"] == 1), 0x7FA0C3, np.where(add, 0, e["colors"]))
    return [x[k * n:(k + 1) * n].copy() for x in (e, back) for k in range(lists)]


def _views(case, seed, heights):
    """Orbit cameras around the terrain; sizes 0: each client's own window, between 640x360 and 1920x1080."""
    rng, windows = np.random.default_rng([seed, 3]), np.random.default_rng(8)
    res, views = case["res"], []
    zc = float(heights[res // 2, res // 2])
    for _ in range(case["views"]):
        w = case.get("width") or int(windows.integers(VIEW_MIN[0], VIEW_MAX[0] + 1))
        h = case.get("height") or int(windows.integers(VIEW_MIN[1], VIEW_MAX[1] + 1))
        vb = W.orbit_view((res / 2, res / 2, zc), 0.9 * res, int(rng.integers(1 << 30)), w, h, res=res,
                          lod=case.get("lod", True), elevation=(0.35, 0.6))
        flags = (capi.TRACE_SHADOW if case.get("shadow", True) else 0) | (capi.TRACE_BEAM if case.get("beam") else 0)
        views.append((vb, w, h, flags))
    return views


def _view_array(views):
    arr, off = (capi.hd_view * len(views))(), 0
    for i, (vb, w, h, flags) in enumerate(views):
        arr[i] = capi.make_view(vb, w, h, flags, off)
        off += w * h
    return arr, off


def _requests(case, heights, seed, n_lists):
    """Ticks of client requests that have all arrived: 70% edits, 30% renders of 256x256 to 1080p."""
    n, res = case["requests"], case["res"]
    rng = np.random.default_rng([seed, 4])
    lists = _session(case, heights, seed, n, mixed=True)[:n_lists]
    zc = float(heights[res // 2, res // 2])
    out = []
    for edits in lists:
        q = np.zeros(n, W.REQUEST_DTYPE)
        q["client"] = rng.integers(0, 64, n)
        q["edit"] = edits
        for i in np.nonzero(rng.random(n) >= 0.7)[0]:
            w, h = int(rng.integers(256, 1921)), int(rng.integers(256, 1081))
            vb = W.orbit_view((res / 2, res / 2, zc), 0.8 * res, int(rng.integers(1 << 30)), w, h, res=res)
            q[i]["kind"] = W.REQ_RENDER
            q[i]["edit"] = np.zeros((), W.EDIT_DTYPE)
            q[i]["view"] = W.view_record(vb, w, h, capi.TRACE_SHADOW)
        out.append(q)
    return out


def _rays(n, seed, steep):
    """Rays from above the terrain down into it: origins in the air over the world, directions long
    enough to cross it. steep: a cursor's or a probe's, which all hit; else a sensor's, to the horizon."""
    rng = np.random.default_rng([seed, 5])
    o = rng.random((n, 3), dtype=np.float32)
    o[:, :2] = 0.4 + 0.2 * o[:, :2] if steep else o[:, :2]
    o[:, 2] = 0.78 + 0.2 * o[:, 2]
    a = rng.random(n, dtype=np.float32) * np.float32(2 * math.pi)
    down = (2.5 if steep else 0.1) + 1.4 * rng.random(n, dtype=np.float32)
    d = np.stack([np.cos(a), np.sin(a), -down], axis=1).astype(np.float32)
    return o, d * np.float32(2.0)


def _on_gpu(rays):
    return tuple(torch.from_numpy(x).cuda() for x in rays)


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind, res = case["kind"], case["res"]
    s = {"case": case, "at": 0}
    if kind in ("pick", "rays"):
        s["pool"], _ = _world(res, seed, colored=False)
        s["o"], s["d"] = _rays(case["rays"], seed, kind == "pick")
        if kind == "rays":
            s["o"], s["d"] = _on_gpu((s["o"], s["d"]))
            s["hits"] = torch.zeros((case["rays"], 4), dtype=torch.float32, device="cuda")
    elif kind == "terrain":
        autotune.load()
        s["pool"] = capi.DevicePool(_config(res))
        s["seed"] = seed * 16
        # where things of the new world are put: probes down to the ground
        s["o"], s["d"] = _on_gpu(_rays(16384, seed, True))
        s["hits"] = torch.zeros((16384, 4), dtype=torch.float32, device="cuda")
    else:
        s["pool"], heights = _world(res, seed, keep_history=kind == "serve", colored=case.get("colored", True))
        if kind == "frame":
            s["pool"].edit(_edits({"res": res, "rmin": 4, "rmax": res // 32}, heights, seed, 64, mixed=True),
                           capi.MODE_BATCHED)
            s["views"], pixels = _view_array(_views(case, seed, heights))
            s["rgba"] = torch.zeros(pixels, dtype=torch.int32, device="cuda")
        elif kind == "edit":
            s["lists"] = _session(case, heights, seed, case["edits"], case["batched"])
            s["mode"] = capi.MODE_BATCHED if case["batched"] else capi.MODE_PLAIN
            s["pool"].reserve(max(s["lists"][:8], key=lambda e: int(e["r2"].sum())), s["mode"])
            if case["frame"]:
                s["views"], pixels = _view_array(_views({"res": res, "views": 1, "width": 1920, "height": 1080}, seed,
                                                        heights))
                s["rgba"] = torch.zeros(pixels, dtype=torch.int32, device="cuda")
        elif kind == "serve":
            s["requests"] = _requests(case, heights, seed, 32)
            s["rgba"] = torch.zeros(case["requests"] * 1920 * 1080, dtype=torch.int32, device="cuda")
        elif kind == "gc":
            s["before"] = s["pool"].root
            s["pool"].edit(_edits(case, heights, seed, case["edits"]))
            s["views"], pixels = _view_array(_views({"res": res, "views": 1, "width": 640, "height": 360}, seed,
                                                    heights))
            s["rgba"] = torch.zeros(pixels, dtype=torch.int32, device="cuda")
        elif kind == "graph":
            s["lists"] = _session(case, heights, seed, case["edits"], mixed=True)
            s["views"] = _views({**case, "width": 1280, "height": 720}, seed, heights)
            s["frame"] = capi.Frame(s["pool"], max_edits=32, max_passes=4, max_radius=64, n_views=case["views"],
                                    max_width=1280, max_height=720, colors=True, gc=True)
            s["rgba"] = torch.zeros(case["views"] * 1280 * 720, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


def _next(s, lists):
    x = lists[s["at"] % len(lists)]
    s["at"] += 1
    return x


def _render(s):
    pool = s["pool"]
    capi.check(capi.lib().hd_trace(pool.h, pool.root, pool.color_root, s["views"], len(s["views"]),
                                   s["rgba"].data_ptr(), None))
    return s["rgba"]


def _cast(s):
    pool = s["pool"]
    capi.check(capi.lib().hd_traversal(pool.h, pool.root, s["o"].data_ptr(), s["d"].data_ptr(), len(s["o"]),
                                       s["hits"].data_ptr()))
    return s["hits"]


def run(s):
    kind, pool = s["case"]["kind"], s["pool"]
    if kind == "pick":
        return pool.traversal(s["o"], s["d"])
    if kind == "rays":
        return _cast(s)
    if kind == "frame":
        return _render(s)
    if kind == "edit":
        pool.edit(_next(s, s["lists"]), s["mode"])
        roots = [pool.root, pool.color_root]
        return {"roots": roots, "rgba": _render(s)} if s["case"]["frame"] else {"roots": roots}
    if kind == "serve":
        requests = _next(s, s["requests"])
        results = np.zeros(len(requests), W.RESULT_DTYPE)
        cfg = capi.hd_serve_config(32, 0, 1 << 24, 0)
        root, color_root, stats = ctypes.c_uint32(0), ctypes.c_uint32(0), capi.hd_serve_stats()
        capi.check(capi.lib().hd_serve_run(pool.h, ctypes.byref(cfg), pool.root, pool.color_root,
                                           requests.ctypes.data, len(requests), s["rgba"].data_ptr(),
                                           s["rgba"].numel(), results.ctypes.data, ctypes.byref(root),
                                           ctypes.byref(color_root), ctypes.byref(stats)))
        pool.root, pool.color_root = root.value, color_root.value
        return {"rgba": s["rgba"], "root": results["root"].astype(np.int64), "tick": results["tick"].astype(np.int64)}
    if kind == "gc":
        roots = pool.gc([s["before"]])
        s["before"] = int(roots[1])
        return {"roots": roots.astype(np.int64), "rgba": _render(s)}
    if kind == "graph":
        f = s["frame"]
        f.set(_next(s, s["lists"]), s["views"])
        f.launch()
        roots = f.wait()
        capi.check(capi.lib().hd_device_copy(s["rgba"].data_ptr(), capi.lib().hd_frame_rgba(f.h), s["rgba"].numel() * 4,
                                             pool.h))
        return {"roots": list(roots), "rgba": s["rgba"]}
    # terrain: another heightfield each time, four in turn
    seed = s["seed"] + s["at"] % 4
    s["at"] += 1
    res = s["case"]["res"]
    pool.root = W.HD_NULL
    pool.value_noise_heightmap(s["case"].get("octaves", 6), seed, res // 8, res * 3 // 4, download=False)
    pool.edit(W.terrain_edit(res, seed=seed % 65536, colored=False))
    return {"root": pool.root, "ground": _cast(s)}


# ---------------------------------------------------------------- what a pass cannot do without
def _ray_bytes(res):
    """A ray's descent to a voxel: a mask word and a child pointer per level, the leaf's two words."""
    return 8 * (int(math.log2(res)) - 1)


def _edit_bytes(case, n):
    """n edits: the leaf nodes that their surfaces cross (8 bytes read, 8 written), the inner nodes above
    (an eighth as many per level, 36 bytes), a root path each, and (colored) a byte per surface voxel."""
    lo, hi = case.get("rmin", 2), case["rmax"]
    r2 = (hi * hi - lo * lo) / (2 * math.log(hi / lo)) if hi > lo else hi * hi
    surface = 4 * math.pi * r2
    leaves = surface / 16 + 8
    path = 2 * 36 * int(math.log2(case["res"]))
    return n * (leaves * (16 + 72 / 7) + path + (surface if case.get("colored", True) else 0))


def work(case):
    kind, res = case["kind"], case["res"]
    if kind in ("pick", "rays"):
        return {"bytes": case["rays"] * (24 + 16 + _ray_bytes(res)), "flops": 0}
    pixel = 4 + _ray_bytes(res) * (2 if case.get("shadow", True) else 1)
    if kind == "frame":
        mean = (VIEW_MIN[0] + VIEW_MAX[0]) / 2 * (VIEW_MIN[1] + VIEW_MAX[1]) / 2
        return {"bytes": case["views"] * (case["width"] * case["height"] or mean) * pixel, "flops": 0}
    if kind == "edit":
        return {"bytes": _edit_bytes(case, case["edits"]) + (1920 * 1080 * pixel if case["frame"] else 0), "flops": 0}
    if kind == "serve":
        return {"bytes": _edit_bytes(case, 0.7 * case["requests"]) + 0.3 * case["requests"] * 1088 * 668 * pixel,
                "flops": 0}
    # a terrain's surface: its leaves (a 4^3 block crossed by about 1.5 per column block), the nodes above
    surface = (res / 4) ** 2 * 1.5 * (8 + 36 / 3)
    if kind == "gc":
        return {"bytes": 2 * surface + 2 * _edit_bytes({**case, "colored": False}, case["edits"]) + 640 * 360 * pixel,
                "flops": 0}
    if kind == "graph":
        return {"bytes": 2 * surface + _edit_bytes(case, case["edits"]) + case["views"] * 1280 * 720 * pixel,
                "flops": 0}
    return {"bytes": 4 * res * res + surface + 16384 * (40 + _ray_bytes(res)), "flops": 0}


# ---------------------------------------------------------------- hits in 64 bits
def exact(case, seed):
    """Ray hits on the heightfield by a column walk in 64 bits: column by column, where the ray first is
    below the column's height; the hit is where it enters that voxel. Other outputs are whole numbers."""
    if case["kind"] not in ("pick", "rays"):
        return None
    res = case["res"]
    heights = _heights(res, seed).to(torch.float64)
    o, d = (x.to(torch.float64) for x in _on_gpu(_rays(case["rays"], seed, case["kind"] == "pick")))
    o = o * res
    d = d * res
    n = len(o)
    hit_t = torch.full((n,), -1.0, dtype=torch.float64, device="cuda")
    alive = torch.arange(n, device="cuda")
    cell = torch.floor(o[:, :2]).clamp(0, res - 1).to(torch.int64)
    t = torch.zeros(n, dtype=torch.float64, device="cuda")
    step = torch.where(d[:, :2] > 0, 1, -1).to(torch.int64)
    while len(alive):
        edge = (cell + (step > 0)).to(torch.float64)
        tx = (edge - o[:, :2]) / d[:, :2]
        t1 = tx.min(dim=1).values
        h = heights[cell[:, 1], cell[:, 0]]
        side = o[:, 2] + t * d[:, 2] < h  # already below the column's top where the ray enters it
        top = (h - o[:, 2]) / d[:, 2]
        hit = (side | (top <= t1)) & (torch.where(side, t, top) <= 1.0)
        hit_t[alive[hit]] = torch.where(side, t, top)[hit]
        first = (tx[:, 0] <= tx[:, 1]).to(torch.int64)
        move = torch.stack([first, 1 - first], dim=1) * step
        cell = cell + move
        t = t1
        keep = ~hit & (t < 1.0) & (cell >= 0).all(dim=1) & (cell < res).all(dim=1)
        alive, cell, t, step, o, d = alive[keep], cell[keep], t[keep], step[keep], o[keep], d[keep]
    o, d = (x.to(torch.float64) for x in _on_gpu(_rays(case["rays"], seed, case["kind"] == "pick")))
    found = hit_t >= 0
    out = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
    out[:, :3] = torch.where(found[:, None], o + hit_t[:, None] * d, 0.0)
    out[:, 3] = found
    return out if case["kind"] == "rays" else out.cpu().numpy()
