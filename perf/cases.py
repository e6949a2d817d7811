"""The work a user of this library has it do, as measured cases.

Every case is one pass through the public bindings (``grt``), with scenes,
cameras, ray buffers and outputs resident as an application keeps them.  Five
kinds of work:

  frame   an animated or static frame: rebuild the grid, primary rays, shadow
          rays, mirror bounces with their shadow rays, Phong shading;
  trace   one traversal stage over rays the caller has in hand (primary,
          shadow or mirror-bounce rays) through a built grid;
  ao      a large scene's frame: rebuild, primary rays, ambient-occlusion rays;
  batch   many scenes of mixed sizes, one launch per bounce level;
  serve   a set of render requests through the continuous-batching server.

Scenes, cameras and parameters are those of the library's own workloads
(``grt.workloads`` and the benchmark): sphere scenes, the stadium of clustered
triangles over a ground plane, clustered spheres for ambient occlusion.

Results are specified bit for bit (the CPU restatement of the algorithm and
every schedule give the same binary32 values), so outputs are compared exactly.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "grid-rt_amd"))

import grt  # noqa: E402
from grt import workloads as W  # noqa: E402

DEV = "cuda:0"
OFFSET = 1e-4
STADIUM_EYE, STADIUM_CENTER = (0.5, 0.6, -1.5), (0.5, 0.3, 0.5)
MAX_BATCH_TRIS, MAX_SERVE_TRIS = 500_000, 1_000_000


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _frame(name, scene, tris, width, height, lam, sub, bounces, mode, graph=False, **more):
    c = {"kind": "frame", "scene": scene, "tris": tris, "width": width, "height": height,
         "lam": lam, "sub": sub, "bounces": bounces, "mode": mode, "graph": graph}
    c.update(more)
    if name:
        c["name"] = name
    return c


def _trace(name, scene, tris, width, height, lam, sub, rays, mode):
    c = {"kind": "trace", "scene": scene, "tris": tris, "width": width, "height": height,
         "lam": lam, "sub": sub, "rays": rays, "mode": mode}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # A thumbnail of a small model, replayed from a launch graph: the
        # smallest call, bound by its chain of launches.
        _frame("thumbnail graph", "spheres", 2048, 64, 64, 5.0, 0, 0, "simple", True),
        # The 16k-triangle sphere frame of the first configuration (512 x 512,
        # rebuilt every frame), launched from Python, with one mirror bounce.
        _frame("spheres 16k frame", "spheres", 16384, 512, 512, 5.0, 0, 1, "simple"),
        # An odd-sized view of a resident mid-sized model, a few lanes per ray:
        # the ordinary small request.
        _trace("odd view 25k", "spheres", 25600, 333, 217, 8.0, 0, "primary", "split4"),
        # The benchmark's frame: 2^20 moving triangles at 1920 x 1080, both
        # grid levels rebuilt, one bounce, shading.
        _frame("stadium frame", "stadium", 1 << 20, 1920, 1080, 16.0, 4, 1, "simple"),
        # The same animation at preview size, where the rebuild dominates.
        _frame("stadium preview", "stadium", 1 << 20, 480, 270, 16.0, 8, 0, "simple"),
        # Its traversal stages alone: coherent closest hit, any hit, and
        # incoherent closest hit through the two-level grid.
        _trace("stadium primary", "stadium", 1 << 20, 1920, 1080, 16.0, 8, "primary", "simple"),
        _trace("stadium shadow", "stadium", 1 << 20, 1920, 1080, 16.0, 8, "shadow", "simple"),
        _trace("stadium bounce", "stadium", 1 << 20, 1920, 1080, 16.0, 8, "bounce", "simple"),
        # The same scene on the plain one-level grid, rebuilt for a 720p view
        # with shadows.
        _frame("stadium one level", "stadium", 1 << 20, 1280, 720, 128.0, 0, 0, "pooled"),
        # Ambient occlusion over clustered spheres: 4M triangles rebuilt, 8
        # rays per pixel at an odd image size.
        {"kind": "ao", "name": "ao 4M", "clusters": 1024, "width": 601, "height": 339, "spp": 8,
         "lam": 4.0, "mode": "simple"},
        # A queue of mixed jobs (thumbnails to 1024 pixels a side, depth 1..3).
        {"kind": "batch", "name": "batch of 16", "jobs": 16, "lam": 5.0, "mode": "pooled"},
        # Requests of a render service over resident scenes.
        {"kind": "serve", "name": "serve 24 requests", "scenes": 4, "requests": 24, "lam": 8.0,
         "mode": "simple"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, pixels):
    """An image of at most `pixels` pixels, odd sizes among them."""
    n = _log(rng, 48 * 48, pixels)
    ratio = rng.choice([1.0, 4 / 3, 16 / 9])
    h = max(24, int(math.sqrt(n / ratio)))
    return max(24, min(int(h * ratio), pixels // h)), h


MODES = ("simple", "simple", "pooled", "split2", "split4", "persistent")


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "trace", "trace", "trace", "ao", "batch",
                       "serve"])
    if kind in ("frame", "trace"):
        scene = rng.choice(["spheres", "stadium"])
        sub = rng.choice([0, 4, 8])
        if scene == "spheres":
            tris = 256 * int(_log(rng, 8, 2048))
            lam = round(rng.uniform(2.0, 8.0), 2)
            width, height = _size(rng, 1024 * 1024)
        else:
            tris = int(_log(rng, 20_000, 1 << 20))
            lam = round(_log(rng, 8.0, 16.0) if sub else _log(rng, 64.0, 256.0), 2)
            width, height = _size(rng, 1920 * 1080 if sub else 960 * 540)
        mode = rng.choice(MODES)
        if kind == "frame":
            graph = scene == "spheres" and rng.random() < 0.3
            return _frame(None, scene, tris, width, height, lam, sub, rng.randrange(2), mode,
                          graph)
        return _trace(None, scene, tris, width, height, lam, sub,
                      rng.choice(["primary", "shadow", "bounce"]), mode)
    if kind == "ao":
        width, height = _size(rng, 600 * 338)
        return {"kind": "ao", "clusters": int(_log(rng, 64, 1024)), "width": width,
                "height": height, "spp": rng.randint(1, 8), "lam": round(rng.uniform(2.0, 4.0), 2),
                "mode": rng.choice(["simple", "pooled", "persistent"])}
    if kind == "batch":
        return {"kind": "batch", "jobs": rng.randint(2, 12), "lam": round(rng.uniform(2.0, 8.0), 2),
                "mode": rng.choice(["simple", "pooled"])}
    return {"kind": "serve", "scenes": rng.randint(1, 4), "requests": rng.randint(2, 20),
            "lam": round(rng.uniform(2.0, 8.0), 2), "mode": rng.choice(["simple", "pooled"])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _geometry(case, seed):
    """(vertices, normals, cluster centres or None, (triangles per cluster,
    cluster triangles))."""
    if case["scene"] == "spheres":
        v, n = W.sphere_scene(W.SEED_SPHERES + 7919 * seed, case["tris"])
        return v, n, None, (0, 0)
    clusters = max(4, min(256, case["tris"] // 4096))
    inside = case["tris"] - 2               # the ground plane's two follow
    per = -(-inside // clusters)
    v, n, centers = grt.gen_stadium(W.SEED_STADIUM + 7919 * seed, clusters, per, inside)
    return v, n, centers, (per, inside)


def _camera(case):
    if case.get("scene") == "stadium":
        return grt.camera_lookat(STADIUM_EYE, STADIUM_CENTER, W.UP, W.FOVY, case["width"],
                                 case["height"])
    return W.camera(case["width"], case["height"])


def _batch_jobs(case):
    """(triangles, side, depth) per job: the case's own, whatever the seed."""
    rng = np.random.default_rng(W.SEED_BATCH + 31 * case["jobs"])
    n = case["jobs"]
    tris = W.log_uniform(rng, 2_000, MAX_BATCH_TRIS, n).astype(np.int64)
    side = np.round(W.log_uniform(rng, 64, 1024, n)).astype(np.int64)
    depth = rng.integers(1, 4, n)
    return [(int(t), int(s), int(d)) for t, s, d in zip(tris, side, depth)]


def _serve_spec(case):
    """Scene sizes and (scene, width, height, depth) per request."""
    rng = np.random.default_rng(W.SEED_SERVE + 131 * case["scenes"] + case["requests"])
    tris = [int(x) for x in W.log_uniform(rng, 10_000, MAX_SERVE_TRIS, case["scenes"])]
    res = rng.integers(0, len(W.SERVE_RESOLUTIONS), case["requests"])
    scene = rng.integers(0, case["scenes"], case["requests"])
    depth = rng.integers(2, 5, case["requests"])
    return tris, [(int(s),) + W.SERVE_RESOLUTIONS[r] + (int(d),)
                  for s, r, d in zip(scene, res, depth)]


def _hits(n):
    h = grt.HitBatch.empty(n, DEV)
    h.f["id"].fill_(-1)
    for k in ("t", "u", "v"):
        h.f[k].zero_()
    return h


def _zeros(n, dtype):
    return torch.zeros(n, dtype=dtype, device=DEV)


def _set_mode(ctx, mode):
    if mode.startswith("split"):
        ctx.set_trace_mode("split", int(mode[5:]))
    else:
        ctx.set_trace_mode(mode, 16)


class State:
    """A program's context, scenes and buffers; closed with the last reference."""

    def __init__(self, case):
        self.case = case
        self.ctx = grt.Context(0)
        self.close_first = []
        self.stream = None
        _set_mode(self.ctx, case["mode"])

    def scene(self, v, n):
        sc = grt.Scene(self.ctx)
        sc.upload(v, n)
        return sc

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for x in self.close_first:
                x.close()
            self.ctx.close()
            if self.stream is not None:
                grt.stream_destroy(self.stream)
        except Exception:
            pass


def _reserve(sc, extra=1.25):
    info = sc.grid_info()
    sc.reserve_grid(int(info["m"] * extra) + 4096, int(info["r"] * extra) + 4096)
    return info


def _prepare_scene(st, case, seed):
    v, n, centers, st.clusters = _geometry(case, seed)
    st.sc = st.scene(v, n)
    st.xf = None
    if centers is not None:
        # two poses of the animation, used in turn
        st.xf = [grt.gen_cluster_transforms(W.SEED_STADIUM + seed, f, centers, 0.05)
                 for f in range(2)]
        st.sc.transform_clusters(st.xf[0], *st.clusters)
    st.sc.set_subgrid(4.0 if case["sub"] else 0.0, case["sub"] or 8)
    st.sc.build_grid(case["lam"])
    st.cam = _camera(case)
    st.n = case["width"] * case["height"]


def _prepare_frame(st, case, seed):
    _prepare_scene(st, case, seed)
    _reserve(st.sc, 1.5)
    st.rays = [grt.RayBatch.empty(st.n, DEV) for _ in range(1 + case["bounces"])]
    st.hits = [_hits(st.n) for _ in st.rays]
    st.shadow = [grt.RayBatch.empty(st.n, DEV) for _ in st.rays]
    st.occ = [_zeros(st.n, torch.uint8) for _ in st.rays]
    st.rgb = _zeros((st.n, 3), torch.float32)
    st.rgba = _zeros(st.n, torch.int32)
    st.phong = grt.phong({"light": W.LIGHT})
    st.graph = None
    if case["graph"]:
        st.stream = grt.stream_create()
        torch.cuda.synchronize()
        st.ctx.set_stream(st.stream)
        _frame_calls(st)
        st.ctx.synchronize()
        st.graph = grt.Graph(st.ctx)
        st.graph.begin()
        _frame_calls(st)
        st.graph.end()
        st.close_first.append(st.graph)
        st.ctx.set_stream(torch.cuda.current_stream().cuda_stream)


def _frame_calls(st):
    sc, case, w = st.sc, st.case, st.case["width"]
    if st.xf is not None:
        sc.transform_clusters(st.xf[1], *st.clusters)
    sc.rebuild_grid_async(case["lam"])
    st.ctx.gen_primary(st.cam, st.rays[0])
    for k, (rays, hits) in enumerate(zip(st.rays, st.hits)):
        sc.trace_closest(rays, hits, image_width=w)
        sc.gen_shadow(rays, hits, W.LIGHT, OFFSET, st.shadow[k])
        sc.trace_any(st.shadow[k], st.occ[k], image_width=w)
        if k < case["bounces"]:
            sc.gen_reflection(rays, hits, OFFSET, st.rays[k + 1])
        sc.shade_phong(rays, hits, st.rgb, st.occ[k], k, st.phong,
                       rgba=st.rgba if k == case["bounces"] else None)


def _run_frame(st):
    if st.graph is not None:
        st.graph.launch()
    else:
        _frame_calls(st)
    return {"rgb": st.rgb, "rgba": st.rgba,
            "hits": [h.f for h in st.hits], "occluded": st.occ}


def _prepare_trace(st, case, seed):
    _prepare_scene(st, case, seed)
    w = case["width"]
    prim, hits = grt.RayBatch.empty(st.n, DEV), _hits(st.n)
    st.ctx.gen_primary(st.cam, prim)
    st.rays = prim
    if case["rays"] != "primary":
        st.ctx.set_trace_mode("simple", 16)
        st.sc.trace_closest(prim, hits, image_width=w)
        st.rays = grt.RayBatch.empty(st.n, DEV)
        if case["rays"] == "shadow":
            st.sc.gen_shadow(prim, hits, W.LIGHT, OFFSET, st.rays)
        else:
            st.sc.gen_reflection(prim, hits, OFFSET, st.rays)
        _set_mode(st.ctx, case["mode"])
    st.hits = _hits(st.n) if case["rays"] != "shadow" else None
    st.occ = _zeros(st.n, torch.uint8) if case["rays"] == "shadow" else None


def _run_trace(st):
    w = st.case["width"]
    if st.hits is None:
        st.sc.trace_any(st.rays, st.occ, image_width=w)
        return {"occluded": st.occ}
    st.sc.trace_closest(st.rays, st.hits, image_width=w)
    return {"hits": st.hits.f}


def _prepare_ao(st, case, seed):
    v, n = grt.gen_sphere_clusters(W.SEED_AO + 7919 * seed, case["clusters"], 16, 0.02, 0.003,
                                   0.012)
    st.sc = st.scene(v, n)
    st.sc.build_grid(case["lam"])
    info = _reserve(st.sc, 1.1)
    st.tmax = 0.05 * float(np.max(info["bmax"] - info["bmin"]))
    st.cam = W.ao_camera(case["width"], case["height"])
    st.n = case["width"] * case["height"]
    st.prim, st.hits = grt.RayBatch.empty(st.n, DEV), _hits(st.n)
    st.rays = grt.RayBatch.empty(st.n * case["spp"], DEV)
    st.occ = _zeros(st.n * case["spp"], torch.uint8)
    st.seed = W.SEED_AO + seed


def _run_ao(st):
    case = st.case
    st.sc.rebuild_grid_async(case["lam"])
    st.ctx.gen_primary(st.cam, st.prim)
    st.sc.trace_closest(st.prim, st.hits, image_width=case["width"])
    st.sc.gen_ao(st.prim, st.hits, case["spp"], st.seed, OFFSET, st.tmax, st.rays)
    st.sc.trace_any(st.rays, st.occ)
    return {"hits": st.hits.f, "occluded": st.occ}


def _slices(total_hits, occ, sizes):
    """Per-job hit and occlusion buffers out of whole ones."""
    at, out = 0, []
    for n in sizes:
        out.append((grt.HitBatch({k: x[at:at + n] for k, x in total_hits.f.items()}),
                    None if occ is None else occ[at:at + n]))
        at += n
    return out


def _prepare_batch(st, case, seed):
    jobs = _batch_jobs(case)
    sizes = [s * s for _, s, _ in jobs]
    total = sum(sizes)
    st.all_hits = [_hits(total), _hits(total)]
    st.all_occ = _zeros(total, torch.uint8)
    even = _slices(st.all_hits[0], st.all_occ, sizes)
    odd = _slices(st.all_hits[1], None, sizes)
    st.jobs = []
    for i, (tris, side, depth) in enumerate(jobs):
        sc = st.scene(*W.sphere_scene(W.SEED_BATCH + 1000 * seed + i, tris))
        sc.build_grid(case["lam"])
        n = side * side
        st.jobs.append({"scene": sc, "cam": W.camera(side, side), "side": side, "depth": depth,
                        "rays": [grt.RayBatch.empty(n, DEV), grt.RayBatch.empty(n, DEV)],
                        "hits": [even[i][0], odd[i][0]], "occ": even[i][1],
                        "shadow": grt.RayBatch.empty(n, DEV)})
    st.levels = 1 + max(j["depth"] for j in st.jobs)
    st.batches = []
    for level in range(st.levels):
        items = []
        for j in st.jobs:
            if level == 0:
                items.append((j["scene"], j["rays"][0], j["hits"][0], None, j["side"]))
            elif level <= j["depth"]:
                c = (level - 1) & 1
                items.append((j["scene"], j["shadow"], None, j["occ"], j["side"]))
                if level < j["depth"]:
                    items.append((j["scene"], j["rays"][1 - c], j["hits"][1 - c], None,
                                  j["side"]))
        b = grt.Batch(st.ctx, len(items))
        b.set(items)
        st.batches.append(b)
        st.close_first.append(b)


def _run_batch(st):
    for level in range(st.levels):
        for j in st.jobs:
            if level == 0:
                st.ctx.gen_primary(j["cam"], j["rays"][0])
            elif level <= j["depth"]:
                c = (level - 1) & 1
                j["scene"].gen_shadow(j["rays"][c], j["hits"][c], W.LIGHT, OFFSET, j["shadow"])
                if level < j["depth"]:
                    j["scene"].gen_reflection(j["rays"][c], j["hits"][c], OFFSET,
                                              j["rays"][1 - c])
        st.batches[level].trace()
    return {"hits": [h.f for h in st.all_hits], "occluded": st.all_occ}


def _prepare_serve(st, case, seed):
    tris, spec = _serve_spec(case)
    scenes = []
    for i, t in enumerate(tris):
        sc = st.scene(*W.sphere_scene(W.SEED_SERVE + 1000 * seed + i, t))
        sc.build_grid(case["lam"])
        scenes.append(sc)
    sizes = [w * h for _, w, h, _ in spec]
    st.all_hits, st.all_occ = _hits(sum(sizes)), _zeros(sum(sizes), torch.uint8)
    st.requests = [(scenes[s], W.camera(w, h), d) + out
                   for (s, w, h, d), out in zip(spec, _slices(st.all_hits, st.all_occ, sizes))]
    # the server runs on a stream of its own, kept for the program's life
    st.stream = grt.stream_create()
    torch.cuda.synchronize()
    st.ctx.set_stream(st.stream)
    st.server = grt.Server(st.ctx, 1 << 30, 64, True, W.LIGHT, OFFSET)
    st.close_first.append(st.server)


def _run_serve(st):
    tickets = [st.server.submit(sc, cam, depth, hits, occ)
               for sc, cam, depth, hits, occ in st.requests]
    rays = [st.server.wait(t)["rays"] for t in tickets]
    return {"hits": st.all_hits.f, "occluded": st.all_occ,
            "rays": np.array(rays, np.int64)}


def prepare(case, seed):
    st = State(case)
    globals()["_prepare_" + case["kind"]](st, case, seed)
    torch.cuda.synchronize()
    return st


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how near its outputs have to be
# ---------------------------------------------------------------------------
TEST_FLOPS = 50     # one ray-triangle test


def _grid_bytes(tris, lam):
    """A rebuild reads every triangle and writes an offset per cell and at
    least one reference per triangle."""
    return tris * (36 + 4) + 4 * lam * tris


def work(case):
    kind = case["kind"]
    if kind == "frame":
        n = case["width"] * case["height"]
        rays = n * (1 + case["bounces"])
        # per level: the hit record, the shadow flag; then the image
        out = rays * (16 + 1) + n * 16
        moved = case["tris"] * 2 * 72 if case["scene"] == "stadium" else 0
        return {"bytes": _grid_bytes(case["tris"], case["lam"]) + moved + out,
                "flops": rays * 2 * TEST_FLOPS}
    if kind == "trace":
        n = case["width"] * case["height"]
        return {"bytes": n * (32 + (1 if case["rays"] == "shadow" else 16)) + 36 * case["tris"],
                "flops": n * TEST_FLOPS}
    if kind == "ao":
        n, tris = case["width"] * case["height"], case["clusters"] * 16 * 256
        return {"bytes": _grid_bytes(tris, case["lam"]) + n * (16 + case["spp"]),
                "flops": n * (1 + case["spp"]) * TEST_FLOPS}
    if kind == "batch":
        jobs = _batch_jobs(case)
        rays = sum(s * s * d for _, s, d in jobs)
        return {"bytes": sum(36 * t for t, _, _ in jobs) + rays * 17,
                "flops": 2 * rays * TEST_FLOPS}
    tris, spec = _serve_spec(case)
    rays = sum(w * h * d for _, w, h, d in spec)
    return {"bytes": 36 * sum(tris) + rays * 17, "flops": 2 * rays * TEST_FLOPS}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits: closest hits by brute force over all triangles
# ---------------------------------------------------------------------------
MAX_PAIRS = 2e10


def _cross(a, b):
    return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _brute_closest(v, o, d, tmin):
    """t, u, v of the nearest triangle of every ray (inf, 0, 0 on a miss):
    v [n, 9], o and d lists of three [rays] tensors, all float64."""
    n, rays = v.shape[0], d[0].numel()
    v0 = [v[:, k][None] for k in range(3)]
    e1 = [(v[:, 3 + k] - v[:, k])[None] for k in range(3)]
    e2 = [(v[:, 6 + k] - v[:, k])[None] for k in range(3)]
    out = [torch.empty(rays, dtype=torch.float64, device=v.device) for _ in range(3)]
    step = max(1, int((1 << 24) // n))
    for a in range(0, rays, step):
        oo = [x[a:a + step, None] for x in o]
        dd = [x[a:a + step, None] for x in d]
        p = _cross(dd, e2)
        inv = 1.0 / _dot(p, e1)
        tv = [x - y for x, y in zip(oo, v0)]
        u = _dot(p, tv) * inv
        q = _cross(tv, e1)
        w = _dot(q, dd) * inv
        t = _dot(q, e2) * inv
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t > tmin)
        t, at = torch.where(ok, t, torch.full_like(t, math.inf)).min(1)
        miss = torch.isinf(t)
        out[0][a:a + step] = t
        for k, x in ((1, u), (2, w)):
            x = x.gather(1, at[:, None])[:, 0]
            out[k][a:a + step] = torch.where(miss, torch.zeros_like(x), x)
    return {"id": None, "t": out[0], "u": out[1], "v": out[2]}


def exact(case, seed):
    """Closest hits of the primary rays of a sphere scene; the other outputs
    (ids, flags, colours clamped to bytes, secondary rays that start from a
    rounded hit) have no such value, and larger scenes would take too long."""
    if case["kind"] not in ("frame", "trace") or case["scene"] != "spheres" or \
            case.get("rays", "primary") != "primary" or \
            case["tris"] * case["width"] * case["height"] > MAX_PAIRS:
        return None
    dev = DEV if torch.cuda.is_available() else "cpu"
    v = torch.from_numpy(_geometry(case, seed)[0]).to(dev).double()
    cam, w, h = _camera(case), case["width"], case["height"]
    x = torch.arange(w, device=dev, dtype=torch.float64).repeat(h) / w
    y = torch.arange(h, device=dev, dtype=torch.float64).repeat_interleave(w) / h
    d = [cam.base[k] + cam.nu[k] * x + cam.nv[k] * y for k in range(3)]
    o = [torch.full_like(x, cam.pos[k]) for k in range(3)]
    hits = _brute_closest(v, o, d, float(grt.RAY_EPSILON))
    if case["kind"] == "trace":
        return {"hits": hits}
    levels = 1 + case["bounces"]
    none = {"id": None, "t": None, "u": None, "v": None}
    return {"rgb": None, "rgba": None, "hits": [hits] + [none] * (levels - 1),
            "occluded": [None] * levels}
