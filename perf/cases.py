"""The work a program has this framework do, as measurable cases.

A renderer or simulator that uses the framework (re)builds a BVH over
primitives that already lie in GPU memory and then traces it. So a build case
is one rebuild through the builder API (the previous tree freed, a new one
built) and, for triangle BVH8s, one small batch of closest-hit queries against
the new tree: picking or visibility probes. The hits come back with the
primitive order and the bounds, since a BVH8's node numbering within a level
is free while what a ray hits is not. BVH2 builds return the whole node array.

Sizes: the five workloads of bench.py (300K, 1.1M, 2.9M and 28.1M triangles,
2,048 meshes of 64 to 65,536), the published scene sizes of the method (12.7M
among them), and small odd counts as in the tests.

Kinds:
  bvh8   BuildBVH8 / BuildBVH8Indexed, then the probe rays (none for boxes)
  bvh2   BuildBVH2, or the allocation-free build for serving loops
  batch  one run of a kept batch plan, then probe rays against some meshes
  trace  closest hits of a frame of rays against a kept BVH8
  train  one gradient + Adam step of the radius network
"""
import ctypes
import math
import os
import random
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

# One HIP runtime in the process: torch's. The library's own buffers, streams
# and copies then go through the runtime that torch uses.
os.environ.setdefault("NXB_HIP_RUNTIME", os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so"))

from nexusbvh_amd import builder as B  # noqa: E402
from nexusbvh_amd import learned as L  # noqa: E402
from nexusbvh_amd import native, scenes  # noqa: E402
from nexusbvh_amd.batch import BatchPlan  # noqa: E402

MAX_PAIRS = 4e10       # ray-triangle pairs that exact() tests by brute force
PLANE_EXTENT = 20.53   # side of the blob scene's ground plane
RADII = (1.3, 13.0, 1.0, 1.0)  # bounding radius of: surface, blobs, uniform, slivers


def listed():
    return [
        # The smallest rebuild in use: one animated object of a few thousand
        # triangles, where latency and launches are all there is.
        dict(name="bvh8 2k surface", kind="bvh8", scene="surface", prim="tri", n=2003, bits=64, mode=0, radius=8,
             learned=False, rays=1024),
        # The same for boxes in a serving loop that may not allocate.
        dict(name="bvh2 16k boxes noalloc", kind="bvh2", scene="uniform", prim="box", n=16411, bits=64, mode=0,
             radius=8, noalloc=True),
        # A hair or foliage asset of odd size with the short keys.
        dict(name="bvh8 48k slivers", kind="bvh8", scene="slivers", prim="tri", n=47989, bits=32, mode=0, radius=8,
             learned=False, rays=4096),
        # A character or building as an indexed mesh (the usual asset format).
        dict(name="bvh8 300k indexed", kind="bvh8", scene="surface", prim="indexed", n=300_000, bits=64, mode=0,
             radius=8, learned=False, rays=16384),
        # A scanned surface of 1.1M triangles with the short keys.
        dict(name="bvh8 1m1 surface k32", kind="bvh8", scene="surface", prim="tri", n=1_100_000, bits=32, mode=0,
             radius=8, learned=False, rays=16384),
        # Hair at full size, in the native 64-lane schedule.
        dict(name="bvh8 2m9 slivers wave64", kind="bvh8", scene="slivers", prim="tri", n=2_900_000, bits=64, mode=1,
             radius=8, learned=False, rays=16384),
        # A very uneven scene whose search radius the network picks.
        dict(name="bvh8 1m9 learned", kind="bvh8", scene="blobs", prim="tri", n=1_900_003, bits=64, mode=0, radius=8,
             learned=True, rays=16384),
        # A whole plant as a BVH2 (12.7M triangles, short keys).
        dict(name="bvh2 12m7 blobs k32", kind="bvh2", scene="blobs", prim="tri", n=12_700_000, bits=32, mode=0,
             radius=8, noalloc=False),
        # The headline: 28.1M triangles, 64-bit keys, defaults.
        dict(name="bvh8 28m1 blobs", kind="bvh8", scene="blobs", prim="tri", n=28_100_000, bits=64, mode=0, radius=8,
             learned=False, rays=16384),
        # All objects of a scene rebuilt at once from one kept plan.
        dict(name="batch 2048 meshes", kind="batch", meshes=2048, lo=64, hi=65536, mode=0, radius=8, probed=8,
             rays=4096),
        # A frame of primary rays against a kept 1.1M-triangle BVH8.
        dict(name="trace 1m primary", kind="trace", scene="surface", n=1_100_000, rays=1 << 20, coherent=True),
        # One training step of the radius network (batch of learned.train).
        dict(name="train step 8192", kind="train", rows=8192),
    ]


def _size(rng, lo, hi):
    """Log-uniform, odd more often than not."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n | 1 if rng.random() < 0.7 else n


def draw(rng: random.Random):
    k = rng.random()
    if k < 0.5:
        n = _size(rng, 500, 20_000_000)
        prim = rng.choice(("tri", "tri", "indexed", "box"))
        scene = "surface" if prim == "indexed" else rng.choice(("surface", "blobs", "uniform", "slivers"))
        return dict(kind="bvh8", scene=scene, prim=prim, n=n, bits=rng.choice((32, 64)),
                    mode=rng.choice((0, 0, 1)), radius=rng.choice((8, 8, 8, 4, 16)),
                    learned=n > 50_000 and rng.random() < 0.2, rays=0 if prim == "box" else min(16384, max(512, n // 8)))
    if k < 0.7:
        noalloc = rng.random() < 0.4
        n = _size(rng, 300, 500_000 if noalloc else 20_000_000)
        return dict(kind="bvh2", scene=rng.choice(("surface", "blobs", "uniform", "slivers")),
                    prim=rng.choice(("tri", "box")), n=n, bits=rng.choice((32, 64)), mode=rng.choice((0, 0, 1)),
                    radius=rng.choice((8, 8, 4)), noalloc=noalloc)
    if k < 0.83:
        return dict(kind="batch", meshes=_size(rng, 32, 2048), lo=64, hi=rng.choice((4096, 16384, 65536)),
                    mode=rng.choice((0, 0, 1)), radius=rng.choice((8, 8, 4)), probed=8, rays=4096)
    if k < 0.95:
        return dict(kind="trace", scene=rng.choice(("surface", "uniform", "blobs")), n=_size(rng, 20_000, 3_000_000),
                    rays=_size(rng, 1 << 16, 1 << 20), coherent=rng.random() < 0.5)
    return dict(kind="train", rows=_size(rng, 1024, 32768))


# ---- inputs, made on the GPU from the seed --------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _surface_mesh(n, g):
    """(vertices, indices) of a closed-looking displaced sphere patch: a grid
    of quads in row order, two triangles each, cut at n triangles."""
    side = math.isqrt((n + 1) // 2 - 1) + 1 if n > 2 else 1
    t = torch.arange(side + 1, device="cuda", dtype=torch.float32) / side
    th, ph = torch.meshgrid(0.1 + (math.pi - 0.2) * t, 2 * math.pi * t, indexing="ij")
    p = torch.stack((th.sin() * ph.cos(), th.sin() * ph.sin(), th.cos()), -1).reshape(-1, 3)
    freq = _randn(g, 3, 6) * torch.tensor([2.0, 3.0, 5.0, 8.0, 13.0, 21.0], device="cuda")
    amp = torch.tensor([8.0, 5.0, 3.0, 2.0, 1.0, 0.7], device="cuda") * 0.008
    r = 1.0 + (torch.sin(p @ freq + 6.2831853 * _rand(g, 6)) * amp).sum(-1, keepdim=True)
    verts = (p * r).contiguous()
    q = torch.arange(side * side, device="cuda", dtype=torch.int64)
    a = (q // side) * (side + 1) + q % side
    idx = torch.stack((a, a + side + 1, a + side + 2, a, a + side + 2, a + 1), -1).reshape(-1, 3)[:n]
    return verts, idx.to(torch.int32).contiguous()


def _triangles(scene, n, g):
    """(n, 9) float32 triangles."""
    if scene == "surface":
        v, i = _surface_mesh(n, g)
        return v[i.long().reshape(-1)].reshape(n, 9).contiguous()
    if scene == "uniform":
        c = _rand(g, n, 1, 3)
        return (c + (_rand(g, n, 3, 3) - 0.5) * 0.01).reshape(n, 9).contiguous()
    if scene == "slivers":
        d = _unit(_randn(g, n, 3))
        w = _unit(torch.linalg.cross(d, _unit(_randn(g, n, 3)))) * 1e-4
        p0 = 0.08 + 0.84 * _rand(g, n, 3)
        p1 = p0 + d * (0.02 + 0.06 * _rand(g, n, 1))
        return torch.cat((p0, p1, p0 + w), -1).contiguous()
    # blobs: 64 Gaussian clouds of small triangles over a ground-plane grid
    side = max(1, int(math.sqrt(0.15 * n)))
    plane = 2 * side * side
    nb = n - plane
    mu = torch.cat((_rand(g, 64, 2) * PLANE_EXTENT, 0.05 + 1.95 * _rand(g, 64, 1)), -1)
    sigma = torch.exp(math.log(0.001) + math.log(50.0) * _rand(g, 64))
    k = torch.arange(nb, device="cuda") * 64 // max(1, nb)
    s = sigma[k].reshape(nb, 1, 1)
    c = mu[k].reshape(nb, 1, 3) + s * _randn(g, nb, 1, 3)
    out = torch.empty(n, 9, device="cuda")
    out[:nb] = (c + 0.2 * s * (_rand(g, nb, 3, 3) - 0.5)).reshape(nb, 9)
    t = torch.arange(plane, device="cuda")
    q = t // 2
    lo = torch.stack((q % side, q // side), -1).float()
    corner = torch.tensor([[[0, 0], [1, 0], [1, 1]], [[0, 0], [1, 1], [0, 1]]], device="cuda", dtype=torch.float32)
    xy = (lo[:, None, :] + corner[t % 2]) * (PLANE_EXTENT / side)
    out[nb:] = torch.cat((xy, torch.zeros(plane, 3, 1, device="cuda")), -1).reshape(plane, 9)
    return out


def _radius(scene):
    return RADII[("surface", "blobs", "uniform", "slivers").index(scene)]


def _probe_rays(tris, count, radius, g):
    """Short probes (contact, occlusion, picking under a cursor): each starts a
    twentieth of the scene's radius away from a point of a random triangle,
    points at it and ends as far behind it."""
    pick = (_rand(g, count) * (len(tris) - 0.5)).long().clamp_(0, len(tris) - 1)
    target = tris[pick].reshape(count, 3, 3).mean(1)
    d = _unit(_randn(g, count, 3))
    return _rays(target - d * (0.05 * radius), d, 0.1 * radius)


def _rays(o, d, tmax):
    r = torch.zeros(len(o), 8, device="cuda")
    r[:, :3], r[:, 4:7], r[:, 7] = o, d, tmax
    return r


def _camera_rays(tris, count, radius, g):
    """Pinhole primary rays, row by row, at the middle of the scene."""
    v = tris[:: max(1, len(tris) // 65536)].reshape(-1, 3)
    centre = (v.amin(0) + v.amax(0)) * 0.5
    view = _unit(_randn(g, 3))
    right = _unit(torch.linalg.cross(view, _unit(_randn(g, 3))))
    up = torch.linalg.cross(right, view)
    w = max(1, math.isqrt(count))
    i = torch.arange(count, device="cuda")
    rows = -(-count // w)
    x = ((i % w).float() + 0.5) / w * 2 - 1
    y = ((i // w).float() + 0.5) / rows * 2 - 1
    d = _unit(view + 0.36 * (x[:, None] * right + y[:, None] * up))
    return _rays((centre - view * (2.5 * radius)).expand(count, 3), d, 6.0 * radius)


def _random_rays(tris, count, radius, g):
    """Incoherent rays: origins in the grown scene box, any direction."""
    v = tris[:: max(1, len(tris) // 65536)].reshape(-1, 3)
    lo, hi = v.amin(0), v.amax(0)
    o = lo - 0.5 * (hi - lo) + _rand(g, count, 3) * (2.0 * (hi - lo))
    return _rays(o, _unit(_randn(g, count, 3)), 6.0 * radius)


def _batch_counts(case):
    """Triangles per mesh: fixed by the case, log-uniform in [lo, hi]."""
    rng = np.random.default_rng(case["meshes"])
    c = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["meshes"]))
    return np.clip(np.round(c).astype(np.int64), case["lo"], case["hi"])


def _batch_triangles(counts, seed):
    """bench.py's spheres, boxes and tori, back to back, each under its own
    rotation, scale and place."""
    offsets = np.concatenate(([0], np.cumsum(counts)))
    tris = np.empty((int(offsets[-1]), 9), dtype=np.float32)

    def fill(m):
        tris[offsets[m]:offsets[m + 1]] = scenes.batch_mesh(m, int(counts[m]), seed + 1)

    with ThreadPoolExecutor(8) as pool:
        list(pool.map(fill, range(len(counts))))
    return torch.from_numpy(tris).cuda()


def _boxes(tris):
    v = tris.reshape(-1, 3, 3)
    return torch.cat((v.amin(1), v.amax(1)), -1).contiguous()


def _network():
    """The shipped weights of the radius network."""
    return torch.tensor(L.load(), device="cuda")


def _training(case, g):
    """(features, labels, parameters, Adam moments) of a run in progress."""
    x = _randn(g, case["rows"], L.FEATURES) * 0.5
    w = _randn(g, L.FEATURES, L.CLASSES)
    y = (x @ w + 0.5 * _randn(g, case["rows"], L.CLASSES)).argmax(-1).to(torch.uint8)
    p = torch.tensor(L.init_params(3), device="cuda")
    m = 1e-3 * _randn(g, L.PARAMS)
    return x.contiguous(), y, p, m, m * m + 1e-6


# ---- preparation and one pass ---------------------------------------------

def _view(t):
    """The framework's non-owning buffer over a torch tensor."""
    return native.DeviceView(t.data_ptr(), t.numel() * t.element_size(), t)


class _Memory:
    """int32 device memory as torch sees it."""

    def __init__(self, address, *shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<i4", data=(address, False), version=2)


def _tensor(address, *shape):
    return torch.as_tensor(_Memory(address, *shape), device="cuda")


class _Tree:
    """The current BVH of a program that rebuilds it."""

    def __init__(self):
        self.bvh = None

    def replace(self, bvh=None):
        if self.bvh is not None:
            B.FreeDeviceBVH(self.bvh)
        self.bvh = bvh

    def __del__(self):
        try:
            self.replace()
        except Exception:
            pass


def _config(case):
    cfg = B.BuildConfig(mortonBits=case["bits"], searchRadius=case["radius"], mergeMode=B.MergeMode(case["mode"]))
    weights = None
    if case.get("learned"):
        weights = _network()
        cfg.radiusPolicy = B.RadiusPolicy.LEARNED
        cfg.mlpParams = _view(weights)
    return cfg, weights


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("bvh8", "bvh2"):
        n = case["n"]
        s["cfg"], s["weights"] = _config(case)
        if case["prim"] == "indexed":
            v, i = _surface_mesh(n, g)
            s["mesh"] = B.DeviceIndexedMesh(_view(v), _view(i), len(v), n)
            s["vertices"], s["indices"] = v, i
            tris = v[i[:: max(1, n // 65536)].long().reshape(-1)].reshape(-1, 9)
        else:
            tris = _triangles(case["scene"], n, g)
            data = _boxes(tris) if case["prim"] == "box" else tris
            s["data"] = data
            s["prims"] = B.DevicePrimitives(_view(data), n,
                                            B.PrimType.AABB if case["prim"] == "box" else B.PrimType.TRIANGLE)
        if case.get("rays"):
            s["rays"] = _probe_rays(tris, case["rays"], _radius(case["scene"]), g)
            s["hits"] = torch.empty(case["rays"], 4, device="cuda")
        if case.get("noalloc"):
            s["nodes"] = torch.empty(2 * n - 1, 8, dtype=torch.int32, device="cuda")
        s["tree"] = _Tree()
    elif kind == "batch":
        counts = _batch_counts(case)
        tris = _batch_triangles(counts, seed)
        offsets = np.concatenate(([0], np.cumsum(counts))).astype(np.uint32)
        s["data"] = tris
        s["prims"] = B.DevicePrimitives(_view(tris), len(tris), B.PrimType.TRIANGLE)
        torch.cuda.synchronize()
        s["plan"] = BatchPlan(s["prims"], offsets, B.BuildConfig(mortonBits=32, searchRadius=case["radius"],
                                                                 mergeMode=B.MergeMode(case["mode"])))
        s["probed"] = _probed(case, seed)
        s["rays"], s["hits"] = [], []
        for m in s["probed"]:
            part = tris[int(offsets[m]):int(offsets[m + 1])]
            v = part.reshape(-1, 3)
            s["rays"].append(_probe_rays(part, case["rays"], float((v.amax(0) - v.amin(0)).norm()) * 0.5, g))
            s["hits"].append(torch.empty(case["rays"], 4, device="cuda"))
        s["offsets"] = offsets
    elif kind == "trace":
        tris = _triangles(case["scene"], case["n"], g)
        s["data"] = tris
        s["prims"] = B.DevicePrimitives(_view(tris), case["n"], B.PrimType.TRIANGLE)
        make = _camera_rays if case["coherent"] else _random_rays
        s["rays"] = make(tris, case["rays"], _radius(case["scene"]), g)
        s["hits"] = torch.empty(case["rays"], 4, device="cuda")
        torch.cuda.synchronize()
        s["tree"] = _Tree()
        s["tree"].replace(B.BuildBVH8(s["prims"], case["n"]))
    else:
        x, y, p, m, v = _training(case, g)
        s.update(x=x, y=y, p=p, m=m, v=v, step=100, grads=torch.empty_like(p), loss=torch.empty(1, device="cuda"))
        s["views"] = [_view(s[k]) for k in ("p", "x", "y", "grads", "loss")]
    torch.cuda.synchronize()
    return s


def _probed(case, seed):
    rng = np.random.default_rng(seed)
    return [int(m) for m in np.sort(rng.choice(case["meshes"], case["probed"], replace=False))]


def _bounds(bvh):
    return np.array(B.bvh_bounds(bvh), dtype=np.float32)


def _trace(bvh, s, rays, hits, tris=None):
    """Closest hits into a kept buffer: (t, u, v per ray; primitive per ray)."""
    if "mesh" in s:
        m = s["mesh"]
        native.check(native.lib().nxb_trace_closest_indexed(
            ctypes.byref(bvh), m.vertices.address, m.vertexCount, m.indices.address, rays.data_ptr(), len(rays),
            hits.data_ptr(), None, None), "nxb_trace_closest_indexed")
    else:
        native.check(native.lib().nxb_trace_closest(ctypes.byref(bvh), tris or s["prims"].address, rays.data_ptr(),
                                                    len(rays), hits.data_ptr(), None, None), "nxb_trace_closest")
    return {"t": hits[:, 0], "uv": hits[:, 2:4], "prim": hits[:, 1].view(torch.int32)}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "bvh8":
        s["tree"].replace()
        if "mesh" in s:
            bvh = B.BuildBVH8Indexed(s["mesh"], s["cfg"])
        else:
            bvh = B.BuildBVH8(s["prims"], case["n"], s["cfg"])
        s["tree"].replace(bvh)
        out = {"bounds": _bounds(bvh), "nodes": int(bvh.node_count),
               "primIdx": _tensor(bvh.prim_idx, case["n"])}
        if "rays" in s:
            out["hits"] = _trace(bvh, s, s["rays"], s["hits"])
        return out
    if kind == "bvh2":
        if case["noalloc"]:
            out = native.BVH2()
            native.check(native.lib().nxb_build_bvh2_noalloc(
                s["prims"].address, int(s["prims"].prim_type), case["n"], ctypes.byref(s["cfg"].to_c()),
                s["nodes"].data_ptr(), ctypes.byref(out), None), "nxb_build_bvh2_noalloc")
            return {"bounds": _bounds(out), "nodes": s["nodes"]}
        s["tree"].replace()
        bvh = B.BuildBVH2(s["prims"], case["n"], s["cfg"])
        s["tree"].replace(bvh)
        return {"bounds": _bounds(bvh), "nodes": _tensor(bvh.nodes, 2 * case["n"] - 1, 8)}
    if kind == "batch":
        s["plan"].run()
        out = []
        for m, rays, hits in zip(s["probed"], s["rays"], s["hits"]):
            bvh = s["plan"].mesh(m)
            first = int(s["offsets"][m]) * 36
            out.append({"nodes": int(bvh.node_count), "bounds": _bounds(bvh),
                        "hits": _trace(bvh, s, rays, hits, s["prims"].address + first)})
        return {"nodes": s["plan"].node_total, "meshes": out}
    if kind == "trace":
        return _trace(s["tree"].bvh, s, s["rays"], s["hits"])
    p, x, y, grads, loss = s["views"]
    L.mlp_gradients(p, x, y, case["rows"], grads, loss)
    native.check(native.lib().nxb_mlp_adam_step(p.address, grads.address, s["m"].data_ptr(), s["v"].data_ptr(),
                                                s["step"], ctypes.c_float(3e-3), ctypes.c_float(0.9),
                                                ctypes.c_float(0.999), ctypes.c_float(1e-8), None), "adam")
    s["step"] += 1
    return {"loss": s["loss"], "grads": s["grads"], "params": s["p"], "m": s["m"], "v": s["v"]}


# ---- what a pass cannot do without ----------------------------------------

def work(case):
    """Primitives and rays read once, trees and hits written once. A BVH8 node
    holds about five children, so a tree of n primitives has about n / 4 of
    its 80-byte nodes. Operations: about 60 per primitive for box, key and
    node area, 8 slab tests of 20 per node a ray meets (about 10)."""
    kind = case["kind"]
    rays = case.get("rays", 0)
    ray_bytes, ray_flops = rays * 48.0, rays * 1600.0
    if kind == "bvh8":
        n = case["n"]
        per = {"tri": 36.0, "box": 24.0, "indexed": 18.0}[case["prim"]]
        return {"bytes": n * (per + 4.0 + 20.0) + ray_bytes, "flops": n * 60.0 + ray_flops}
    if kind == "bvh2":
        n = case["n"]
        return {"bytes": n * ((36.0 if case["prim"] == "tri" else 24.0) + 64.0), "flops": n * 60.0}
    if kind == "batch":
        n = float(_batch_counts(case).sum())
        return {"bytes": n * 60.0 + case["probed"] * ray_bytes, "flops": n * 60.0 + case["probed"] * ray_flops}
    if kind == "trace":
        # the tree and triangles once, or what the rays meet if that is less
        return {"bytes": ray_bytes + min(case["n"] * 60.0, rays * 860.0), "flops": ray_flops}
    return {"bytes": case["rows"] * 65.0 + L.PARAMS * 4.0 * 7, "flops": case["rows"] * 6.0 * L.PARAMS}


# ---- the same in 64 bits --------------------------------------------------

def _exact_bounds(tris):
    v = tris.reshape(-1, 3).double()
    return torch.stack((v.amin(0), v.amax(0)))


def _exact_hits(tris, rays):
    """Closest hits by testing every triangle (Moller and Trumbore)."""
    if len(tris) * float(len(rays)) > MAX_PAIRS:
        return None
    ts, us, vs = [], [], []
    step = min(len(tris), 1 << 20)
    block = max(1, int(3e7) // step)
    for r0 in range(0, len(rays), block):
        r = rays[r0:r0 + block].double()
        o, d, tmin, best = r[:, None, :3], r[:, None, 4:7], r[:, 3], r[:, 7].clone()
        bu, bv = torch.zeros_like(best), torch.zeros_like(best)
        for t0 in range(0, len(tris), step):
            v = tris[t0:t0 + step].double().reshape(1, -1, 3, 3)
            e1, e2 = v[:, :, 1] - v[:, :, 0], v[:, :, 2] - v[:, :, 0]
            pv = torch.linalg.cross(d.expand(-1, e2.shape[1], -1), e2.expand(len(r), -1, -1))
            inv = 1.0 / (e1 * pv).sum(-1)
            tv = o - v[:, :, 0]
            u = (tv * pv).sum(-1) * inv
            qv = torch.linalg.cross(tv, e1.expand(len(r), -1, -1))
            w = (d * qv).sum(-1) * inv
            t = (e2 * qv).sum(-1) * inv
            ok = (u >= 0) & (u <= 1) & (w >= 0) & (u + w <= 1) & (t >= tmin[:, None])
            near, at = torch.where(ok, t, torch.full_like(t, math.inf)).min(1)
            hit = near < best
            best = torch.where(hit, near, best)
            bu = torch.where(hit, u.gather(1, at[:, None])[:, 0], bu)
            bv = torch.where(hit, w.gather(1, at[:, None])[:, 0], bv)
        ts.append(best)
        us.append(bu)
        vs.append(bv)
    return {"t": torch.cat(ts), "uv": torch.stack((torch.cat(us), torch.cat(vs)), -1), "prim": None}


def _exact_training(case, seed):
    x, y, p, m, v = (t.double() if t.is_floating_point() else t.long() for t in _training(case, _gen(seed)))
    p.requires_grad_(True)
    sizes = (L.FEATURES * L.HIDDEN, L.HIDDEN, L.HIDDEN * L.HIDDEN, L.HIDDEN, L.HIDDEN * L.CLASSES, L.CLASSES)
    w1, b1, w2, b2, w3, b3 = torch.split(p, sizes)
    h = torch.relu(x @ w1.reshape(L.FEATURES, L.HIDDEN) + b1)
    h = torch.relu(h @ w2.reshape(L.HIDDEN, L.HIDDEN) + b2)
    loss = torch.nn.functional.cross_entropy(h @ w3.reshape(L.HIDDEN, L.CLASSES) + b3, y)
    grad, = torch.autograd.grad(loss, p)
    m = 0.9 * m + 0.1 * grad
    v = 0.999 * v + 0.001 * grad * grad
    new = p.detach() - 3e-3 * (m / (1 - 0.9 ** 100)) / ((v / (1 - 0.999 ** 100)).sqrt() + 1e-8)
    return {"loss": loss.detach().reshape(1), "grads": grad, "params": new, "m": m, "v": v}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_training(case, seed)
    g = _gen(seed)
    if kind == "batch":
        counts = _batch_counts(case)
        tris = _batch_triangles(counts, seed)
        offsets = np.concatenate(([0], np.cumsum(counts)))
        out = []
        for m in _probed(case, seed):
            part = tris[int(offsets[m]):int(offsets[m + 1])]
            v = part.reshape(-1, 3)
            rays = _probe_rays(part, case["rays"], float((v.amax(0) - v.amin(0)).norm()) * 0.5, g)
            out.append({"nodes": None, "bounds": _exact_bounds(part), "hits": _exact_hits(part, rays)})
        return {"nodes": None, "meshes": out}
    if kind == "trace":
        tris = _triangles(case["scene"], case["n"], g)
        make = _camera_rays if case["coherent"] else _random_rays
        return _exact_hits(tris, make(tris, case["rays"], _radius(case["scene"]), g))
    if case["prim"] == "indexed":
        v, i = _surface_mesh(case["n"], g)
        tris = v[i.long().reshape(-1)].reshape(-1, 9)
        aim = tris[:: max(1, case["n"] // 65536)]
        out = {"bounds": _exact_bounds(v[i.long().reshape(-1)])}
    else:
        tris = aim = _triangles(case["scene"], case["n"], g)
        out = {"bounds": _exact_bounds(tris)}
    if kind == "bvh2":
        return dict(out, nodes=None)
    out.update(nodes=None, primIdx=None)
    if case["rays"]:
        out["hits"] = _exact_hits(tris, _probe_rays(aim, case["rays"], _radius(case["scene"]), g))
    return out
