"""Workload cases of the library: what its users have it do, through its public entry points.

Each case is one call (or the calls of one step) on one scene: queries through the
Python classes and through device-resident buffers, tree builds, refits,
differentiable queries and batches of scenes.  Scenes, sizes and options are those
of the benchmark, the tests and the generators in quarry.scenes; draw() takes more
of the same ranges.

    listed()              the fixed cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   scene, tree, query buffers: what a program holds before the call
    run(state)            one pass; returns the pass's whole outputs
    work(case)            bytes and operations the pass cannot do without
    tolerance(case)       how far another correct implementation's outputs may be
    exact(case, seed)     the outputs in 64 bits by plain torch, or None
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quarry-gpu_amd"))

import quarry  # noqa: E402
from quarry import _abi as A  # noqa: E402
from quarry import autograd as G  # noqa: E402
from quarry import scenes as S  # noqa: E402

KIND = {"terrain": A.PRIM_TRI, "city": A.PRIM_TRI, "icosphere": A.PRIM_TRI,
        "points": A.PRIM_POINT, "gaussians": A.PRIM_GAUSS}
BUILDER = {"lbvh": A.BUILDER_LBVH, "sah": A.BUILDER_SAH}
ORDER = {"input": A.ORDER_INPUT, "morton": A.ORDER_MORTON, "morton_direction": A.ORDER_MORTON_DIRECTION}
ITEM_BYTES = {A.PRIM_TRI: 36, A.PRIM_POINT: 12, A.PRIM_GAUSS: 40}
# operations of one leaf test and one box test (adds, multiplies, compares)
LEAF_OPS = {A.PRIM_TRI: 70, A.PRIM_POINT: 8, A.PRIM_GAUSS: 500}
BOX_OPS = 18


def listed():
    return [
        # One interactive pick: a few hundred points against a small mesh through the
        # Python class with its default options; latency and launches are the cost.
        {"name": "host_closest_small", "op": "host", "query": "closest", "scene": "terrain", "prims": 8191,
         "queries": 257, "k": 0, "order": "input", "wide": False, "builder": "lbvh"},
        # Serving on resident buffers: distance of sample points to a large terrain.
        {"name": "closest_terrain_2M", "op": "closest", "scene": "terrain", "prims": 2097152, "queries": 100000,
         "k": 0, "order": "morton", "wide": True, "builder": "sah"},
        # The same index asked for the 16 nearest triangles (interpolation stencils).
        {"name": "knn16_terrain_2M", "op": "knn", "scene": "terrain", "prims": 2097152, "queries": 100000,
         "k": 16, "order": "morton", "wide": True, "builder": "sah"},
        # Fixed-radius neighbours in a scanned cloud (normals, densities); long ragged segments.
        {"name": "radius_points_1M", "op": "radius", "scene": "points", "prims": 1048576, "queries": 20000,
         "radius": 1.0, "order": "morton", "wide": True, "builder": "lbvh"},
        # Neighbours among Gaussian splats (solid ellipsoids): the costliest leaf test.
        {"name": "knn8_gaussians_1M", "op": "knn", "scene": "gaussians", "prims": 1048576, "queries": 20000,
         "k": 8, "order": "morton", "wide": True, "builder": "lbvh"},
        # Visibility over a city: a million closest-hit rays, cosine-distributed.
        {"name": "rays_city_1M", "op": "rays", "scene": "city", "prims": 1343488, "queries": 1000000,
         "rays": "cosine", "order": "morton", "wide": True, "builder": "sah"},
        # Building the index of a large mesh already on the GPU, up to its first answers.
        {"name": "build_lbvh_terrain_2M", "op": "build", "scene": "terrain", "prims": 2097152, "wide": True,
         "builder": "lbvh"},
        # The higher-quality index of an uneven scene.
        {"name": "build_sah_city_1M", "op": "build", "scene": "city", "prims": 1343488, "wide": True,
         "builder": "sah"},
        # A frame of a dynamic scene: 1 % of the vertices moved, new triangles from the host.
        {"name": "refit_dirty_terrain_131k", "op": "refit", "scene": "terrain", "prims": 131072, "mode": "dirty",
         "frac": 0.01, "wide": True, "builder": "lbvh"},
        # One optimisation step of a mesh distance loss: forward (build, closest) and backward.
        {"name": "grad_icosphere_328k", "op": "grad", "fn": "mesh", "scene": "icosphere", "prims": 327680,
         "queries": 262144, "builder": "lbvh"},
        # Many small scenes new each step: build them all, then 8 nearest for every scene's queries.
        {"name": "batch_step_64", "op": "batch", "mode": "step", "scenes": 64, "nmax": 65536, "qmax": 8192, "k": 8},
        # Many small scenes kept: one replay of the prepared closest-point plan.
        {"name": "batch_closest_256", "op": "batch", "mode": "query", "scenes": 256, "nmax": 65536, "qmax": 8192,
         "k": 0},
    ]


def _log(rng, lo, hi):
    """Log-uniform whole number in [lo, hi]."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["host", "closest", "knn", "radius", "rays", "build", "build", "refit", "grad", "batch"])
    builder = rng.choice(["lbvh", "sah"])
    scene = rng.choice(["terrain", "terrain", "city", "points", "gaussians"])
    if op == "host":
        query = rng.choice(["closest", "knn", "radius", "raycast"])
        if query == "raycast":
            scene = rng.choice(["terrain", "city"])
        c = {"op": op, "query": query, "scene": scene, "prims": _log(rng, 300, 131072), "queries": _log(rng, 1, 4096),
             "k": rng.randint(1, 32) if query == "knn" else 0, "order": rng.choice(["input", "morton"]),
             "wide": rng.choice([False, True]), "builder": builder}
        if query == "radius":
            c["radius"] = _draw_radius(rng, c)
        return c
    if op in ("closest", "knn", "radius"):
        c = {"op": op, "scene": scene, "prims": _log(rng, 4096, 2097152), "queries": _log(rng, 256, 100000),
             "order": rng.choice(["morton", "morton", "input"]), "wide": True, "builder": builder}
        if c["queries"] <= 20000 and rng.random() < 0.3:
            c["wide"] = False
        if scene == "gaussians":
            c["prims"], c["queries"] = min(c["prims"], 1048576), min(c["queries"], 20000)
        if op == "radius":
            c["queries"] = min(c["queries"], 20000)
            c["radius"] = _draw_radius(rng, c)
        else:
            c["k"] = rng.choice([1, 2, 4, 5, 8, 12, 16, 27, 32]) if op == "knn" else 0
        return c
    if op == "rays":
        scene = rng.choice(["terrain", "city"])
        return {"op": op, "scene": scene, "prims": _log(rng, 4096, 1343488), "queries": _log(rng, 1000, 1000000),
                "rays": rng.choice(["down", "cosine"]), "order": rng.choice(["input", "morton", "morton_direction"]),
                "wide": rng.random() < 0.8, "builder": builder}
    if op == "build":
        return {"op": op, "scene": scene, "prims": _log(rng, 1000, 2097152 if scene == "terrain" else 1048576),
                "wide": rng.choice([False, True]), "builder": builder}
    if op == "refit":
        mode = rng.choice(["dirty", "full"])
        return {"op": op, "scene": "terrain", "prims": _log(rng, 2000, 262144 if mode == "dirty" else 2097152),
                "mode": mode, "frac": round(math.exp(rng.uniform(math.log(0.0005), math.log(0.05))), 5),
                "wide": rng.choice([False, True]), "builder": builder}
    if op == "grad":
        fn = rng.choice(["mesh", "rays", "points", "gaussians"])
        return {"op": op, "fn": fn, "scene": {"mesh": "icosphere", "rays": "icosphere"}.get(fn, fn),
                "prims": _log(rng, 1280, 327680), "queries": _log(rng, 1000, 262144 if fn != "gaussians" else 65536),
                "builder": builder if fn in ("mesh", "rays") else "lbvh"}
    return {"op": "batch", "mode": rng.choice(["step", "query"]), "scenes": rng.randint(3, 128),
            "nmax": rng.choice([4096, 16384, 65536]), "qmax": rng.choice([512, 4096, 8192]),
            "k": rng.choice([0, 1, 4, 8])}


def _draw_radius(rng, c):
    if c["scene"] in ("points", "gaussians"):  # one to two mean spacings of the cloud
        return round(rng.uniform(0.6, 1.6) * 64.0 / c["prims"] ** (1.0 / 3.0), 4)
    return round(rng.uniform(0.5, 3.0), 3)


# ---- inputs ---------------------------------------------------------------------------


def _items(case, seed):
    """The scene's primitives, (prims, 9 | 3 | 10) float32."""
    if "radius" not in case:
        return _scene(case, seed)
    # the number of hits is to depend on the case alone: one scene per case, which the
    # seed starts at another primitive and scales by a power of two (exact)
    items = np.roll(_scene(case, 1), seed % case["prims"], axis=0)
    cols = [0, 1, 2, 7, 8, 9] if case["scene"] == "gaussians" else slice(None)
    items[:, cols] *= _radius_scale(seed)
    return items


def _radius_scale(seed):
    return np.float32(2.0) ** (seed % 7 - 3)


def _scene(case, seed):
    scene, n = case["scene"], case["prims"]
    if scene == "terrain":
        return np.ascontiguousarray(S.terrain(max(1, math.ceil(math.sqrt(n / 2.0))), seed)[:n])
    if scene == "city":
        ground = 128 if n >= 100000 else 8
        return np.ascontiguousarray(S.city(max(1, -(-(n - 2 * ground * ground) // 10)), seed, ground_cells=ground)[:n])
    if scene == "points":
        return S.point_cloud(n, seed)
    return S.gaussians(n, seed)


def _bounds(case, items):
    if KIND[case["scene"]] == A.PRIM_TRI:
        b = S.bounds_of(items)
        return b[:3] - np.float32(4.0), b[3:] + np.float32(4.0)
    return items[:, :3].min(axis=0), items[:, :3].max(axis=0)


def _queries(case, items, seed):
    if "radius" in case:
        lo, hi = _bounds(case, _scene(case, 1))
        q = S.query_points(lo, hi, case["queries"], 3)
        return np.random.default_rng([seed, 33]).permutation(q) * _radius_scale(seed)
    lo, hi = _bounds(case, items)
    return S.query_points(lo, hi, case["queries"], seed + 2)


def _batch(case, seed):
    """Scene-major primitives and offsets, query points and offsets; the sizes (log-uniform,
    as in S.workload_c5) depend on the case alone."""
    rng = np.random.default_rng([case["scenes"], case["nmax"], case["qmax"], case["k"]])
    ns = np.floor(np.exp(rng.uniform(math.log(256), math.log(case["nmax"]), case["scenes"]))).astype(int)
    qs = np.floor(np.exp(rng.uniform(math.log(32), math.log(case["qmax"] / 2), case["scenes"]))).astype(int)
    items = [S.batch_scene(i, int(n), seed) for i, n in enumerate(ns)]
    points = [S.query_points(*np.split(S.bounds_of(t), 2), int(q), seed * 7919 + i)
              for i, (t, q) in enumerate(zip(items, qs))]
    offsets = [np.concatenate([[0], np.cumsum([x.shape[0] for x in part])]).astype(np.int32)
               for part in (items, points)]
    return np.concatenate(items), offsets[0], np.concatenate(points), offsets[1]


def _rays(case, items, seed):
    f = S.down_rays if case.get("rays") == "down" else S.cosine_down_rays
    return f(items, case["queries"], seed + 3)


def _mesh(case, seed):
    """A noisy icosphere cut to the case's face count: vertices, faces."""
    level = 1
    while 20 * 4 ** level < case["prims"]:
        level += 1
    v, f, _ = S.icosphere(levels=level, seed=seed)
    return v, np.ascontiguousarray(f[: case["prims"]])


class _DeviceArray:
    """A device array of `owner`, as torch takes it: a tensor made from it keeps this
    object, and with it the handle whose memory it shows."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<i4", "data": (int(ptr), False),
                                         "version": 2}


def _tensor(owner, ptr, shape):
    if 0 in shape:
        return torch.empty(shape, dtype=torch.int32, device="cuda")
    return torch.as_tensor(_DeviceArray(owner, ptr, shape), device="cuda")


def _records(owner, ptr, n, stride):
    """{dist2, index} records of closest / kNN results."""
    r = _tensor(owner, ptr, (n, stride, 2))
    return {"dist2": r[:, :, 0].view(torch.float32), "index": r[:, :, 1]}


def _tree(bvh):
    """The tree's arrays: boxes and children of the nodes, primitive order."""
    i = bvh.info()
    nodes = _tensor(bvh, i.d_nodes, (i.node_count, 8))
    return {"box": nodes[:, :6].view(torch.float32), "children": nodes[:, 6:],
            "prims": _tensor(bvh, i.d_prim_ids, (i.prim_count,))}


def _prepare_probe(s, case, items, seed):
    """A tree with 4-wide nodes is built or refitted to be queried: a few thousand points
    follow, and show those nodes' contents (their number varies with the scene)."""
    if case["wide"]:
        s["points"] = A.PointBuffer(_queries({**case, "queries": PROBES}, items, seed), 1)
        ptr = ctypes.c_void_p()
        A.check(A.lib().qr_points_device_ptrs(s["points"].h, None, ctypes.byref(ptr)))
        s["out"] = _records(s["points"], ptr.value, PROBES, 1)


def _tree_and_probe(s, bvh):
    if not s["case"]["wide"]:
        return _tree(bvh)
    s["points"].closest(bvh, A.ORDER_MORTON, True)
    return {**_tree(bvh), **s["out"]}


PROBES = 2048


def prepare(case, seed):
    op = case["op"]
    s = {"case": case}
    if op == "grad":
        return _prepare_grad(s, case, seed)
    if op == "batch":
        items, s["poff"], s["points"], s["qoff"] = _batch(case, seed)
        s["items"] = torch.from_numpy(items).cuda()
        if case["mode"] == "query":
            s["batch"] = A.Batch.from_device(A.PRIM_TRI, s["items"].data_ptr(), s["poff"])
            # the configuration that tuning picks on the batched benchmark
            s["plan"] = A.BatchPlan(s["batch"], s["points"], s["qoff"], case["k"], tune=BATCH_CONFIG[case["k"] > 1])
        return s
    items = _items(case, seed)
    kind = KIND[case["scene"]]
    if "radius" in case:
        s["radius"] = case["radius"] * float(_radius_scale(seed))
    if op == "host":
        if kind == A.PRIM_TRI:
            s["scene"] = quarry.Scene(items.reshape(-1, 3, 3), builder=case["builder"])
        elif kind == A.PRIM_POINT:
            s["scene"] = quarry.PointCloud(items, builder=case["builder"])
        else:
            s["scene"] = quarry.GaussianCloud(items[:, :3], items[:, 3:7], items[:, 7:], builder=case["builder"])
        if case["wide"]:
            s["scene"].build_wide()
        if case["query"] == "raycast":
            r = _rays(case, items, seed)
            s["origins"], s["dirs"] = np.ascontiguousarray(r[:, :3]), np.ascontiguousarray(r[:, 3:6])
        else:
            s["points"] = _queries(case, items, seed)
        return s
    if op == "build":
        s["items"] = torch.from_numpy(items).cuda()
        _prepare_probe(s, case, items, seed)
        return s
    s["bvh"] = A.Bvh(kind, items, BUILDER[case["builder"]])
    if case["wide"]:
        s["bvh"].build_wide()
    if op == "refit":
        rng = np.random.default_rng([seed, 31])
        frames, dirty = [items], None
        moved = items.copy()
        if case["mode"] == "dirty":
            dirty = np.sort(rng.choice(items.shape[0], max(1, round(case["frac"] * items.shape[0])), replace=False))
            moved[dirty] += rng.normal(0.0, 0.05, (dirty.size, items.shape[1])).astype(np.float32)
            s["dirty"] = dirty.astype(np.int32)
        else:
            moved += rng.normal(0.0, 0.05, items.shape).astype(np.float32)
        frames.append(moved)
        s["frames"] = frames if case["mode"] == "dirty" else [torch.from_numpy(f).cuda() for f in frames]
        s["frame"] = 0
        _prepare_probe(s, case, items, seed)
        return s
    if op == "rays":
        s["rays"] = A.RayBuffer(_rays(case, items, seed))
        ptr = ctypes.c_void_p()
        A.check(A.lib().qr_rays_device_ptrs(s["rays"].h, None, ctypes.byref(ptr), None))
        r = _tensor(s["rays"], ptr.value, (case["queries"], 2))
        s["out"] = {"t": r[:, 0].view(torch.float32), "hit": r[:, 1]}
        return s
    stride = max(1, case.get("k", 0))
    s["points"] = A.PointBuffer(_queries(case, items, seed), stride)
    if op != "radius":
        ptr = ctypes.c_void_p()
        A.check(A.lib().qr_points_device_ptrs(s["points"].h, None, ctypes.byref(ptr)))
        s["out"] = _records(s["points"], ptr.value, case["queries"], stride)
    return s


# (variant, Morton order of the queries) of the batched plans: closest, kNN
BATCH_CONFIG = {False: (A.BATCH_VARIANTS.index("wide_lds64"), False),
                True: (A.BATCH_VARIANTS.index("wide_lds64"), True)}


def _grad_inputs(case, seed):
    """Leaf tensors of the differentiable call, the faces (meshes) and the upstream gradient."""
    rng = np.random.default_rng([seed, 32])
    n = case["queries"]
    up = rng.uniform(0.5, 1.5, n).astype(np.float32)
    if case["fn"] == "mesh":
        v, f = _mesh(case, seed)
        return [rng.uniform(-15, 15, (n, 3)).astype(np.float32), v], f, up
    if case["fn"] == "rays":
        v, f = _mesh(case, seed)
        r = S.sphere_rays(n, seed=seed + 14)
        return [np.ascontiguousarray(r[:, :3]), np.ascontiguousarray(r[:, 3:6]), v], f, up
    items = _items(case, seed)
    q = rng.uniform(0.0, 64.0, (n, 3)).astype(np.float32)
    if case["fn"] == "points":
        return [q, items], None, up
    return [q] + [np.ascontiguousarray(items[:, a:b]) for a, b in ((0, 3), (3, 7), (7, 10))], None, up


def _prepare_grad(s, case, seed):
    leaves, faces, up = _grad_inputs(case, seed)
    s["leaves"] = [torch.from_numpy(x).cuda().requires_grad_() for x in leaves]
    s["faces"] = None if faces is None else torch.from_numpy(faces).cuda()
    s["up"] = torch.from_numpy(up).cuda()
    return s


# ---- one pass -------------------------------------------------------------------------


class _Csr:
    """A radius result kept on the device."""

    def __init__(self):
        self.h = ctypes.c_void_p()

    def __del__(self):
        if self.h.value:
            A.lib().qr_radius_destroy(self.h)


def _run_radius(s):
    c = s["case"]
    csr, ms = _Csr(), ctypes.c_double()
    A.check(A.lib().qr_radius(s["bvh"].h, s["points"].h, s["radius"], 0, ORDER[c["order"]], int(c["wide"]),
                              ctypes.byref(csr.h), ctypes.byref(ms)))
    n, total = ctypes.c_int(), ctypes.c_int()
    A.check(A.lib().qr_radius_info(csr.h, ctypes.byref(n), ctypes.byref(total)))
    offs, keys = ctypes.c_void_p(), ctypes.c_void_p()
    A.check(A.lib().qr_radius_device_ptrs(csr.h, ctypes.byref(offs), ctypes.byref(keys)))
    k = _tensor(csr, keys.value, (total.value, 2))
    return {"offsets": _tensor(csr, offs.value, (n.value + 1,)), "dist2": k[:, 1].view(torch.float32), "index": k[:, 0]}


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "host":
        if c["query"] == "closest":
            return s["scene"].closest(s["points"], order=c["order"], wide=c["wide"])
        if c["query"] == "knn":
            return s["scene"].knn(s["points"], c["k"], order=c["order"], wide=c["wide"])
        if c["query"] == "radius":
            return s["scene"].radius(s["points"], s["radius"], order=c["order"], wide=c["wide"])
        return s["scene"].raycast(s["origins"], s["dirs"], order=c["order"], wide=c["wide"])
    if op == "closest":
        s["points"].closest(s["bvh"], ORDER[c["order"]], c["wide"])
        return s["out"]
    if op == "knn":
        s["points"].knn(s["bvh"], c["k"], ORDER[c["order"]], c["wide"])
        return s["out"]
    if op == "radius":
        return _run_radius(s)
    if op == "rays":
        s["rays"].cast(s["bvh"], ORDER[c["order"]], c["wide"])
        return s["out"]
    if op == "build":
        bvh = A.Bvh.from_device(KIND[c["scene"]], s["items"].data_ptr(), s["items"].shape[0], BUILDER[c["builder"]])
        if c["wide"]:
            bvh.build_wide()
        return _tree_and_probe(s, bvh)
    if op == "refit":
        s["frame"] ^= 1
        f = s["frames"][s["frame"]]
        if c["mode"] == "dirty":
            s["bvh"].refit(f, s["dirty"])
        else:
            s["bvh"].refit_device(f.data_ptr(), f.shape[0])
        return _tree_and_probe(s, s["bvh"])
    if op == "grad":
        x = s["leaves"]
        if c["fn"] == "mesh":
            value, index = G.closest_point_dist2(x[0], x[1], s["faces"], builder=c["builder"])
        elif c["fn"] == "rays":
            value, index = G.ray_hit_t(x[0], x[1], x[2], s["faces"], builder=c["builder"])
        elif c["fn"] == "points":
            value, index = G.point_closest_dist2(x[0], x[1])
        else:
            value, index = G.gaussian_closest_dist2(x[0], x[1], x[2], x[3])
        grads = torch.autograd.grad(value, x, s["up"])
        return {"value": value.detach(), "index": index, "grads": list(grads)}
    if c["mode"] == "step":
        batch = A.Batch.from_device(A.PRIM_TRI, s["items"].data_ptr(), s["poff"])
        plan = A.BatchPlan(batch, s["points"], s["qoff"], c["k"], tune=BATCH_CONFIG[c["k"] > 1])
    else:
        plan = s["plan"]
    plan.run()
    r = plan.read()
    return {"dist2": r[:, :, 0].view(np.float32), "index": r[:, :, 1].view(np.int32)}


# ---- floors and tolerances -----------------------------------------------------------


def _walk(prims, kind, k):
    """Bytes and operations of one query's shortest walk: a root-to-leaf path of 4-wide
    nodes and k leaves."""
    depth = max(1.0, math.log(max(prims, 2), 4))
    return depth * 128 + k * (ITEM_BYTES[kind] + 4), depth * 4 * BOX_OPS + k * LEAF_OPS[kind]


def _tree_bytes(prims, kind):
    return prims * (ITEM_BYTES[kind] + 4) + (2 * prims - 1) * 32


def work(case):
    op = case["op"]
    if op == "batch":
        # expected primitives and queries of the log-uniform ranges
        n = case["scenes"] * (case["nmax"] - 256) / math.log(case["nmax"] / 256)
        q = case["scenes"] * (case["qmax"] / 2 - 32) / math.log(case["qmax"] / 64)
        k = max(1, case["k"])
        b, f = _walk(n / case["scenes"], A.PRIM_TRI, k)
        tree = _tree_bytes(n, A.PRIM_TRI)
        out = {"bytes": q * (12 + 8 * k) + min(q * b, tree), "flops": q * f}
        if case["mode"] == "step":
            out["bytes"] += n * 36 + tree + q * 8 * k
            out["flops"] += n * 60
        return out
    n, kind = case["prims"], KIND[case["scene"]]
    tree = _tree_bytes(n, kind)
    if op == "build":
        # items in, tree out, and the 4-wide nodes (about one per two primitives)
        return {"bytes": n * ITEM_BYTES[kind] + tree + (n // 2) * 128 * bool(case["wide"]),
                "flops": n * (60 if case["builder"] == "lbvh" else 60 + 40 * math.log2(max(n, 2)))}
    if op == "refit":
        m = n if case["mode"] == "full" else max(1, round(case["frac"] * n))
        path = min(2 * n, m * max(1.0, math.log2(n / m) + 1))
        return {"bytes": m * 2 * (ITEM_BYTES[kind] + 4) + path * 56 + (path / 2) * 56 * bool(case["wide"]),
                "flops": path * 12}
    q = case["queries"]
    if op == "grad":
        b, f = _walk(n, kind, 1)
        leaf = ITEM_BYTES[kind]
        bytes_ = n * leaf + tree + q * (12 + 8 + 4) + min(q * b, tree) + q * (2 * 12 + 8 + leaf) + n * leaf
        return {"bytes": bytes_, "flops": n * 60 + q * (f + 3 * LEAF_OPS[kind])}
    k = max(1, case.get("k", 0))
    if op == "radius" or case.get("query") == "radius":
        k = 8
    ray = op == "rays" or case.get("query") == "raycast"
    b, f = _walk(n, kind, k)
    return {"bytes": q * ((32 + 8) if ray else (12 + 8 * k)) + min(q * b, tree), "flops": q * f}


def tolerance(case):
    """Distances, hits, indices and trees are the same bits whatever the walk, by the
    library's definition (single precision in a stated operation order).  Gradients
    add up per primitive in any order in 32 bits."""
    if case["op"] == "grad":
        return {"rel": 2e-5, "max": 1e-3}
    return "exact"


# ---- the same in 64 bits --------------------------------------------------------------


def _morton(x):
    lo, hi = x.amin(0), x.amax(0)
    c = ((x - lo) / (hi - lo).clamp_min(1e-30) * 1023.0).long().clamp(0, 1023)
    code = torch.zeros(x.shape[0], dtype=torch.int64, device=x.device)
    for bit in range(10):
        for a in range(3):
            code |= ((c[:, a] >> bit) & 1) << (3 * bit + a)
    return torch.argsort(code)


def _axes64(rot):
    x, y, z, w = (rot / rot.norm(dim=-1, keepdim=True)).unbind(-1)
    return torch.stack([torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)], -1),
                        torch.stack([2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)], -1),
                        torch.stack([2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], -1)], -2)


def _boxes64(kind, items):
    if kind == A.PRIM_TRI:
        t = items.view(-1, 3, 3)
        return t.amin(1), t.amax(1)
    if kind == A.PRIM_POINT:
        return items, items
    h = (_axes64(items[:, 3:7]) * items[:, None, 7:10]).square().sum(-1).sqrt()
    return items[:, :3] - h, items[:, :3] + h


def _bary64(p, t):
    """Barycentric weights (of a, b, c) of the point of triangles t (..., 3, 3) nearest p (..., 3)."""
    a, b, c = t.unbind(-2)
    ab, ac, ap = b - a, c - a, p - a
    aa, bb, cc = (ab * ab).sum(-1), (ac * ac).sum(-1), (ab * ac).sum(-1)
    e, f = (ap * ab).sum(-1), (ap * ac).sum(-1)
    det = aa * bb - cc * cc
    v, w = (bb * e - cc * f) / det, (aa * f - cc * e) / det
    inside = (v >= 0) & (w >= 0) & (v + w <= 1)
    best = torch.where(inside, torch.zeros_like(v), torch.full_like(v, math.inf))
    one, zero = torch.ones_like(v), torch.zeros_like(v)
    wt = torch.stack([1 - v - w, v, w], -1)
    for i, j in ((0, 1), (0, 2), (1, 2)):
        d = t[..., j, :] - t[..., i, :]
        s = (((p - t[..., i, :]) * d).sum(-1) / (d * d).sum(-1).clamp_min(1e-300)).clamp(0, 1)
        r = p - t[..., i, :] - s[..., None] * d
        d2 = (r * r).sum(-1)
        parts = [zero, zero, zero]
        parts[i], parts[j] = one - s, s
        nearer = d2 < best
        wt = torch.where(nearer[..., None], torch.stack(parts, -1), wt)
        best = torch.where(nearer, d2, best)
    return wt


def _ellipsoid64(p, g):
    """The point of the solid ellipsoids g nearest p, as unit coordinates u (p = m + R (s u)); p itself inside."""
    s = g[..., 7:10]
    y = ((p - g[..., :3])[..., None, :] @ _axes64(g[..., 3:7])).squeeze(-2)
    inside = (y / s).square().sum(-1) <= 1
    lo = torch.zeros_like(y[..., 0])
    hi = s.amax(-1) * y.norm(dim=-1) * 2 + 1e-12
    for _ in range(64):
        t = 0.5 * (lo + hi)
        out = (s * y / (t[..., None] + s * s)).square().sum(-1) > 1
        lo, hi = torch.where(out, t, lo), torch.where(out, hi, t)
    u = torch.where(inside[..., None], y / s, s * y / (0.5 * (lo + hi)[..., None] + s * s))
    return u, inside


def _dist64(kind, p, items):
    """Squared distances of points p (..., 3) and primitives (..., F)."""
    if kind == A.PRIM_POINT:
        return (p - items).square().sum(-1)
    if kind == A.PRIM_TRI:
        t = items.unflatten(-1, (3, 3))
        return (p - (_bary64(p, t)[..., None] * t).sum(-2)).square().sum(-1)
    u, inside = _ellipsoid64(p, items)
    c = items[..., :3] + (_axes64(items[..., 3:7]) @ (items[..., 7:10] * u)[..., None]).squeeze(-1)
    return torch.where(inside, torch.zeros_like(u[..., 0]), (p - c).square().sum(-1))


def _nearest64(kind, items, q, k):
    """The k nearest primitives of each point: squared distances (n, k) ascending and indices.

    Primitives and queries go in groups of 64 along a Morton curve; a group of
    primitives is tested where its box may hold one of the k nearest."""
    order = _morton(_boxes64(kind, items)[0])
    m = -(-items.shape[0] // 64)
    slot = torch.arange(m * 64, device=items.device).clamp_max(items.shape[0] - 1)
    real = (torch.arange(m * 64, device=items.device) < items.shape[0]).view(m, 64)
    ids = order[slot].view(m, 64)
    lo, hi = _boxes64(kind, items[ids.view(-1)])
    lo, hi = lo.view(m, 64, 3).amin(1), hi.view(m, 64, 3).amax(1)
    counts = real.sum(1)
    d2 = torch.empty((q.shape[0], k), dtype=torch.float64, device=q.device)
    index = torch.empty((q.shape[0], k), dtype=torch.int64, device=q.device)
    step = 2048 if kind == A.PRIM_GAUSS else 16384
    for rows in _morton(q).split(64):
        p = q[rows]
        plo, phi = p.amin(0), p.amax(0)
        near = torch.maximum(lo - phi, plo - hi).clamp_min(0.0).square().sum(-1)
        far = torch.maximum(phi - lo, hi - plo).square().sum(-1)
        bound = far[counts >= k].amin() if bool((counts >= k).any()) else far.amax()
        c = torch.nonzero(near <= bound).squeeze(1)
        # again for each point alone
        near = torch.maximum(lo[c] - p[:, None], p[:, None] - hi[c]).clamp_min(0.0).square().sum(-1)
        far = torch.maximum((p[:, None] - lo[c]).abs(), (hi[c] - p[:, None]).abs()).square().sum(-1)
        enough = counts[c] >= k
        bound = far[:, enough].amin(1, keepdim=True) if bool(enough.any()) else far.amax(1, keepdim=True)
        c = c[(near <= bound).any(0)]
        cand = ids[c][real[c]]
        best, at = None, None
        for part in cand.split(step):
            d = _dist64(kind, p[:, None, :], items[part][None])
            i = part.expand(d.shape)
            if best is not None:
                d, i = torch.cat([best, d], 1), torch.cat([at, i], 1)
            best, sel = d.topk(min(k, d.shape[1]), 1, largest=False)
            at = i.gather(1, sel)
        d2[rows], index[rows] = best, at
    return d2, index


def _exact_grad(case, seed):
    if case["fn"] == "rays":
        return None  # needs the hit triangle, which 64 bits may see on the other side of an edge
    leaves, faces, up = _grad_inputs(case, seed)
    x = [torch.from_numpy(v).cuda().double().requires_grad_() for v in leaves]
    q, up = x[0], torch.from_numpy(up).cuda().double()
    if case["fn"] == "mesh":
        tri = x[1][torch.from_numpy(faces).cuda().long()]
        kind, items = A.PRIM_TRI, tri.detach().reshape(-1, 9)
    elif case["fn"] == "points":
        kind, items = A.PRIM_POINT, x[1].detach()
    else:
        g = torch.cat(x[1:], 1)
        kind, items = A.PRIM_GAUSS, g.detach()
    at = _nearest64(kind, items, q.detach(), 1)[1][:, 0]
    # the nearest point in its primitive's own coordinates: these are at a minimum, so
    # the gradient with them held is the whole gradient
    if kind == A.PRIM_TRI:
        near = (_bary64(q.detach(), tri.detach()[at])[..., None] * tri[at]).sum(1)
        value = (q - near).square().sum(-1)
    elif kind == A.PRIM_POINT:
        value = (q - x[1][at]).square().sum(-1)
    else:
        u, inside = _ellipsoid64(q.detach(), items[at])
        near = g[at, :3] + (_axes64(g[at, 3:7]) @ (g[at, 7:10] * u)[..., None]).squeeze(-1)
        value = torch.where(inside, torch.zeros_like(up), (q - near).square().sum(-1))
    return {"value": value.detach(), "index": None, "grads": list(torch.autograd.grad(value, x, up))}


def exact(case, seed):
    """Distances and their gradients; indices may tie, so they have no such value.  None
    for trees (boxes are minima of inputs, the rest whole numbers), rays (64 bits may
    see a hit on the other side of an edge) and radius results (a hit at the radius
    itself changes the segments' lengths)."""
    op = case["op"]
    if op == "grad":
        return _exact_grad(case, seed)
    if op == "batch":
        items, poff, pts, qoff = _batch(case, seed)
        k = max(1, case["k"])
        items, pts = torch.from_numpy(items).cuda().double(), torch.from_numpy(pts).cuda().double()
        parts = [_nearest64(A.PRIM_TRI, items[poff[i]:poff[i + 1]], pts[qoff[i]:qoff[i + 1]], k)[0]
                 for i in range(case["scenes"]) if qoff[i + 1] > qoff[i]]
        return {"dist2": torch.cat(parts), "index": None}
    query = case.get("query", op)
    if query not in ("closest", "knn"):
        return None
    host = _items(case, seed)
    items = torch.from_numpy(host).cuda().double()
    q = torch.from_numpy(_queries(case, host, seed)).cuda().double()
    d2 = _nearest64(KIND[case["scene"]], items, q, max(1, case["k"]))[0]
    if op == "host":
        return (d2[:, 0] if query == "closest" else d2), None
    return {"dist2": d2, "index": None}
