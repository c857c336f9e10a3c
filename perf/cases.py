"""Performance cases: what programs built on blazert_amd ask of it, through its Python entry points.

A case is a dict of plain values; its "kind" says which call it makes:

* ``one``      intersect1, one ray in host memory (the drop-in call of blazeRT's scene API);
* ``trace``    Scene.intersect over device-resident rays: camera, incoherent or shadow rays; FP64, split precision or
               Scene<float>; closest or any hit; with or without normals; rays as three columns or as an (n, 3) tensor;
* ``batch``    Batch: many scenes of uneven size, captured once and replayed;
* ``mirror``   mirror_trace_autograd and its backward: one step of an inverse-rendering loop;
* ``rebuild``  a frame of a deforming mesh: a new Scene, add_mesh, commit on the device, trace;
* ``closest``  Scene.closest_surface over a point cloud.

``listed()`` holds the cases that are always measured, ``draw(rng)`` more of the same ranges. ``prepare(case, seed)``
makes inputs and the committed scene, ``run(state)`` is one call, ``exact(case, seed)`` its 64-bit brute force where
that is affordable, ``work(case)`` the bytes and operations it cannot do without.
"""
from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

import blazert_amd as B
from blazert_amd import workloads as W
from blazert_amd.mirror import mirror_trace_autograd

SPLIT = B.PRECISION_FP32_TRAV_FP64_HIT
FP64 = B.PRECISION_FP64
DEVICE_BUILD_FROM = 20_000  # primitives from which the programs here build their trees on the device
BRUTE_FORCE_PAIRS = 4e9     # ray-primitive pairs up to which `exact` tests every pair


# ---------------------------------------------------------------------------------------------------- cases
def listed() -> list:
    return [
        # A renderer written against blazeRT's API calls intersect1 per ray: the latency of one such call.
        {"name": "one_ray_mesh5k", "kind": "one", "scene": "icosphere", "level": 4, "dtype": "f64", "any_hit": False},
        # The small configuration of the library: 1,024 spheres under a 512x512 pinhole camera, with normals for
        # shading. A launch of tens of microseconds, so everything around the traversal counts.
        {"name": "spheres1k_camera512", "kind": "trace", "scene": "spheres", "spheres": 1024, "rays": "camera",
         "width": 512, "height": 512, "dtype": "f64", "precision": "fp64", "any_hit": False, "normals": True,
         "form": "columns"},
        # The headline: a 1.31M-triangle displaced icosphere and 4,194,304 incoherent rays, as the drop-in in FP64 ...
        {"name": "mesh1310k_incoherent4m_fp64", "kind": "trace", "scene": "icosphere", "level": 8,
         "rays": "incoherent", "n": 4194304, "dtype": "f64", "precision": "fp64", "any_hit": False, "normals": False,
         "form": "columns"},
        # ... and in split precision (FP32 traversal, FP64 hit).
        {"name": "mesh1310k_incoherent4m_split", "kind": "trace", "scene": "icosphere", "level": 8,
         "rays": "incoherent", "n": 4194304, "dtype": "f64", "precision": "split", "any_hit": False, "normals": False,
         "form": "columns"},
        # Primary rays of a full-HD frame on the same mesh, with normals, from an (n, 3) tensor as a torch program
        # holds them.
        {"name": "mesh1310k_camera1080p_fp64", "kind": "trace", "scene": "icosphere", "level": 8, "rays": "camera",
         "width": 1920, "height": 1080, "dtype": "f64", "precision": "fp64", "any_hit": False, "normals": True,
         "form": "rows"},
        # Shadow rays: any hit between a surface point and a light, per-ray tmin / tmax, an odd number of them on a
        # mid-size mesh.
        {"name": "mesh100k_shadow500k_any", "kind": "trace", "scene": "torus", "triangles": 100000, "rays": "shadow",
         "n": 500009, "dtype": "f64", "precision": "split", "any_hit": True, "normals": False, "form": "rows"},
        # All four geometry types in one scene, 8,388,608 incoherent rays.
        {"name": "mixed260k_incoherent8m_fp64", "kind": "trace", "scene": "mixed", "triangles": 200000,
         "spheres": 50000, "cylinders": 10000, "planes": 100, "rays": "incoherent", "n": 8388608, "dtype": "f64",
         "precision": "fp64", "any_hit": False, "normals": False, "form": "columns"},
        # Scene<float>: FP32 geometry, traversal and hits; a ragged number of rays.
        {"name": "mesh328k_incoherent1m_f32", "kind": "trace", "scene": "icosphere", "level": 7, "rays": "incoherent",
         "n": 1000003, "dtype": "f32", "precision": "fp64", "any_hit": False, "normals": True, "form": "columns"},
        # 12 scenes of 1k-500k triangles with 16k-2M rays each, traced together from a captured graph.
        {"name": "batch12_uneven_split", "kind": "batch", "scenes": 12, "mix": 41, "tri_lo": 1000, "tri_hi": 500000,
         "ray_lo": 16384, "ray_hi": 2097152, "precision": "split"},
        # Inverse rendering: three mirror bounces of 4,194,304 rays inside a box, forward and backward.
        {"name": "mirror3_mesh1310k_4m", "kind": "mirror", "level": 8, "n": 4194304, "bounces": 3},
        # A deforming mesh is rebuilt every frame and then rendered in split precision.
        {"name": "rebuild1310k_camera1080p", "kind": "rebuild", "level": 8, "width": 1920, "height": 1080,
         "precision": "split"},
        # Distance field samples: the closest surface of 1,048,576 points.
        {"name": "closest_mesh1310k_1m", "kind": "closest", "scene": "icosphere", "level": 8, "n": 1048576},
    ]


def _log_int(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["one", "trace", "trace", "trace", "trace", "trace", "batch", "mirror", "rebuild", "closest"])
    if kind == "one":
        return {"kind": "one", "scene": "icosphere", "level": rng.randint(1, 8), "dtype": rng.choice(["f64", "f32"]),
                "any_hit": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": "batch", "scenes": rng.randint(2, 12), "mix": rng.randint(0, 1 << 20), "tri_lo": 200,
                "tri_hi": _log_int(rng, 2000, 500000), "ray_lo": 1000, "ray_hi": _log_int(rng, 5000, 1000000),
                "precision": rng.choice(["fp64", "split"])}
    if kind == "mirror":
        return {"kind": "mirror", "level": rng.randint(3, 8), "n": _log_int(rng, 1000, 4000000),
                "bounces": rng.randint(1, 3)}
    if kind == "rebuild":
        return {"kind": "rebuild", "level": rng.randint(4, 8), "width": _log_int(rng, 64, 1920),
                "height": _log_int(rng, 64, 1080), "precision": rng.choice(["fp64", "split"])}
    if kind == "closest":
        if rng.random() < 0.3:
            return {"kind": "closest", "scene": "spheres", "spheres": _log_int(rng, 100, 100000),
                    "n": _log_int(rng, 100, 1000000)}
        return {"kind": "closest", "scene": "icosphere", "level": rng.randint(3, 8), "n": _log_int(rng, 100, 1000000)}
    c = {"kind": "trace"}
    scene = rng.choice(["icosphere", "icosphere", "torus", "spheres", "mixed"])
    c["scene"] = scene
    if scene == "icosphere":
        c["level"] = rng.randint(2, 8)
    elif scene == "torus":
        c["triangles"] = _log_int(rng, 100, 500000)
    elif scene == "spheres":
        c["spheres"] = _log_int(rng, 10, 100000)
    else:
        c.update(triangles=_log_int(rng, 5200, 200000), spheres=_log_int(rng, 100, 50000),
                 cylinders=_log_int(rng, 20, 10000), planes=_log_int(rng, 1, 100))
    kinds = ["camera", "incoherent", "incoherent"] + (["shadow"] if scene == "torus" else [])
    c["rays"] = rng.choice(kinds)
    if c["rays"] == "camera":
        c["width"], c["height"] = _log_int(rng, 16, 1920), _log_int(rng, 16, 1080)
    else:
        c["n"] = _log_int(rng, 64, 2000000)
    c["dtype"] = "f32" if rng.random() < 0.2 else "f64"
    c["precision"] = "fp64" if c["dtype"] == "f32" else rng.choice(["fp64", "split"])
    c["any_hit"] = c["rays"] == "shadow"
    c["normals"] = not c["any_hit"] and rng.random() < 0.5
    c["form"] = rng.choice(["columns", "rows"])
    return c


# ---------------------------------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _unit_icosphere(level: int):
    return W.icosphere(level, displacement=0.0)


def _icosphere(level: int, seed: int):
    """Displaced icosphere: every vertex scaled radially by 1 + 0.05 N(0, 1)."""
    v, f = _unit_icosphere(level)
    g = np.random.default_rng([seed, 1]).standard_normal(len(v))
    return v * (1.0 + 0.05 * g)[:, None], f


def _geometry(case: dict, seed: int) -> dict:
    """Host arrays of the case's scene, by geometry type."""
    kind = case["scene"]
    if kind == "icosphere":
        return {"mesh": _icosphere(case["level"], seed)}
    if kind == "torus":
        return {"mesh": W.torus(case["triangles"], seed=seed)}
    if kind == "spheres":
        return {"spheres": W.sphere_field(case["spheres"], seed=seed)}
    return W.mixed_scene(case["triangles"], case["spheres"], case["cylinders"], case["planes"], seed=seed)


def _add(scene, geo: dict) -> int:
    """Adds every geometry of `geo` to the scene; returns the number of primitives."""
    n = 0
    for key, add in (("mesh", scene.add_mesh), ("spheres", scene.add_spheres), ("cylinders", scene.add_cylinders),
                     ("planes", scene.add_planes)):
        if key in geo:
            add(*geo[key])
            n += len(geo[key][1])
    return n


def _scene(geo: dict, dtype: str = "f64"):
    s = B.Scene(dtype=np.float32 if dtype == "f32" else np.float64)
    n = _add(s, geo)
    if dtype == "f64" and n >= DEVICE_BUILD_FROM:
        s.commit(device=True)
    else:
        s.commit()
        s.upload()
    return s


def _generator(seed: int, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(seed * 7919 + 13)
    return g


def _directions(n: int, g, dev):
    """Directions uniform on the sphere, (n, 3)."""
    z = torch.rand(n, generator=g, device=dev, dtype=torch.float64) * 2 - 1
    phi = torch.rand(n, generator=g, device=dev, dtype=torch.float64) * (2 * math.pi)
    s = torch.sqrt(torch.clamp(1 - z * z, min=0))
    return torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], dim=1)


def _incoherent(n: int, half: float, g, dev):
    o = (torch.rand((n, 3), generator=g, device=dev, dtype=torch.float64) * 2 - 1) * half
    return o, _directions(n, g, dev)


def _camera(width: int, height: int, distance: float, g, dev):
    """Pinhole rays through pixel centres (45 degrees vertical) from `distance` along a random axis."""
    eye = _directions(1, g, dev)[0]
    look = -eye
    up = torch.tensor([0.0, 1.0, 0.0] if abs(float(eye[1])) < 0.9 else [0.0, 0.0, 1.0], dtype=torch.float64,
                      device=dev)
    right = torch.linalg.cross(look, up)
    right = right / torch.linalg.norm(right)
    up = torch.linalg.cross(right, look)
    th = math.tan(math.radians(22.5))
    x = ((torch.arange(width, device=dev, dtype=torch.float64) + 0.5) / width * 2 - 1) * (th * width / height)
    y = ((torch.arange(height, device=dev, dtype=torch.float64) + 0.5) / height * 2 - 1) * th
    d = look + x[None, :, None] * right + y[:, None, None] * up
    d = (d / torch.linalg.norm(d, dim=2, keepdim=True)).reshape(-1, 3)
    o = (eye * distance).expand(len(d), 3)
    return o.contiguous(), d


def _shadow(geo: dict, n: int, g, dev):
    """From random surface points to points of a square light above the mesh; tmin / tmax keep both ends out."""
    v, f = geo["mesh"]
    V = torch.from_numpy(v).to(dev)
    F = torch.from_numpy(f.astype(np.int64)).to(dev)
    tri = F[torch.randint(len(f), (n,), generator=g, device=dev)]
    a = torch.rand((n, 2), generator=g, device=dev, dtype=torch.float64)
    a = torch.where((a.sum(1) > 1)[:, None], 1 - a, a)
    p = V[tri[:, 0]] * (1 - a.sum(1))[:, None] + V[tri[:, 1]] * a[:, :1] + V[tri[:, 2]] * a[:, 1:]
    light = torch.rand((n, 3), generator=g, device=dev, dtype=torch.float64) - 0.5
    light[:, 2] = 4.0
    d = light - p
    dist = torch.linalg.norm(d, dim=1)
    return p, d / dist[:, None], torch.full_like(dist, 1e-6), dist * (1 - 1e-6)


RAY_BOX = {"icosphere": 2.0, "torus": 1.5, "spheres": 11.0, "mixed": 22.0}
EYE = {"icosphere": 4.0, "torus": 4.0, "spheres": 30.0, "mixed": 60.0}


def _rays(case: dict, geo: dict, seed: int, dev):
    """(origins, directions, tmin, tmax) of a trace case in its scene type."""
    g = _generator(seed, dev)
    tmin = tmax = None
    if case["rays"] == "camera":
        o, d = _camera(case["width"], case["height"], EYE[case["scene"]], g, dev)
    elif case["rays"] == "shadow":
        o, d, tmin, tmax = _shadow(geo, case["n"], g, dev)
    else:
        o, d = _incoherent(case["n"], RAY_BOX[case["scene"]], g, dev)
    if case["dtype"] == "f32":
        o, d = o.float(), d.float()
        tmin, tmax = (None, None) if tmin is None else (tmin.float(), tmax.float())
    return o, d, tmin, tmax


def _columns(x):
    return tuple(x[:, k].contiguous() for k in range(3))


def _batch_sizes(case: dict):
    """(triangles, rays) of every scene of a batch, log-uniform; the same for every seed."""
    r = random.Random(case["mix"])
    return [(_log_int(r, case["tri_lo"], case["tri_hi"]), _log_int(r, case["ray_lo"], case["ray_hi"]))
            for _ in range(case["scenes"])]


def _batch_level(triangles: int) -> int:
    return max(1, int(round(math.log(max(triangles, 20) / 20.0, 4))))


def _precision(case: dict) -> int:
    return SPLIT if case["precision"] == "split" else FP64


def _one_ray(case: dict, seed: int):
    """A ray from outside towards a point inside the mesh, rounded to the scene type."""
    r = np.random.default_rng([seed, 2])
    o = r.standard_normal(3)
    o *= 3.0 / np.linalg.norm(o)
    d = r.uniform(-0.4, 0.4, 3) - o
    if case["dtype"] == "f32":
        o, d = o.astype(np.float32).astype(np.float64), d.astype(np.float32).astype(np.float64)
    return tuple(float(x) for x in o), tuple(float(x) for x in d)


def prepare(case: dict, seed: int) -> dict:
    dev = torch.device("cuda")
    kind = case["kind"]
    if kind == "one":
        o, d = _one_ray(case, seed)
        return {"case": case, "scene": _scene(_geometry(case, seed), case["dtype"]),
                "ray": B.Ray(o, d, any_hit=case["any_hit"])}
    if kind == "trace":
        geo = _geometry(case, seed)
        o, d, tmin, tmax = _rays(case, geo, seed, dev)
        if case["form"] == "columns":
            o, d = _columns(o), _columns(d)
        return {"case": case, "scene": _scene(geo, case["dtype"]), "o": o, "d": d, "tmin": tmin, "tmax": tmax}
    if kind == "batch":
        items = []
        g = _generator(seed, dev)
        for k, (tris, rays) in enumerate(_batch_sizes(case)):
            mesh = _icosphere(_batch_level(tris), seed + k) if k % 2 == 0 else W.torus(tris, seed=seed + k)
            o, d = _incoherent(rays, 1.5, g, dev)
            items.append((_scene({"mesh": mesh}), _columns(o), _columns(d)))
        batch = B.Batch(items, precision=_precision(case))
        batch.capture(torch.cuda.Stream())
        return {"case": case, "batch": batch}
    if kind == "mirror":
        sv, sf = _icosphere(case["level"], seed)
        bv, bf = W.box_mesh(3.0)
        v = np.concatenate([sv, bv])
        f = np.concatenate([sf, (bf + len(sv)).astype(np.uint32)])
        g = _generator(seed, dev)
        o, d = _incoherent(case["n"], 2.0, g, dev)
        nb = case["bounces"]
        return {"case": case, "scene": _scene({"mesh": (v, f)}), "v": torch.from_numpy(v).to(dev).requires_grad_(),
                "o": o.requires_grad_(), "d": d.requires_grad_(),
                "gt": torch.rand((nb, case["n"]), generator=g, device=dev, dtype=torch.float64),
                "gx": torch.rand((nb, case["n"], 3), generator=g, device=dev, dtype=torch.float64)}
    if kind == "rebuild":
        g = _generator(seed, dev)
        o, d = _camera(case["width"], case["height"], EYE["icosphere"], g, dev)
        v, f = _icosphere(case["level"], seed)
        return {"case": case, "v": np.ascontiguousarray(v), "f": f, "o": o, "d": d}
    geo = _geometry(case, seed)
    g = _generator(seed, dev)
    p = (torch.rand((case["n"], 3), generator=g, device=dev, dtype=torch.float64) * 2 - 1) * RAY_BOX[case["scene"]]
    return {"case": case, "scene": _scene(geo), "p": p}


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "one":
        hit = B.RayHit()
        ok = B.intersect1(state["scene"], state["ray"], hit)
        return {"hit": int(ok), "t": hit.hit_distance, "uv": list(hit.uv), "normal": list(hit.normal),
                "prim_id": hit.prim_id, "geom_id": hit.geom_id}
    if kind == "trace":
        return state["scene"].intersect(state["o"], state["d"], state["tmin"], state["tmax"],
                                        precision=_precision(case), any_hit=case["any_hit"], normals=case["normals"])
    if kind == "batch":
        state["batch"].replay()
        return state["batch"].hits
    if kind == "mirror":
        t, x, prim = mirror_trace_autograd(state["scene"], state["v"], state["o"], state["d"], case["bounces"])
        gv, go, gd = torch.autograd.grad([t, x], [state["v"], state["o"], state["d"]], [state["gt"], state["gx"]])
        return {"t": t.detach(), "x": x.detach(), "prim_id": prim, "gv": gv, "go": go, "gd": gd}
    if kind == "rebuild":
        s = B.Scene()
        s.add_mesh(state["v"], state["f"])
        s.commit(device=True)
        hits = s.intersect(state["o"], state["d"], precision=_precision(case))
        state["scene"] = s  # the frame's scene lives until the next one replaces it
        return hits
    return state["scene"].closest_surface(state["p"])


# ---------------------------------------------------------------------------------------------------- exact
def _brute_triangles(v, f, o, d, tmin, tmax):
    """Closest hit of every ray by testing every triangle (Moeller-Trumbore, float64): t, u, v, normal."""
    dev = o.device
    V = torch.from_numpy(np.asarray(v, np.float64)).to(dev)
    F = torch.from_numpy(np.asarray(f, np.int64)).to(dev)
    p0, e1, e2 = V[F[:, 0]], V[F[:, 1]] - V[F[:, 0]], V[F[:, 2]] - V[F[:, 0]]
    fn = torch.linalg.cross(e1, e2)
    fn = fn / torch.linalg.norm(fn, dim=1, keepdim=True)
    vn = torch.zeros_like(V)
    for k in range(3):
        vn.index_add_(0, F[:, k], fn / 3.0)
    big = torch.finfo(torch.float64).max
    n = len(o)
    T, U, Wv = torch.full((n,), big, dtype=torch.float64, device=dev), torch.zeros_like(o[:, 0]), \
        torch.zeros_like(o[:, 0])
    N = torch.zeros((3, n), dtype=torch.float64, device=dev)
    step = max(1, int(2e7 // len(f)))
    for a in range(0, n, step):
        oo, dd = o[a:a + step, None, :], d[a:a + step, None, :]
        pv = torch.linalg.cross(dd, e2[None])
        det = (pv * e1).sum(-1)
        s = oo - p0
        u = (s * pv).sum(-1) / det
        q = torch.linalg.cross(s, e1[None].expand_as(s))
        w = (q * dd).sum(-1) / det
        t = (q * e2).sum(-1) / det
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= tmin[a:a + step, None]) & (t < tmax[a:a + step, None])
        t = torch.where(ok, t, torch.full_like(t, float("inf")))
        tm, k = t.min(1)
        hit = torch.isfinite(tm)
        rows = torch.arange(len(k), device=dev)
        uu, ww = u[rows, k], w[rows, k]
        c = F[k]
        nn = (1 - uu - ww)[:, None] * vn[c[:, 0]] + uu[:, None] * vn[c[:, 1]] + ww[:, None] * vn[c[:, 2]]
        nn = nn / torch.linalg.norm(nn, dim=1, keepdim=True)
        z = torch.zeros_like(uu)
        T[a:a + step] = torch.where(hit, tm, torch.full_like(tm, big))
        U[a:a + step] = torch.where(hit, uu, z)
        Wv[a:a + step] = torch.where(hit, ww, z)
        N[:, a:a + step] = torch.where(hit[:, None], nn, torch.zeros_like(nn)).T
    return T, U, Wv, N


def _brute_spheres(c, r, o, d, tmin, tmax):
    dev = o.device
    C, R = torch.from_numpy(np.asarray(c, np.float64)).to(dev), torch.from_numpy(np.asarray(r, np.float64)).to(dev)
    big = torch.finfo(torch.float64).max
    n = len(o)
    T = torch.full((n,), big, dtype=torch.float64, device=dev)
    N = torch.zeros((3, n), dtype=torch.float64, device=dev)
    step = max(1, int(4e7 // len(r)))
    for a in range(0, n, step):
        oo, dd = o[a:a + step], d[a:a + step]
        oc = oo[:, None, :] - C
        b = (oc * dd[:, None, :]).sum(-1)
        w = oc - b[..., None] * dd[:, None, :]
        disc = R * R - (w * w).sum(-1)
        q = torch.sqrt(torch.clamp(disc, min=0))
        lo, hi = tmin[a:a + step, None], tmax[a:a + step, None]
        t0, t1 = -b - q, -b + q
        inf = torch.full_like(t0, float("inf"))
        t = torch.where((disc >= 0) & (t0 > lo) & (t0 < hi), t0,
                        torch.where((disc >= 0) & (t1 > lo) & (t1 < hi), t1, inf))
        tm, k = t.min(1)
        hit = torch.isfinite(tm)
        nn = oo + torch.where(hit, tm, torch.zeros_like(tm))[:, None] * dd - C[k]
        nn = nn / torch.linalg.norm(nn, dim=1, keepdim=True)
        T[a:a + step] = torch.where(hit, tm, torch.full_like(tm, big))
        N[:, a:a + step] = torch.where(hit[:, None], nn, torch.zeros_like(nn)).T
    return T, N


def _f32_geometry(geo: dict) -> dict:
    return {k: tuple(np.asarray(a).astype(np.float32).astype(np.float64) if np.asarray(a).dtype == np.float64
                     else a for a in v) for k, v in geo.items()}


def exact(case: dict, seed: int):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    kind = case["kind"]
    if kind not in ("one", "trace") or case["any_hit"] or case.get("scene") == "mixed":
        return None  # any hit and cylinders have no value but the order of the reference's traversal
    prims = case.get("spheres") or case.get("triangles") or 20 * 4 ** case.get("level", 0)
    n = 1 if kind == "one" else case.get("n", case.get("width", 0) * case.get("height", 0))
    if float(prims) * n > BRUTE_FORCE_PAIRS:
        return None
    geo = _geometry(case, seed)
    if case["dtype"] == "f32":
        geo = _f32_geometry(geo)
    if kind == "one":
        ro, rd = _one_ray(case, seed)
        o, d = (torch.tensor([x], dtype=torch.float64, device=dev) for x in (ro, rd))
    else:
        o, d, _, _ = _rays(case, geo, seed, dev)
        o, d = o.double(), d.double()
    d = d / torch.linalg.norm(d, dim=1, keepdim=True)
    tmin = torch.zeros(n, dtype=torch.float64, device=dev)
    tmax = torch.full_like(tmin, float("inf"))
    if "mesh" in geo:
        t, u, w, nrm = _brute_triangles(*geo["mesh"], o, d, tmin, tmax)
    else:
        t, nrm = _brute_spheres(*geo["spheres"], o, d, tmin, tmax)
        u = w = torch.zeros_like(t)
    if case["dtype"] == "f32":  # a miss is the scene type's largest value
        t = torch.where(t > 1e300, torch.full_like(t, float(np.finfo(np.float32).max)), t)
    if kind == "one":
        return {"hit": None, "t": float(t[0]), "uv": [float(u[0]), float(w[0])],
                "normal": [float(x) for x in nrm[:, 0]], "prim_id": None, "geom_id": None}
    out = {"t": t, "u": u, "v": w, "prim_id": None, "geom_id": None}
    if case["normals"]:
        out["normal"] = nrm
    return out


# ---------------------------------------------------------------------------------------------------- work
RECORD = {"triangles": 72 / 2 + 12, "spheres": 32, "cylinders": 120, "planes": 112}  # input bytes per primitive (FP64)
TEST = {"triangles": 45, "spheres": 35, "cylinders": 120, "planes": 45}                # operations per primitive test


def _primitives(case: dict) -> dict:
    if case.get("level") is not None:
        return {"triangles": 20 * 4 ** case["level"]}
    return {k: case[k] for k in RECORD if case.get(k)}


def _query(prims: dict, n: int, bytes_per: int, scale: float = 1.0) -> dict:
    """n queries of a scene: its geometry and every ray and result moved once; per query one root-to-leaf path of
    each tree (two boxes of 18 operations per level) and one leaf of four primitives."""
    ops = sum(2 * 18 * max(1.0, math.log2(max(2, m / 4))) + 4 * TEST[k] for k, m in prims.items())
    return {"bytes": scale * (sum(RECORD[k] * m for k, m in prims.items()) + bytes_per * n), "flops": ops * n}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "one":  # one ray needs one path of the tree, not the whole scene
        levels = math.log2(20 * 4 ** case["level"] / 4)
        return {"bytes": 104 + levels * 112 + 4 * 80, "flops": levels * 36 + 4 * 45}
    if kind == "trace":
        n = case.get("n", case.get("width", 0) * case.get("height", 0))
        per = 48 + 32 + (24 if case["normals"] else 0) + (16 if case["rays"] == "shadow" else 0)
        return _query(_primitives(case), n, per, 0.5 if case["dtype"] == "f32" else 1.0)
    if kind == "batch":
        parts = [_query({"triangles": t}, n, 80) for t, n in _batch_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "mirror":
        n, nb = case["n"], case["bounces"]
        tris = 20 * 4 ** case["level"] + 12
        # forward: rays in, hit and next ray out per bounce; backward: upstream and face ids in, ray gradients out
        q = _query({"triangles": tris}, n, 48 + nb * 60 + 48 + nb * 36 + 48)
        return {"bytes": q["bytes"] + 24 * (tris // 2 + 2), "flops": q["flops"] * nb + n * nb * 300}
    if kind == "rebuild":
        tris = 20 * 4 ** case["level"]
        q = _query({"triangles": tris}, case["width"] * case["height"], 80)
        # the build sorts the triangles into a tree: three axis bins per primitive and level, records written once
        return {"bytes": q["bytes"] + tris * (80 + 64 + 4 + 45), "flops": q["flops"] + tris * math.log2(tris) * 12}
    return _query(_primitives(case), case["n"], 24 + 16)
