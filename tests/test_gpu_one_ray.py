"""intersect1 (one ray, traced from host memory by one wave; rays the fast traversal refuses go to the exact kernel) gives
the bits of an in/out batch traced by the exact kernel, and what the triangles leave is what the later types merge into."""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Ray, RayHit, Scene, intersect1, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def rays(v, f, n, seed):
    """Incoherent rays, some through vertices, short, along an axis or not a number, with windows around their hits."""
    o, d = W.incoherent_rays(n, seed, 1.5)
    o, d = o.copy(), d.copy()
    r = np.random.default_rng(seed)
    to = v[f[r.integers(len(f), size=n), 0]] - o
    d[::4] = (to / np.linalg.norm(to, axis=1, keepdims=True))[::4]
    d[1::16] *= 0.5
    d[2::16] = [0.0, 0.0, -1.0]
    d[3::32, 1] = np.nan
    o[5::32, 2] = np.nan
    tmax = np.where(r.random(n) < 0.2, r.uniform(0.2, 3.0, n), 1e308)
    return o, d, np.where(r.random(n) < 0.2, 0.3, 0.0), tmax


def scene(v, f, leaf, rest):
    s = Scene(min_leaf_primitives=leaf)
    s.add_mesh(v, f)
    if rest:
        r = np.random.default_rng(1)
        s.add_spheres(r.uniform(-1.2, 1.2, (40, 3)), r.uniform(0.05, 0.3, 40))
    s.commit()
    return s


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("triangles,leaf,rest", [(1, 4, False), (3, 4, True), (1280, 4, False), (1280, 300, True),
                                                 (20480, 1, False)])
def test_bits_of_a_batch(dev, triangles, leaf, rest, any_hit):
    v, f = W.icosphere(5 if triangles > 1280 else 3)
    f = f[:triangles]
    s = scene(v, f, leaf, rest)
    o, d, tmin, tmax = rays(v, f, 320, triangles)
    col = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    n = len(o)
    h = {k: torch.full((n,), x, dtype=torch.float64, device=dev) for k, x in zip("tuv", (1.5, 0.25, 0.125))}
    h["prim_id"] = torch.full((n,), 7, dtype=torch.int32, device=dev)
    h["geom_id"] = torch.full((n,), 3, dtype=torch.int32, device=dev)
    h["normal"] = torch.full((3, n), 9.0, dtype=torch.float64, device=dev)
    s.intersect(tuple(col(o[:, k]) for k in range(3)), tuple(col(d[:, k]) for k in range(3)), col(tmin), col(tmax),
                hits=h, schedule=SCHEDULE_PER_THREAD, any_hit=any_hit)
    ref = {k: x.cpu().numpy() for k, x in h.items()}
    hits = 0
    for i in range(n):
        rh = RayHit(normal=[9.0] * 3, uv=[0.25, 0.125], hit_distance=1.5, prim_id=7, geom_id=3)
        got = intersect1(s, Ray(o[i], d[i], tmin[i], tmax[i], any_hit), rh)
        row = np.array([rh.hit_distance, *rh.uv, *rh.normal])
        want = np.array([ref["t"][i], ref["u"][i], ref["v"][i], *ref["normal"][:, i]])
        assert row.tobytes() == want.tobytes() and (rh.prim_id, rh.geom_id) == (ref["prim_id"][i], ref["geom_id"][i]), i
        assert got == (rh.geom_id != 3), i
        hits += got
    assert hits or triangles < 10


def test_threads_on_one_scene(dev):
    v, f = W.icosphere(3)
    s = scene(v, f, 4, True)
    o, d, tmin, tmax = rays(v, f, 64, 3)
    trace = lambda i: (lambda rh: (intersect1(s, Ray(o[i], d[i], tmin[i], tmax[i]), rh), rh.hit_distance, rh.prim_id))(
        RayHit())
    want = [trace(i) for i in range(64)]
    bad = []

    def work(k):
        for i in range(64):
            if trace((i * 7 + k) % 64) != want[(i * 7 + k) % 64]:
                bad.append((k, i))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
