"""The fast closest-hit traversal of spheres and cylinders (FP32 reference-order boxes; the leaf of a hit is checked
with the reference's own FP64 box tests) gives the bits of the exact FP64 kernel, which the one-ray-per-thread schedule
still runs: on overlapping, repeated, touching and tiny primitives, leaves of any size, launches around the wave sizes, rays
that graze, and rays outside its assumptions."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu
KEYS = ("t", "u", "v", "prim_id", "geom_id", "normal")
TYPES = ("spheres", "cylinders")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def rotations(n, r):
    q, _ = np.linalg.qr(r.standard_normal((n, 3, 3)))
    return q


def make(kind, n, leaf=4, size=0.2, scale=1.0, repeat=1, seed=0, device=False):
    r = np.random.default_rng(seed)
    c = r.uniform(-1, 1, (n, 3)) * scale
    w = lambda: r.uniform(0.1, 1.0, n) * size * scale
    s = Scene(min_leaf_primitives=leaf)
    rep = lambda a: np.concatenate([a] * repeat)
    if kind == "spheres":
        s.add_spheres(rep(c), rep(w()))
    elif kind == "planes":
        s.add_planes(rep(c), rep(w()), rep(w()), rep(rotations(n, r)))
    else:
        s.add_cylinders(rep(c), rep(w()), rep(w()), rep(w() * 3), rep(rotations(n, r)))
    s.commit(device=device)
    return s, c


def check(s, o, d, dev, tmin=None, tmax=None, **kw):
    col = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    O, D = (tuple(col(a[:, k]) for k in range(3)) for a in (o, d))
    ref = s.intersect(O, D, col(tmin), col(tmax), normals=True, schedule=SCHEDULE_PER_THREAD)
    h = s.intersect(O, D, col(tmin), col(tmax), normals=True, **kw)
    for k in KEYS:
        a, b = h[k], ref[k]
        assert torch.equal(a.view(torch.int64), b.view(torch.int64)) if a.dtype == torch.float64 else torch.equal(a, b), k
    return ref["t"].cpu().numpy()


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("n", [1, 63, 65, 4097, 300011])
def test_launch_sizes(dev, kind, n):
    s, _ = make(kind, 500, device=True)
    o, d = W.incoherent_rays(n, 5, 1.5)
    check(s, o, d, dev)


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("prims,leaf", [(1, 4), (2, 1), (3, 4), (300, 1), (300, 3), (600, 255), (600, 256), (600, 10 ** 6)])
def test_leaf_sizes(dev, kind, prims, leaf):
    s, _ = make(kind, prims, leaf)
    o, d = W.incoherent_rays(20011, 6, 1.5)
    check(s, o, d, dev)


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("size,scale,repeat", [(2.0, 1.0, 1), (0.3, 1.0, 3), (1e-6, 1.0, 1), (0.2, 1e-6, 2), (0.2, 1e11, 1),
                                               (0.2, 1e13, 1)])
def test_overlaps_sizes_and_windows(dev, kind, size, scale, repeat):
    s, c = make(kind, 400, size=size, scale=scale, repeat=repeat)
    o, d = W.incoherent_rays(30011, 7, 1.5)
    o = o * scale
    r = np.random.default_rng(8)
    to = c[r.integers(len(c), size=len(o))] + r.standard_normal(o.shape) * size * scale * 0.3 - o
    d[::2] = (to / np.linalg.norm(to, axis=1, keepdims=True))[::2]
    t = check(s, o, d, dev)
    t = np.where(t < 1e300, t, scale)
    ulp = r.integers(-2, 3, len(t)) * np.spacing(t)
    check(s, o, d, dev, tmax=t + ulp)
    check(s, o, d, dev, tmin=np.maximum(t + ulp, 0.0))
    check(s, o, d, dev, tmin=t * r.uniform(0, 1.1, len(t)), tmax=t * 1.5)


@pytest.mark.parametrize("kind", TYPES)
def test_grazing_rays(dev, kind):
    # axis-aligned primitives on a grid, rays along box planes up to rounding
    g = np.stack(np.meshgrid(*[np.arange(6.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(g)
    s = Scene()
    eye = np.broadcast_to(np.eye(3), (n, 3, 3)).copy()
    half = np.full(n, 0.5)
    if kind == "spheres":
        s.add_spheres(g, half)
    elif kind == "planes":
        s.add_planes(g, half * 2, half * 2, eye)
    else:
        s.add_cylinders(g, half, half, half * 2, eye)
    s.commit()
    r = np.random.default_rng(9)
    m = 40000
    o = np.round(r.uniform(-1, 6, (m, 3)) * 2) / 2
    d = r.standard_normal((m, 3))
    k = r.integers(3, size=m)
    d[np.arange(m), k] *= 10.0 ** r.uniform(-18, -6, m)
    o += r.standard_normal((m, 3)) * 10.0 ** r.uniform(-18, -1, (m, 1))
    check(s, o, d / np.linalg.norm(d, axis=1, keepdims=True), dev)
    check(s, o, d * 10.0 ** r.uniform(-3, 3, (m, 1)), dev)


@pytest.mark.parametrize("kind", TYPES)
def test_rays_left_to_the_exact_kernel(dev, kind):
    s, _ = make(kind, 500)
    o, d = W.incoherent_rays(5000, 14, 1.5)
    o, d = o.copy(), d.copy()
    d[0::5, 0] = 0.0
    d[1::5, 1] = -0.0
    d[2::5] = [0.0, 0.0, 1.0]
    o[3::25, 2] = np.nan
    d[4::25, 1] = np.inf
    o[8::25] = 1e14
    d[9::25] *= 1e-31
    tmin = np.zeros(len(o))
    tmin[7::25] = -1.0
    tmin[12::25] = np.nan
    tmax = np.full(len(o), np.inf)
    tmax[11::25] = np.nan
    check(s, o, d, dev, tmin=tmin, tmax=tmax)


@pytest.mark.parametrize("kw", [{"stack_ring": 4}, {"stack_ring": 8}, {"block_size": 64}, {"refill": 1}, {"refill": 64},
                                {"pool_size": 128}, {"sort": 1}])
def test_launch_shapes(dev, kw):
    o, d = W.incoherent_rays(300007, 6, 1.5)
    for kind in TYPES:
        check(make(kind, 2000, size=0.1)[0], o, d, dev, **kw)
