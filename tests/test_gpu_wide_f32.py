"""The fast closest-hit traversal of Scene<float> (4-wide boxes widened by the reference's FP32 rounding; the leaf of a hit is
checked with the reference's own FP32 box tests) gives the bits of the binary FP32 kernel, which the one-ray-per-thread
schedule still runs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu
KEYS = ("t", "u", "v", "prim_id", "geom_id", "normal")
TYPES = ("mesh", "spheres", "cylinders")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def make(kind, n, leaf=4, scale=1.0, repeat=1):
    r = np.random.default_rng(n)
    s = Scene(dtype=np.float32, min_leaf_primitives=leaf)
    c = r.uniform(-1, 1, (n, 3)) * scale
    w = lambda: np.concatenate([r.uniform(0.02, 0.3, n) * scale] * repeat)
    rep = lambda a: np.concatenate([a] * repeat)
    if kind == "mesh":
        v, f = W.icosphere(5)
        s.add_mesh(v * scale, rep(f[:n]))
        c = v[f[:n, 0]] * scale
    elif kind == "spheres":
        s.add_spheres(rep(c), w())
    else:
        s.add_cylinders(rep(c), w(), w(), w(), rep(np.linalg.qr(r.standard_normal((n, 3, 3)))[0]))
    s.commit()
    return s, c


def check(s, o, d, dev, tmin=None, tmax=None, **kw):
    col = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dev)
    O, D = (tuple(col(a[:, k]) for k in range(3)) for a in (o, d))
    ref = s.intersect(O, D, col(tmin), col(tmax), normals=True, schedule=SCHEDULE_PER_THREAD)
    h = s.intersect(O, D, col(tmin), col(tmax), normals=True, **kw)
    for k in KEYS:
        assert torch.equal(h[k].view(torch.int32), ref[k].view(torch.int32)), k
    return ref["t"].cpu().numpy()


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("n", [1, 64, 65, 4097, 300011])
def test_launch_sizes(dev, kind, n):
    o, d = W.incoherent_rays(n, 5, 1.5)
    check(make(kind, 2000)[0], o, d, dev)


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("prims,leaf", [(1, 4), (2, 1), (3, 4), (300, 1), (300, 3), (600, 255), (600, 256), (600, 10 ** 6)])
def test_leaf_sizes(dev, kind, prims, leaf):
    o, d = W.incoherent_rays(20011, 6, 1.5)
    check(make(kind, prims, leaf)[0], o, d, dev)


@pytest.mark.parametrize("kind", TYPES)
@pytest.mark.parametrize("scale,repeat", [(1.0, 1), (1.0, 3), (1e-6, 1), (1e-18, 1), (1e8, 1), (1e13, 1)])
def test_aimed_rays_and_windows(dev, kind, scale, repeat):
    s, c = make(kind, 1500, scale=scale, repeat=repeat)
    o, d = W.incoherent_rays(30011, 7, 1.5)
    o = (o * scale).astype(np.float32).astype(np.float64)
    r = np.random.default_rng(8)
    to = c[r.integers(len(c), size=len(o))] - o  # through vertices and centres
    d[::2] = (to / np.linalg.norm(to, axis=1, keepdims=True))[::2]
    t = check(s, o, d, dev)
    t = np.where(t < 1e30, t, scale).astype(np.float32)
    ulp = (r.integers(-2, 3, len(t)) * np.spacing(t)).astype(np.float32)
    check(s, o, d, dev, tmax=t + ulp)
    check(s, o, d, dev, tmin=np.maximum(t + ulp, 0))
    check(s, o, d * 10.0 ** r.uniform(-3, 3, (len(d), 1)), dev, tmin=t * 0.5, tmax=t * 1.5)


@pytest.mark.parametrize("kind", TYPES)
def test_grazing_and_refused_rays(dev, kind):
    s, _ = make(kind, 1500)
    r = np.random.default_rng(9)
    o, d = W.incoherent_rays(40000, 14, 1.5)
    d = d.copy()
    k = r.integers(3, size=len(d))
    d[np.arange(len(d)), k] *= 10.0 ** r.uniform(-44, -4, len(d))
    check(s, o, d, dev)
    o = np.round(o * 4) / 4
    check(s, o, d, dev)
    d[0::5, 0] = 0.0
    d[1::5, 1] = -0.0
    o[3::25, 2] = np.nan
    d[4::25, 1] = np.inf
    o[8::25] = 1e14
    d[9::25] *= 1e-31
    tmin = np.zeros(len(o))
    tmin[7::25] = -1.0
    tmin[12::25] = np.nan
    check(s, o, d, dev, tmin=tmin)


@pytest.mark.parametrize("kw", [{"stack_ring": 4}, {"block_size": 64}, {"refill": 1}, {"refill": 64}, {"pool_size": 32}])
def test_launch_shapes(dev, kw):
    o, d = W.incoherent_rays(300007, 6, 1.5)
    for kind in TYPES:
        check(make(kind, 2000)[0], o, d, dev, **kw)
