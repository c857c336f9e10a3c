"""The fast closest-hit traversal of triangle trees (k_trace_tri: FP32 reference-order boxes and pre-tests, certified
FP64 hits, shared work in the drain) gives the bits of the exact FP64 kernel, which the one-ray-per-thread schedule
still runs: on launches around its wave, claim and block sizes, rays that its certificate must refuse (vertices, edges,
ties, windows ending at the hit, triangles in several copies), rays outside its assumptions (long, short, axis-parallel,
NaN), any leaf size, and batches of any number of jobs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Batch, Scene, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu
KEYS = ("t", "u", "v", "prim_id", "geom_id", "normal")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def make(v, f, leaf=4, device=False):
    s = Scene(min_leaf_primitives=leaf)
    s.add_mesh(v, f)
    s.commit(device=device)
    return s


def cols(a, dev):
    return tuple(torch.from_numpy(np.ascontiguousarray(a[:, k])).to(dev) for k in range(3))


def bits(x):
    return x.view(torch.int64) if x.dtype == torch.float64 else x


def check(s, o, d, dev, tmin=None, tmax=None, **kw):
    col = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    O, D = cols(o, dev), cols(d, dev)
    ref = s.intersect(O, D, col(tmin), col(tmax), normals=True, schedule=SCHEDULE_PER_THREAD)
    for precision in (0, 1):
        h = s.intersect(O, D, col(tmin), col(tmax), normals=True, precision=precision, **kw)
        for k in KEYS:
            assert torch.equal(bits(h[k]), bits(ref[k])), (precision, k)
    return {k: ref[k].cpu().numpy() for k in KEYS}


@pytest.fixture(scope="module")
def sphere():
    return W.icosphere(5)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257, 4097, 262144, 262145, 600011])
def test_launch_sizes(dev, sphere, n):
    s = make(*sphere, device=True)
    o, d = W.incoherent_rays(n, 5, 1.5)
    check(s, o, d, dev)


@pytest.mark.parametrize("kw", [{"stack_ring": 4}, {"stack_ring": 8}, {"block_size": 64}, {"block_size": 192},
                                {"refill": 1}, {"refill": 64}, {"pool_size": 32}, {"sort": 1}])
def test_launch_shapes(dev, sphere, kw):
    s = make(*sphere)
    o, d = W.incoherent_rays(300007, 6, 1.5)
    check(s, o, d, dev, **kw)


@pytest.mark.parametrize("leaf", [1, 3, 40, 255, 256, 100000])
def test_leaf_sizes(dev, sphere, leaf):
    # a leaf of more than 255 triangles keeps the exact kernels; 100000 makes the root a leaf
    v, f = sphere
    s = make(v, f[:2000] if leaf >= 255 else f, leaf)
    o, d = W.incoherent_rays(3001, 7, 1.5)
    check(s, o, d, dev)


def aimed(v, f, n, seed):
    """Rays through vertices, edge points and points within rounding of an edge."""
    r = np.random.default_rng(seed)
    tri = f[r.integers(len(f), size=n)]
    w = r.random((n, 3))
    kind = r.integers(4, size=n)
    w[kind == 0] = [1.0, 0.0, 0.0]
    w[kind == 1, 2] = 0.0
    near = kind == 2
    w[near, 2] = np.where(r.random(near.sum()) < 0.5, -1, 1) * 10.0 ** r.uniform(-17, -9, near.sum())
    w /= w.sum(1, keepdims=True)
    p = (v[tri] * w[:, :, None]).sum(1)
    scale = np.abs(v).max()
    o = r.standard_normal((n, 3)) * 3.0 * scale
    d = p - o
    return o, d / np.linalg.norm(d, axis=1, keepdims=True)


@pytest.mark.parametrize("scale", [1e-6, 1.0, 3e3, 1e11, 1e13])
def test_edges_vertices_and_windows(dev, sphere, scale):
    v, f = sphere
    v = v * scale
    s = make(v, f)
    o, d = aimed(v, f, 20000, 8)
    ref = check(s, o, d, dev)
    t = np.where(ref["t"] < 1e300, ref["t"], scale)
    r = np.random.default_rng(9)
    ulp = r.integers(-2, 3, len(t)) * np.spacing(t)
    check(s, o, d, dev, tmax=t + ulp)
    check(s, o, d, dev, tmin=t + ulp)
    check(s, o, d, dev, tmin=t * (1 + 1e-9 * r.standard_normal(len(t))), tmax=t * 1.5)


@pytest.mark.parametrize("factor", [0.5, 1 - 1e-7, 1 + 1e-7, 2.0, 1e12])
def test_direction_lengths(dev, sphere, factor):
    s = make(*sphere)
    o, d = W.incoherent_rays(20000, 10, 1.5)
    check(s, o, d * factor, dev)
    check(s, o, d * factor, dev, tmin=np.full(len(o), 0.3), tmax=np.full(len(o), 1.7))


def test_copies_of_every_triangle(dev, sphere):
    # every hit is a tie: the rays overflow the list, and the exact kernel traces them all
    v, f = sphere
    s = make(v, np.concatenate([f, f[::-1], f]))
    o, d = W.incoherent_rays(60000, 11, 1.5)
    check(s, o, d, dev)


def test_rays_in_the_plane_of_triangles(dev):
    # a tilted floor of coplanar triangles and rays inside its plane, up to rounding, with a mesh on it
    q, _ = np.linalg.qr(np.random.default_rng(12).standard_normal((3, 3)))
    g = np.linspace(-1, 1, 33)
    x, y = np.meshgrid(g, g, indexing="ij")
    v = np.stack([x.ravel(), y.ravel(), np.zeros(x.size)], 1)
    i = (np.arange(32)[:, None] * 33 + np.arange(32)[None, :]).ravel()
    f = np.concatenate([np.stack([i, i + 33, i + 34], 1), np.stack([i, i + 34, i + 1], 1)])
    sv, sf = W.icosphere(3)
    v = np.concatenate([v, sv * 0.3])
    f = np.concatenate([f, sf.astype(np.int64) + 33 * 33]).astype(np.uint32)
    s = make(v @ q.T, f)
    r = np.random.default_rng(13)
    n = 20000
    a = r.uniform(0, 2 * np.pi, n)
    d = np.stack([np.cos(a), np.sin(a), np.zeros(n)], 1) @ q.T
    o = np.stack([r.uniform(-1.5, 1.5, n), r.uniform(-1.5, 1.5, n), np.zeros(n)], 1) @ q.T
    check(s, o, d, dev)


def test_rays_left_to_the_exact_kernel(dev, sphere):
    s = make(*sphere)
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
    tmax = np.full(len(o), np.inf)
    tmax[11::25] = np.nan
    check(s, o, d, dev, tmin=tmin, tmax=tmax)


def test_in_out_hits(dev, sphere):
    s = make(*sphere)
    o, d = W.incoherent_rays(5003, 15, 1.5)
    O, D = cols(o, dev), cols(d, dev)
    out = []
    for schedule in (SCHEDULE_PER_THREAD, 0):
        h = {k: torch.full((len(o),), 0.25 * i, dtype=torch.float64, device=dev) for i, k in enumerate("tuv")}
        h["prim_id"] = torch.full((len(o),), 7, dtype=torch.int32, device=dev)
        h["geom_id"] = torch.full((len(o),), 3, dtype=torch.int32, device=dev)
        out.append(s.intersect(O, D, hits=h, schedule=schedule))
    for k in out[0]:
        assert torch.equal(bits(out[0][k]), bits(out[1][k])), k


@pytest.mark.parametrize("jobs", [1, 2, 32, 33])
@pytest.mark.parametrize("precision", [0, 1])
def test_batches(dev, jobs, precision):
    items, refs = [], []
    for k in range(jobs):
        v, f = W.icosphere(1 + k % 4, seed=k) if k % 2 == 0 else W.torus(200 + 100 * k, seed=k)
        s = make(v, f)
        o, d = W.incoherent_rays(1 + 617 * k, 20 + k, 1.5)
        if k % 3 == 0:
            d = d * 0.5  # left to the exact kernel
        O, D = cols(o, dev), cols(d, dev)
        items.append((s, O, D))
        refs.append(s.intersect(O, D, normals=True, schedule=SCHEDULE_PER_THREAD))
    b = Batch(items, precision=precision, normals=True)
    st = torch.cuda.Stream()
    b.launch()
    torch.cuda.synchronize()
    b.capture(st)
    for replay in range(3):
        if replay:
            for h in b.hits:
                for x in h.values():
                    x.zero_()
            torch.cuda.synchronize()
            b.replay(st)
            torch.cuda.synchronize()
        for h, ref in zip(b.hits, refs):
            for k in KEYS:
                assert torch.equal(bits(h[k]), bits(ref[k])), (replay, k)
