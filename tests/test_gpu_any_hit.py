"""Any hits of triangles in split precision (k_trace_any: nearest-first order, work shared at the end of a launch) are those of
the one-ray-per-thread kernel, whichever of a ray's many hits comes first in the visiting order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.capi import PRECISION_FP32_TRAV_FP64_HIT, SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu
KEYS = ("t", "u", "v", "prim_id", "geom_id", "normal")


def scene(layers, level=4, leaf=4):
    """Concentric spheres: every ray inside has many hits to choose from."""
    v, f = W.icosphere(level)
    vs = [v * (1.0 - 0.05 * k) for k in range(layers)]
    fs = [f.astype(np.int64) + k * len(v) for k in range(layers)]
    s = Scene(min_leaf_primitives=leaf)
    s.add_mesh(np.concatenate(vs), np.concatenate(fs).astype(np.uint32))
    s.commit()
    return s


def check(s, o, d, tmin=None, tmax=None, **kw):
    col = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()
    O, D = (tuple(col(a[:, k]) for k in range(3)) for a in (o, d))
    run = lambda **k: s.intersect(O, D, col(tmin), col(tmax), precision=PRECISION_FP32_TRAV_FP64_HIT, any_hit=True,
                                  normals=True, **k)
    ref, got = run(schedule=SCHEDULE_PER_THREAD), run(**kw)
    for k in KEYS:
        bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
        assert torch.equal(bits(got[k]), bits(ref[k])), k
    return ref["t"].cpu().numpy()


@pytest.mark.parametrize("layers", [1, 8])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 4097, 262145, 500009])
def test_launch_sizes(layers, n):
    o, d = W.incoherent_rays(n, 5, 1.5)
    check(scene(layers), o, d)


@pytest.mark.parametrize("leaf", [1, 3, 300, 10 ** 6])
def test_leaf_sizes(leaf):
    o, d = W.incoherent_rays(3001, 6, 1.5)
    check(scene(2, 3, leaf), o, d)


def test_windows_and_refused_rays():
    s = scene(6)
    o, d = W.incoherent_rays(40001, 7, 1.5)
    o, d = o.copy(), d.copy()
    t = check(s, o, d)
    t = np.where(t < 1e300, t, 1.0)
    r = np.random.default_rng(8)
    ulp = r.integers(-2, 3, len(t)) * np.spacing(t)
    check(s, o, d, tmax=t + ulp)
    check(s, o, d, tmin=t + ulp)
    check(s, o, d, tmin=np.full(len(o), -0.5), tmax=np.where(r.random(len(o)) < 0.1, np.nan, 2.0))
    check(s, o * 0.0, d)  # every ray from one point inside many boxes: ties between entry distances
    d[0::5, 0] = 0.0
    d[1::5, 1] = -0.0
    d[2::5, 2] = 1e-32
    o[3::25, 2] = np.nan
    o[8::25] = 1e14
    check(s, o, d)


@pytest.mark.parametrize("kw", [{"stack_ring": 4}, {"block_size": 64}, {"refill": 1}, {"refill": 64}, {"pool_size": 32},
                                {"sort": 1}])
def test_launch_shapes(kw):
    o, d = W.incoherent_rays(300007, 9, 1.5)
    check(scene(5), o, d, **kw)
