"""Directions a little shorter than one, whose distances to boxes are a little longer than those to hits: of two hits closer
together than that, the reference may not reach the nearer one behind the other. Rays through many triangles of a thin slab,
traced by one lane, by lanes that share a ray and in batches, give the hits of the one-ray-per-thread kernel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Batch, Ray, RayHit, Scene, intersect1  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thin", [1e-12, 1e-9, 1e-7, 1e-6])
@pytest.mark.parametrize("short", [0.0, 1e-12, 1e-9, 1e-7, 4.7e-7])
def test_thin_slab(thin, short):
    r = np.random.default_rng(3)
    m, n = 3000, 20011
    c = r.uniform(-1.0, 1.0, (m, 1, 2))
    xy = c + r.uniform(-0.2, 0.2, (m, 3, 2))
    z = 0.25 * (1.0 + thin * r.random((m, 1, 1))) * np.ones((m, 3, 1))  # flat triangles, flat boxes
    s = Scene()
    s.add_mesh(np.concatenate([xy, z], 2).reshape(-1, 3), np.arange(3 * m, dtype=np.uint32).reshape(-1, 3))
    s.commit()
    o = np.stack([r.uniform(-0.9, 0.9, n), r.uniform(-0.9, 0.9, n), np.full(n, -1.0)], 1)
    d = np.stack([r.uniform(-0.05, 0.05, n), r.uniform(-0.05, 0.05, n), np.ones(n)], 1)
    d *= ((1.0 - short) / np.linalg.norm(d, axis=1))[:, None]
    O, D = (tuple(torch.from_numpy(np.ascontiguousarray(a[:, k])).cuda() for k in range(3)) for a in (o, d))
    ref = s.intersect(O, D, schedule=SCHEDULE_PER_THREAD)
    bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
    for got in (s.intersect(O, D), s.intersect(O, D, precision=1)):
        for k in ref:
            assert torch.equal(bits(got[k]), bits(ref[k])), k
    b = Batch([(s, O, D)])
    b.launch()
    for k in ("t", "prim_id"):
        assert torch.equal(bits(b.hits[0][k]), bits(ref[k])), k
    prim = ref["prim_id"].cpu().numpy()
    for i in range(0, n, 101):
        hit = RayHit()
        intersect1(s, Ray(tuple(o[i]), tuple(d[i])), hit)
        assert np.int32(np.uint32(hit.prim_id)) == prim[i], i
