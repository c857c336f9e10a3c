"""Directions a little longer than one, with tmin: the reference clips boxes at tmin in units of the direction as given, and
triangles at tmin in units of its normalised form, so a hit just behind tmin in a flat box is not reached. The kernel of
packed waves, of one wave for one ray, and the batch give the hits of the one-ray-per-thread kernel there."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Batch, Ray, RayHit, Scene, intersect1  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


def plane_mesh(n, z):
    x = np.linspace(-1.0, 1.0, n + 1)
    gx, gy = np.meshgrid(x, x, indexing="ij")
    v = np.stack([gx.ravel(), gy.ravel(), np.full(gx.size, z)], 1)
    i = (np.arange(n)[:, None] * (n + 1) + np.arange(n)[None, :]).ravel()
    f = np.concatenate([np.stack([i, i + 1, i + n + 2], 1), np.stack([i, i + n + 2, i + n + 1], 1)])
    return v, f.astype(np.uint32)


@pytest.mark.parametrize("extra", [2.0 ** -50, 1e-12, 1e-8, 3e-7, 4.7e-7, -1e-8, -4.7e-7])
def test_hits_close_behind_tmin(extra):
    s = Scene()
    s.add_mesh(*plane_mesh(24, 0.25))
    s.commit()
    r = np.random.default_rng(1)
    n = 20011
    o = np.stack([r.uniform(-0.9, 0.9, n), r.uniform(-0.9, 0.9, n), np.full(n, -1.0)], 1)
    d = np.stack([r.uniform(-0.05, 0.05, n), r.uniform(-0.05, 0.05, n), np.ones(n)], 1)
    d *= ((1.0 + extra) / np.linalg.norm(d, axis=1))[:, None]
    t = 1.25 * np.linalg.norm(d, axis=1) / d[:, 2]  # distances along the normalised directions
    tmin = t * (1.0 - abs(extra) * r.uniform(-0.5, 1.5, n))
    O, D = (tuple(torch.from_numpy(np.ascontiguousarray(a[:, k])).cuda() for k in range(3)) for a in (o, d))
    T = torch.from_numpy(tmin).cuda()
    ref = s.intersect(O, D, T, schedule=SCHEDULE_PER_THREAD)
    bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
    for got in (s.intersect(O, D, T), s.intersect(O, D, T, precision=1)):
        for k in ref:
            assert torch.equal(bits(got[k]), bits(ref[k])), k
    b = Batch([(s, O, D, T, None), (s, D, O, T, None)])
    b.launch()
    for k in ("t", "prim_id"):
        assert torch.equal(bits(b.hits[0][k]), bits(ref[k])), k
    prim = ref["prim_id"].cpu().numpy()
    assert extra < 1e-9 or (prim < 0).any() and (prim >= 0).any()
    for i in range(0, n, 501):
        hit = RayHit()
        intersect1(s, Ray(tuple(o[i]), tuple(d[i]), float(tmin[i])), hit)
        assert np.int32(np.uint32(hit.prim_id)) == prim[i], i
