"""The rays a fast traversal leaves to the exact kernel, in launches with a fixed range per wave (a bit per ray), in claimed
ones (a list), and in claimed ones that leave more than the list holds."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["mesh", "mesh_f32", "spheres", "cylinders"])
@pytest.mark.parametrize("n", [1, 64, 65, 4095, 4097, 100003, 262144, 262145, 400009])
def test_every_kind(kind, n):
    f32 = kind.endswith("f32")
    s = Scene(dtype=np.float32 if f32 else np.float64)
    r = np.random.default_rng(1)
    if kind.startswith("mesh"):
        v, f = W.icosphere(3)
        s.add_mesh(v, np.concatenate([f, f]))  # every hit is a tie: listed
    else:
        c, w = r.uniform(-1, 1, (200, 3)), r.uniform(0.05, 0.2, 200)
        if kind == "spheres":
            s.add_spheres(c, w)
        else:
            s.add_cylinders(c, w, w, w, np.linalg.qr(r.standard_normal((200, 3, 3)))[0])
    s.commit()
    o, d = W.incoherent_rays(n, 5, 1.5)
    d = d.copy()
    d[::7, 0] = 0.0  # deferred
    col = lambda a: tuple(torch.from_numpy(np.ascontiguousarray(a[:, k], dtype=s.dtype)).cuda() for k in range(3))
    O, D = col(o), col(d)
    bits = lambda x: x.view(torch.int64 if x.element_size() == 8 else torch.int32)
    for kw in ({}, {"any_hit": True, "precision": 0 if f32 else 1}, {"sort": 0 if f32 else 1}, {"block_size": 64}):
        exact = {k: x for k, x in kw.items() if k in ("any_hit", "precision")}
        ref = s.intersect(O, D, normals=True, schedule=SCHEDULE_PER_THREAD, **exact)
        got = s.intersect(O, D, normals=True, **kw)
        for k in ref:
            assert torch.equal(bits(got[k]), bits(ref[k])), (kw, k)
