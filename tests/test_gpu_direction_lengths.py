"""Directions of any length: 1/d below the FP32 range would turn the infinite planes of a 4-wide node's unused slots into NaN,
so such rays belong to the exact kernel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["mesh", "spheres", "cylinders"])
@pytest.mark.parametrize("length,dtype", [(1e-28, np.float64), (1e20, np.float64), (1e29, np.float64), (1e33, np.float64),
                                          (1e60, np.float64), (1e152, np.float64), (1e200, np.float64),
                                          (1e-17, np.float32), (1e15, np.float32), (1e38, np.float32)])
def test_lengths(kind, length, dtype):
    s = Scene(dtype=dtype)
    r = np.random.default_rng(2)
    c, w = r.uniform(-1, 1, (50, 3)), r.uniform(0.1, 0.4, 50)  # 50: records with unused slots
    if kind == "mesh":
        s.add_mesh(*W.icosphere(1))
    elif kind == "spheres":
        s.add_spheres(c, w)
    else:
        s.add_cylinders(c, w, w, w, np.linalg.qr(r.standard_normal((50, 3, 3)))[0])
    s.commit()
    o, d = W.incoherent_rays(3001, 3, 1.5)
    d = d * length
    d[::3, 0] /= length  # one ordinary component
    O, D = (tuple(torch.from_numpy(np.ascontiguousarray(a[:, k], dtype=dtype)).cuda() for k in range(3)) for a in (o, d))
    ref = s.intersect(O, D, schedule=SCHEDULE_PER_THREAD)
    got = s.intersect(O, D)
    for k in ref:
        bits = lambda x: x.view(torch.int64 if x.element_size() == 8 else torch.int32)
        assert torch.equal(bits(got[k]), bits(ref[k])), k
