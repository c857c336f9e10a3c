"""Closest surfaces of meshes with triangles that are lines, or nearly: their normals are roundings, and say nothing about
distances. The FP64 search's results, which a scene without pre-test records (BLAZERT_AMD_SPLIT_PRETEST=0 at upload) keeps."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 295007.30064, 1e-5])
@pytest.mark.parametrize("width", [0.0, 1e-16, 1e-13, 1e-10, 1e-8, 1e-6, 1e-4])
def test_slivers(scale, width):
    r = np.random.default_rng(7)
    m, n = 1500, 100003
    a, e = r.uniform(-1, 1, (m, 3)), r.uniform(-0.3, 0.3, (m, 3))
    v = np.stack([a, a + e, a + e * r.uniform(-1, 2, (m, 1)) + width * r.normal(size=(m, 3))], 1) * scale
    scenes = []
    for pretest in ("1", "0"):
        old = os.environ.get("BLAZERT_AMD_SPLIT_PRETEST")
        os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = pretest
        try:
            s = Scene()
            s.add_mesh(v.reshape(-1, 3), np.arange(3 * m, dtype=np.uint32).reshape(-1, 3))
            s.commit()
            s.upload()
        finally:
            if old is None:
                del os.environ["BLAZERT_AMD_SPLIT_PRETEST"]
            else:
                os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = old
        scenes.append(s)
    w = r.dirichlet(np.ones(3), n)
    p = (v[r.integers(m, size=n)] * w[:, :, None]).sum(1) + scale * r.normal(size=(n, 3)) * 10.0 ** r.uniform(-16, 0, (n, 1))
    P = tuple(torch.from_numpy(np.ascontiguousarray(p[:, k])).cuda() for k in range(3))
    a, b = (s.closest_surface(P) for s in scenes)
    assert torch.equal(a["distance"].view(torch.int64), b["distance"].view(torch.int64))
    assert torch.equal(a["prim_id"], b["prim_id"])
