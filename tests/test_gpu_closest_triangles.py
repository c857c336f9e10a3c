"""The FP32 closest-surface search of triangles (4-wide boxes, pre-test, shared work) against the FP64 search, which a scene
without pre-test records (BLAZERT_AMD_SPLIT_PRETEST=0 at upload) keeps: random points, points on vertices, edges and in the
planes of faces, points outside the FP32 bounds' range and points that are not numbers, with every bit equal."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (1e-6, 0.0), (1e11, 0.0), (1.0, 3e3), (1e-12, 0.0)])
@pytest.mark.parametrize("n", [1, 65, 4097, 300001])
def test_closest_triangles_pretest_never_changes_a_result(dev, scale, shift, n):
    v, f = W.icosphere(4 if n < 300000 else 2)
    f = np.concatenate([f, f[:7]])  # copies: ties go to the lower id
    v = v * scale + shift * scale
    scenes = []
    for pretest in ("1", "0"):
        old = os.environ.get("BLAZERT_AMD_SPLIT_PRETEST")
        os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = pretest
        try:
            s = Scene()
            s.add_mesh(v, f)
            s.commit()
            s.upload()
        finally:
            if old is None:
                del os.environ["BLAZERT_AMD_SPLIT_PRETEST"]
            else:
                os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = old
        scenes.append(s)
    r = np.random.default_rng(n)
    p = (r.uniform(-2, 2, (n, 3)) + shift) * scale
    t = f[r.integers(len(f), size=n)]
    w = r.random((n, 3)) * (r.random((n, 3)) < 0.7)
    w[w.sum(1) == 0, 0] = 1.0
    on = (v[t] * (w / w.sum(1, keepdims=True))[:, :, None]).sum(1)
    p[0::3] = on[0::3]
    if n > 4000:
        p[1::997, 1] = np.nan
        p[2::997] = 1e13
        p[5::997, 0] = np.inf
    P = torch.from_numpy(p).to(dev)
    a, b = (s.closest_surface(P) for s in scenes)
    assert torch.equal(a["distance"].view(torch.int64), b["distance"].view(torch.int64))
    assert torch.equal(a["prim_id"], b["prim_id"]) and torch.equal(a["geom_id"], b["geom_id"])
