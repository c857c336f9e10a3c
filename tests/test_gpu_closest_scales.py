"""Closest surfaces of meshes so small that squared distances leave the FP32 range: the FP64 search's results, which a scene
without pre-test records (BLAZERT_AMD_SPLIT_PRETEST=0 at upload) keeps."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("near", [True, False])
@pytest.mark.parametrize("scale", [1e-40, 1e-27, 1e-25, 1e-23, 1e-22, 1e-21, 1e-20, 1e-18, 1e-15, 9e-13, 2e-12, 1.0])
def test_scales(scale, near):
    r = np.random.default_rng(6)
    m, n = 700, 100003
    v = r.uniform(-0.5, 0.5, (m, 1, 3)) + r.uniform(-0.05, 0.05, (m, 3, 3))
    scenes = []
    for pretest in ("1", "0"):
        old = os.environ.get("BLAZERT_AMD_SPLIT_PRETEST")
        os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = pretest
        try:
            s = Scene()
            s.add_mesh(v.reshape(-1, 3) * scale, np.arange(3 * m, dtype=np.uint32).reshape(-1, 3))
            s.commit()
            s.upload()
        finally:
            if old is None:
                del os.environ["BLAZERT_AMD_SPLIT_PRETEST"]
            else:
                os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = old
        scenes.append(s)
    p = r.uniform(-1, 1, (n, 3))
    if near:
        p = v[r.integers(m, size=n)].mean(1) + r.normal(size=(n, 3)) * 10.0 ** r.uniform(-12, -1, (n, 1))
    P = tuple(torch.from_numpy(np.ascontiguousarray(p[:, k] * scale)).cuda() for k in range(3))
    a, b = (s.closest_surface(P) for s in scenes)
    assert torch.equal(a["distance"].view(torch.int64), b["distance"].view(torch.int64))
    assert torch.equal(a["prim_id"], b["prim_id"])
