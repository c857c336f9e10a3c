"""Any hits of triangles in split precision for scenes without pre-test records (BLAZERT_AMD_SPLIT_PRETEST=0 at upload, or
coordinates above 1e12), where every triangle of a leaf gets the FP64 test: the hits of the one-ray-per-thread kernel."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.capi import PRECISION_FP32_TRAV_FP64_HIT, SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


def scene(pretest, level, leaf, scale):
    v, f = W.icosphere(level)
    old = os.environ.get("BLAZERT_AMD_SPLIT_PRETEST")
    os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = pretest
    try:
        s = Scene(min_leaf_primitives=leaf)
        s.add_mesh(np.concatenate([v, 0.9 * v]) * scale, np.concatenate([f, f + len(v)]).astype(np.uint32))
        s.commit()
        s.upload()
    finally:
        if old is None:
            del os.environ["BLAZERT_AMD_SPLIT_PRETEST"]
        else:
            os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = old
    return s


@pytest.mark.parametrize("pretest,scale", [("0", 1.0), ("1", 1e13)])
@pytest.mark.parametrize("level,leaf", [(0, 4), (0, 64), (1, 1), (3, 4), (3, 33), (5, 4)])
@pytest.mark.parametrize("n", [1, 4097, 300007])
def test_hits(pretest, scale, level, leaf, n):
    s = scene(pretest, level, leaf, scale)
    o, d = W.incoherent_rays(n, 5, 1.5)
    O, D = (tuple(torch.from_numpy(np.ascontiguousarray(a[:, k])).cuda() for k in range(3)) for a in (o * scale, d))
    run = lambda **k: s.intersect(O, D, precision=PRECISION_FP32_TRAV_FP64_HIT, any_hit=True, normals=True, **k)
    ref, got = run(schedule=SCHEDULE_PER_THREAD), run()
    for k in ref:
        bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
        assert torch.equal(bits(got[k]), bits(ref[k])), k
    assert n == 1 or (got["prim_id"] >= 0).any()
