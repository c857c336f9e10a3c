"""The FP32 pre-test of cylinders at scales whose squares leave the FP32 range: closest hits are those of the one-ray-per-thread
FP64 kernel, and split-precision hits those of a scene without pre-test records (BLAZERT_AMD_SPLIT_PRETEST=0 at upload)."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e-35, 1e-24, 1e-23, 1e-22, 3e-22, 1e-21, 1e-20, 1e-19, 1e-17, 1e-14, 1.0, 1e11])
def test_scales(scale):
    r = np.random.default_rng(4)
    m, n = 400, 100003
    c = r.uniform(-1, 1, (m, 3))
    a, b, h = (r.uniform(0.01, 0.2, m) for _ in range(3))
    rot = np.linalg.qr(r.standard_normal((m, 3, 3)))[0]
    scenes = []
    for pretest in ("1", "0"):
        old = os.environ.get("BLAZERT_AMD_SPLIT_PRETEST")
        os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = pretest
        try:
            s = Scene()
            s.add_cylinders(c * scale, a * scale, b * scale, h * scale, rot)
            s.commit()
            s.upload()
        finally:
            if old is None:
                del os.environ["BLAZERT_AMD_SPLIT_PRETEST"]
            else:
                os.environ["BLAZERT_AMD_SPLIT_PRETEST"] = old
        scenes.append(s)
    o = r.uniform(-2, 2, (n, 3))
    d = c[r.integers(m, size=n)] + r.normal(size=(n, 3)) * 0.1 - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    O, D = (tuple(torch.from_numpy(np.ascontiguousarray(x[:, k])).cuda() for k in range(3)) for x in (o * scale, d))
    s, plain = scenes
    for got, ref in ((s.intersect(O, D), s.intersect(O, D, schedule=SCHEDULE_PER_THREAD)),
                     (s.intersect(O, D, precision=1), plain.intersect(O, D, precision=1))):
        for k in ref:
            bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
            assert torch.equal(bits(got[k]), bits(ref[k])), k
