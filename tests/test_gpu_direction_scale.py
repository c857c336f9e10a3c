"""Directions of every length, with and without tmin, in both precisions: FP64 hits are those of the one-ray-per-thread kernel,
whatever the length; split-precision hits are FP64's, too, for rays that no box's rounding decides."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Batch, Scene, workloads as W  # noqa: E402
from blazert_amd.capi import SCHEDULE_PER_THREAD  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [1e-12, 1e-3, 0.3, 0.999, 1.0, 1.001, 3.0, 1e3, 1e9])
@pytest.mark.parametrize("tmin", [None, 0.05])
@pytest.mark.parametrize("n", [501, 30001, 300007])
def test_lengths(length, tmin, n):
    s = Scene()
    v, f = W.icosphere(4)
    s.add_mesh(np.concatenate([v, 0.8 * v]), np.concatenate([f, f + len(v)]).astype(np.uint32))
    s.commit()
    o, d = W.incoherent_rays(n, 3, 1.5)
    O, D = (tuple(torch.from_numpy(np.ascontiguousarray(a[:, k])).cuda() for k in range(3)) for a in (o, d * length))
    T = None if tmin is None else torch.full((n,), tmin, dtype=torch.float64, device="cuda")
    ref = s.intersect(O, D, T, schedule=SCHEDULE_PER_THREAD)
    bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
    got = s.intersect(O, D, T)
    for k in ref:
        assert torch.equal(bits(got[k]), bits(ref[k])), k
    split = s.intersect(O, D, T, precision=1)
    b = Batch([(s, O, D, T, None)], precision=1)
    b.launch()
    for h in (split, b.hits[0]):
        for k in ref:
            assert torch.equal(bits(h[k]), bits(ref[k])), k
