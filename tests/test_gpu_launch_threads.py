"""Threads that trace one scene on one stream at the same time get the hits of traces made one by one. A trace is several
kernels, the later ones reading what the first ones leave in the stream's counters, and every thread's rays leave others: some
of them axis-parallel, which belong to the exact kernel."""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu
THREADS = 6


def scene(kind, dtype):
    s = Scene(dtype=dtype)
    if kind == "mesh":
        s.add_mesh(*W.icosphere(4))
    else:
        s.add_spheres(*W.sphere_field(500, seed=1))
    s.commit()
    s.upload()
    return s


def rays(n, k, dtype):
    o, d = W.incoherent_rays(n, k, 1.5)
    d[k::THREADS, 0] = 0.0
    return tuple(tuple(torch.from_numpy(np.ascontiguousarray(a[:, c], dtype=dtype)).cuda() for c in range(3)) for a in (o, d))


@pytest.mark.parametrize("kind,dtype,kw", [
    ("mesh", np.float64, {}), ("mesh", np.float64, {"precision": 1}), ("mesh", np.float64, {"precision": 1, "any_hit": True}),
    ("spheres", np.float64, {}), ("mesh", np.float32, {})])
@pytest.mark.parametrize("n", [2001, 30001, 300007])
def test_threads_on_one_stream(kind, dtype, kw, n):
    s = scene(kind, dtype)
    R = [rays(n, k, dtype) for k in range(THREADS)]
    ref = [{k: v.clone() for k, v in s.intersect(*r, **kw).items()} for r in R]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        for _ in range(15):
            h = s.intersect(*R[k], **kw)
            if not all(torch.equal(h[f], ref[k][f]) for f in ("t", "prim_id")):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(THREADS)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
