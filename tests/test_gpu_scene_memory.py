"""Device memory of destroyed scenes is reused by new ones: traces still in flight on another stream when their scene goes
away keep their results, scenes of changing sizes and types built one after the other give the hits of scenes built alone,
and threads building at the same time do not share blocks."""
import threading

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


def build(level, device, seed):
    s = Scene()
    s.add_mesh(*W.icosphere(level, seed=seed))
    if seed % 2:
        s.add_spheres(*W.sphere_field(200 + seed, seed=seed))
    s.commit(device=device)
    return s


def trace(s, rays, stream=None):
    return s.intersect(*rays, stream=stream)


def same(a, b):
    return all(torch.equal(a[k].view(torch.int64) if a[k].dtype == torch.float64 else a[k],
                           b[k].view(torch.int64) if b[k].dtype == torch.float64 else b[k]) for k in a)


def test_scenes_one_after_the_other(dev):
    rays = tuple(torch.from_numpy(x).to(dev) for x in W.incoherent_rays(200001, 3, 1.5))
    specs = [(6, True, 0), (6, True, 1), (5, False, 2), (6, True, 3), (3, True, 4), (6, False, 5), (5, True, 6)]
    alone = []
    for spec in specs:
        s = build(*spec)
        alone.append(trace(s, rays))
        torch.cuda.synchronize()
        s.close()
    side = torch.cuda.Stream()
    hits, last = [], None
    for spec in specs * 2:
        s = build(*spec)
        hits.append(trace(s, rays, side))
        if last is not None:
            last.close()  # its trace may still run on the side stream
        last = s
    torch.cuda.synchronize()
    for k, h in enumerate(hits):
        assert same(h, alone[k % len(specs)]), specs[k % len(specs)]


def test_threads(dev):
    rays = tuple(torch.from_numpy(x).to(dev) for x in W.incoherent_rays(20001, 4, 1.5))
    ref = [trace(build(5, True, k), rays) for k in range(4)]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(6):
                s = Scene()
                s.add_mesh(*W.icosphere(5, seed=k))
                if k % 2:
                    s.add_spheres(*W.sphere_field(200 + k, seed=k))
                s.commit(device=True)
                h = trace(s, rays)
                st.synchronize()
                if not same(h, ref[k]):
                    bad.append(k)
                s.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
