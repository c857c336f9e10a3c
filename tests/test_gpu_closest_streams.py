"""Closest-surface searches share nothing between streams, threads and graphs: they can be captured on a stream's first call,
graphs that hold them can be replayed side by side, and threads can search on one stream at the same time."""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu
MANY = 600_011  # more than the resident waves take in one go


def mesh(level=5):
    s = Scene()
    s.add_mesh(*W.icosphere(level))
    s.commit()
    return s


def points(n, seed):
    return torch.from_numpy(np.random.default_rng(seed).uniform(-2, 2, (3, n))).cuda().unbind(0)


def same(a, b):
    bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
    return all(torch.equal(bits(a[k]), bits(b[k])) for k in b)


def capture(s, p, stream):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        out = s.closest_surface(p)
    return g, out


@pytest.mark.parametrize("kind", ["mesh", "spheres"])
@pytest.mark.parametrize("n", [1, 4097, MANY])
def test_first_call_on_a_stream_under_capture(kind, n):
    if kind == "mesh":
        s = mesh()
        s.closest_surface(points(10, 0))  # makes the leaf-order vertices, on another stream
    else:
        s = Scene()
        s.add_spheres(*W.sphere_field(500, seed=1))
        s.commit()
        s.upload()
    p = points(n, 1)
    torch.cuda.synchronize()
    g, out = capture(s, p, torch.cuda.Stream())
    ref = s.closest_surface(p)
    for _ in range(3):
        for x in out.values():
            x.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert same(out, ref)


def test_graphs_of_one_stream_replayed_side_by_side():
    s = mesh()
    ps = [points(MANY + 64 * k, 2 + k) for k in range(2)]
    refs = [{k: v.clone() for k, v in s.closest_surface(p).items()} for p in ps]
    torch.cuda.synchronize()
    first = torch.cuda.Stream()
    graphs = [capture(s, p, first) for p in ps]
    streams = [torch.cuda.Stream() for _ in ps]
    for _ in range(5):
        for _, out in graphs:
            for x in out.values():
                x.zero_()
        torch.cuda.synchronize()
        eager = None
        for st, (g, _) in zip(streams, graphs):
            with torch.cuda.stream(st):
                g.replay()
        with torch.cuda.stream(first):
            eager = s.closest_surface(ps[0])  # beside the replays, with counters
        torch.cuda.synchronize()
        assert same(eager, refs[0])
        for (_, out), ref in zip(graphs, refs):
            assert same(out, ref)


def test_threads_on_one_stream():
    s = mesh()
    ps = [points(MANY + 64 * k, 4 + k) for k in range(4)]
    refs = [{k: v.clone() for k, v in s.closest_surface(p).items()} for p in ps]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        for _ in range(20):
            if not same(s.closest_surface(ps[k]), refs[k]):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
