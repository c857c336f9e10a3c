"""Scene memory kept for the next scene does not get in the way of a stream capture in another thread: launches that take some
of it, and the destruction of scenes, work beside it, and the capture goes on."""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu


def scene():
    s = Scene()
    s.add_mesh(*W.icosphere(4))
    s.commit()
    s.upload()
    return s


@pytest.mark.parametrize("mode", ["thread_local", "relaxed"])
@pytest.mark.parametrize("op", ["intersect", "closest", "close"])
def test_beside_a_capture(mode, op):
    s, last = scene(), scene()
    o, d = W.incoherent_rays(300_007, 1, 1.5)
    o, d = (tuple(torch.from_numpy(np.ascontiguousarray(a[:, k])).cuda() for k in range(3)) for a in (o, d))
    call = {"intersect": lambda: s.intersect(o, d)["t"], "closest": lambda: s.closest_surface(o)["distance"],
            "close": lambda: last.close()}[op]
    ref = call() if op != "close" else None
    if op != "close":
        first = scene()  # leaves blocks that may be in use: launch counters of another stream among them
        with torch.cuda.stream(torch.cuda.Stream()):
            first.intersect(o, d)
            first.closest_surface(o)
        torch.cuda.synchronize()
        first.close()
    x = torch.zeros(1000, device="cuda")
    got, failed = [], []

    def work():
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                got.append(call())
            st.synchronize()
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    torch.cuda.synchronize()
    t = threading.Thread(target=work)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
        x.add_(1)
        t.start()
        t.join()
        x.add_(1)
    for k in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert float(x[0]) == 2.0 * (k + 1)
    assert not failed, failed
    if op != "close":
        assert torch.equal(got[0].view(torch.int64), ref.view(torch.int64))
