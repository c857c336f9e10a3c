"""Vertex normals of a device commit equal the host's bit for bit (each vertex sums its faces' shares in face order): fans
around the lengths at which the device changes its way of summing and beyond what it sums at all, degenerate faces, faces
naming a vertex twice, unused vertices; and inputs the device build leaves to the host."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import GEOM_TRIANGLES, Scene, workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def fan(m, seed=1):
    """m faces around vertex 0, listed in random order, each starting at a random corner."""
    r = np.random.default_rng(seed)
    a = np.linspace(0, 2 * np.pi, m, endpoint=False)
    v = np.concatenate([[[0.1, 0.0, 0.3]], np.stack([np.cos(a), np.sin(a), 0.2 * r.standard_normal(m)], 1)])
    f = np.stack([np.zeros(m, int), 1 + np.arange(m), 1 + (np.arange(m) + 1) % m], 1)[r.permutation(m)]
    f = np.stack([np.roll(x, r.integers(3)) for x in f])
    return v, f.astype(np.uint32)


def meshes():
    yield "sphere", W.icosphere(4)
    for m in (3, 63, 64, 65, 300, 4096, 4097):
        yield f"fan{m}", fan(m)
    v, f = W.icosphere(3)
    odd = f.copy()
    odd[::7, 1] = odd[::7, 0]          # a vertex twice in a face
    odd[::11] = odd[::11, :1]          # a point
    yield "degenerate", (np.concatenate([v, v * 2]), odd)
    for name, x in (("nan", np.nan), ("inf", np.inf), ("-0", -0.0)):
        w = v.copy()
        w[5, 1] = x
        yield name, (w, f)


@pytest.mark.parametrize("name,mesh", list(meshes()), ids=[n for n, _ in meshes()])
def test_normals_of_host_and_device_commits(dev, name, mesh):
    v, f = mesh
    r = np.random.default_rng(2)
    n = 20000
    d = r.standard_normal((n, 3))
    o = r.uniform(-1, 1, (n, 3)) * [1, 1, 0] - 3 * d
    hits = []
    for device in (False, True):
        s = Scene()
        s.add_mesh(v, f)
        s.commit(device=device)
        on_device = s.build_stats(GEOM_TRIANGLES)["built_on_device"]
        if not device or name == "inf":
            assert on_device == 0
        elif name not in ("nan", "-0"):  # whether these reach a box depends on the corner they are at
            assert on_device == 1
        hits.append(s.intersect(torch.from_numpy(o).to(dev), torch.from_numpy(d).to(dev), normals=True))
    assert int((hits[0]["prim_id"] != -1).sum()) > 1000
    for k in hits[0]:
        a, b = (h[k].view(torch.int64) if h[k].dtype == torch.float64 else h[k] for h in hits)
        assert torch.equal(a, b), k
