"""Packed (n,3) tensors reach the kernels through one transposing launch; every other form through torch's copies. Both
give the same columns, and a gradient of positions packed by ray the same vertex gradients as one packed by axis."""
import pytest

torch = pytest.importorskip("torch")

from blazert_amd import Scene, workloads as W  # noqa: E402
from blazert_amd.mirror import mirror_adjoint, mirror_trace  # noqa: E402
from blazert_amd.scene import _columns, _packed_rows  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 255, 1023, 1024, 1025, 300007])
def test_columns(n, dtype):
    base = torch.randn((n + 2, 4), dtype=torch.float64, device="cuda").to(dtype)
    packed = base[:, :3].contiguous()
    other = torch.float32 if dtype == torch.float64 else torch.float64
    forms = [(packed, True), (packed[1:n + 1], True), (packed[:n].requires_grad_(), True), (base[:n, 1:], False),
             (packed[::2], False), (packed.t().contiguous().t()[:n], False), (packed.to(other), False)]
    for x, fast in forms:
        if x.shape[0] > 1:
            assert _packed_rows(x, dtype) == fast
        for k, c in enumerate(_columns(x, dtype)):
            assert c.dtype == dtype and c.is_contiguous() and torch.equal(c, x[:, k].to(dtype))
    with pytest.raises(ValueError):
        _columns(packed, dtype, torch.device("cpu"))


def test_on_another_stream():
    st = torch.cuda.Stream()
    s = Scene()
    s.add_mesh(*W.icosphere(3))
    s.commit()
    o, d = (torch.from_numpy(a).cuda() for a in W.incoherent_rays(4099, 3, 1.5))
    ref = s.intersect(tuple(o.t().contiguous()), tuple(d.t().contiguous()))
    torch.cuda.synchronize()
    got = s.intersect(o, d, stream=st)
    st.synchronize()
    assert all(torch.equal(got[k], ref[k]) for k in ref)


def test_position_gradients():
    v, f = W.icosphere(3)
    s = Scene()
    s.add_mesh(v, f)
    s.commit()
    o, d = (torch.from_numpy(a).cuda() for a in W.incoherent_rays(2049, 4, 1.5))
    out = mirror_trace(s, o, d, 2)
    g = torch.rand((2, 2049, 3), dtype=torch.float64, device="cuda")
    by_ray = mirror_adjoint(s, o, d, out["prim_id"], None, g.permute(2, 0, 1))
    by_axis = mirror_adjoint(s, o, d, out["prim_id"], None, g.permute(2, 0, 1).contiguous())
    assert torch.allclose(by_ray[0], by_axis[0], rtol=1e-12, atol=1e-12)  # summed by atomics, in any order
    assert torch.equal(by_ray[1], by_axis[1]) and torch.equal(by_ray[2], by_axis[2])
