"""Row passes of the hybrid layers in wide accesses (dynamic-tanh residual, gated RMSNorm of wide groups, rotary + K/V store
with value norms) at the edges of their forms, against the fp32 CPU paths of the same operations."""
import pytest
import torch

pytestmark = pytest.mark.gpu
dev = "cuda"
bf = torch.bfloat16


def rnd(g, *s):
    return torch.randn(*s, generator=g)


@pytest.mark.parametrize("T,H", [(1, 4), (1023, 36), (8192, 36), (4098, 1028), (3, 3584), (5, 6)])
@pytest.mark.parametrize("post,rows,vec,pre", [(1, 1, 1, 1), (1, 0, 0, 1), (0, 0, 1, 0), (0, 1, 0, 1), (1, 0, 1, 0), (0, 0, 0, 1)])
def test_dyt_residual(T, H, post, rows, vec, pre):
    from githubrepostorag_amd.ops.norm import dyt_residual

    g = torch.Generator().manual_seed(T + H)
    r, y = rnd(g, T, H), rnd(g, T, H).to(bf) * 3
    tri = lambda a: (a, rnd(g, H), rnd(g, H))
    po, pr = tri(0.7), tri(-1.3)
    ar, av = rnd(g, T, H), rnd(g, H)
    on = lambda t: t if t is None else (t[0], t[1].to(dev), t[2].to(dev))
    r1 = r.clone().to(dev)
    h = dyt_residual(r1, y.to(dev) if post else None, on(po if post else None), ar.to(dev) if rows else None,
                     av.to(dev) if vec else None, on(pr if pre else None))
    x = r.double()
    if post:
        x = x + torch.tanh(po[0] * y.double()) * po[1].double() + po[2].double()
    x = x + (ar.double() if rows else 0) + (av.double() if vec else 0)
    # a handful of fp32 roundings of terms of a few units
    assert (r1.cpu().double() - x).abs().max() <= 4e-6
    if pre:
        o = torch.tanh(pr[0] * x) * pr[1].double() + pr[2].double()
        assert ((h.cpu().double() - o).abs() <= o.abs() * 2 ** -8 + 4e-5).all()  # bf16 rounding of the result
    else:
        assert h is None


def test_dyt_residual_special():
    from githubrepostorag_amd.ops.norm import dyt_residual

    inf, nan = float("inf"), float("nan")
    y = torch.tensor([[inf, -inf, nan, 0.0, 1e-30, -1e30, 1e30, 0.02]], device=dev)
    r = torch.zeros_like(y)
    one, zero = torch.ones(8, device=dev), torch.zeros(8, device=dev)
    dyt_residual(r, y, (1.0, one, zero), out_dtype=torch.float32)
    v = r.cpu()[0]
    assert v[2].isnan() and v[[0, 1, 3, 5, 6]].tolist() == [1.0, -1.0, 0.0, -1.0, 1.0]
    assert abs(v[4].item() - 1e-30) < 1e-36 and abs(v[7].item() - 0.0199973340) < 1e-8
