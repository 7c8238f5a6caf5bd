"""Split-K reduce + residual + RMSNorm in one launch, few rows at four columns a thread, against 64-bit sums: widths around a
block's lanes and both forms' limits, every pass length of planes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [8, 264, 2048, 2056, 3584, 4096, 4104, 8192, 8200])
@pytest.mark.parametrize("T,S", [(1, 1), (3, 9), (17, 2), (256, 7), (257, 3), (2, 17)])
def test_splitk_add_rmsnorm(H, T, S):
    from githubrepostorag_amd.ops._lib import call, ptr

    g = torch.Generator(device="cuda").manual_seed(H + T)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    ws, res, w = rnd(S, T, H), rnd(T, H).bfloat16(), rnd(H).bfloat16()
    x = res.double() + ws.double().sum(0)
    out, r1 = torch.empty_like(res), res.clone()
    call("grag_splitk_add_rmsnorm", ptr(ws), S, ptr(r1), ptr(w), ptr(out), T, H, 1e-6)
    # the stream: bf16 rounding of the sum, and S fp32 additions of a few units
    assert ((r1.double() - x).abs() <= x.abs() * 2 ** -8 + S * 2e-6).all()
    h = r1.double()
    y = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    assert ((out.double() - y).abs() <= y.abs() * 2 ** -8 + 1e-5).all()
