"""Small tiles for plain products of 1152 to 1536 deep (ops/gemm.py, pair_plan): where the line lies, and the products there against
fp32."""
import pytest
import torch

from githubrepostorag_amd.ops import gemm as G
from githubrepostorag_amd.ops import linear as L


def test_rule(monkeypatch):
    monkeypatch.setattr(G, "_num_cus", lambda: 256)
    G.pair_plan.cache_clear()
    at = lambda M, N, K: G.pair_plan(M, N, K)
    assert [at(M, 1536, 1536) for M in (260, 384, 385, 1344, 1365)] == [None, 3, 3, 3, None]  # 120, 144, 168, 504, 528 tiles
    assert [at(400, 2304, K) for K in (1088, 1152, 1536, 1600)] == [None, 3, 3, None]
    assert [at(M, 4608, 1280) for M in (256, 257, 448, 449)] == [None, 3, 3, None]
    assert L.kernel_for(400, 2304, 1152) == "pair" and L.kernel_for(400, 2304, 1152, pair_ok=False) != "pair"
    G.pair_plan.cache_clear()


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", [(257, 2304, 1152), (330, 1536, 1536), (1301, 1512, 1472), (440, 4104, 1216), (257, 6144, 1536)])
def test_products(M, N, K, bias):
    g = torch.Generator().manual_seed(M)
    x, w = (torch.randn(r, K, generator=g).to(torch.bfloat16).cuda() for r in (M, N))
    b = torch.randn(N, generator=g).to(torch.bfloat16).cuda() if bias else None
    assert G.pair_plan(M, N, K) == 3 and L.kernel_for(M, N, K, G.supported(x, w), x.device) == "pair"
    y = L.linear(x, w, b).float()
    want = x.float() @ w.float().T + (0 if b is None else b.float())
    # the sum's own rounding to 8 bits, and fp32 sums of K products in another order
    assert ((y - want).abs() <= want.abs() * 2 ** -8 + K * 2 ** -24 * want.abs().max()).all()
    part = L.linear(x[:, :K], w, b)  # the same rows behind a wider stride
    wide = torch.cat([x, x], 1)
    assert torch.equal(L.linear(wide[:, :K], w, b), part)
    xg = x.clone().requires_grad_()
    L.linear(xg, w, b).float().sum().backward()  # (a gradient goes the library's way)
    assert xg.grad is not None
