"""The rows of whole tiles (csrc/kernels/gemm_tile.hip chain_rows: 256, 192 or 128): which a product takes, and that each gives the
results of a workgroup a tile of 256 rows, bit for bit, also with last tiles that end inside a wave's half or quadrant."""
import pytest
import torch
import torch.nn.functional as F

from githubrepostorag_amd.ops import gemm as G
from githubrepostorag_amd.ops import linear as L
from githubrepostorag_amd.ops._lib import lib


@pytest.mark.parametrize("M,N,K,rows", [(300, 37888, 3584, 128), (900, 37888, 3584, 192), (700, 37888, 3584, 256), (8192, 37888, 3584, 256),
                                        (900, 17920, 1536, 192), (1187, 17920, 1536, 192), (2400, 17920, 1536, 256),
                                        (12000, 3072, 768, 192), (8192, 14336, 3584, 256)])
def test_rule(M, N, K, rows):
    assert lib().grag_gemm_chain_rows(M, N, K, 256) == rows
    us = {r: lib().grag_gemm_chain_ns(M, N, K, r, 256) for r in (256, 192, 128)}
    assert us[rows] == min(us.values()) or us[rows] <= min(us.values()) / 0.98 ** 2


def test_plans(monkeypatch):
    """A streamed tail gives way where whole tiles of fewer rows are clearly shorter, not with deep contractions; the gated unit
    and wide products count the rounds of the tiles that they get."""
    monkeypatch.setattr(G, "_num_cus", lambda: 256)
    G.wide_plan.cache_clear()
    assert G.prefill_plan(320, 37888, 3584, True) == G.prefill_plan(900, 37888, 3584, True) == (1, 0)
    assert G.prefill_plan(512, 37888, 3584, True) == (1, -160) and G.prefill_plan(5000, 3584, 18944)[1] < 0
    assert G.wide_plan(900, 18944, 3584) == (1, 0) and G.wide_plan(300, 18944, 3584) is None  # tiles of 192, of 128 rows
    assert G.chain_fill(300, 37888, 3584) >= L.GLU_FILL[128] > G.chain_fill(300, 37888, 3584, 256)
    assert G.chain_fill(900, 18944, 3584) == 900 * 18944 / (256 * 192 * 2 * 256)
    G.wide_plan.cache_clear()


# last tiles of 1 row, of one row past a wave's first quadrant and half, all but one; ragged columns, a bias that the chain takes
@pytest.mark.gpu
@pytest.mark.parametrize("rows,last", [(r, n) for r in (256, 192, 128) for n in (1, r // 4 + 1, r // 2 + 1, r - 1)])
@pytest.mark.parametrize("N,K", [(14272, 128), (14336, 320)])
def test_rows(dev, monkeypatch, rows, last, N, K):
    M = {256: 768, 192: 576, 128: 384}[rows] + last
    if G._num_cus() == 256:
        assert lib().grag_gemm_chain_rows(M, N, K, 256) == rows
    monkeypatch.setattr(G, "pair_plan", lambda *a: None)  # (the gated unit of these sizes is the small tiles')
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g, device=dev).bfloat16()[:, 8:]
    w, b = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16(), torch.randn(N, generator=g, device=dev).bfloat16()
    assert G.chain_takes(x, w, b)
    z = x.double() @ w.double().T
    zb = z + b.double()
    unit = lambda t: (lambda a, u: F.silu(a) * u)(*(h.T for h in G.deinterleave_gate_up(t.T.contiguous())))  # noqa: E731
    gate, up = z.chunk(2, 1)
    gate = gate.clamp(max=1.0)
    glu = gate * torch.sigmoid(1.702 * gate) * (up.clamp(-1, 1) + 1)
    for f, want in ((lambda: G.gemm(x, w, ksplit=1, sk=0), z), (lambda: G.gemm(x, w, b, act=G.ACT_GELU, ksplit=1, sk=0), F.gelu(zb)),
                    (lambda: G.gemm(x, w, b, act=G.ACT_GELU_TANH, ksplit=1, sk=0), F.gelu(zb, approximate="tanh")),
                    (lambda: G.gemm_silu(x, w, b, ksplit=1, sk=0), unit(zb)), (lambda: G.gemm_silu(x, w, ksplit=1, sk=0), unit(z)),
                    (lambda: G.gemm_glu(x, w, 1.0, 1.702, 1.0), glu)):
        got = f()
        # half an ulp of bf16 of the value, the fp32 sums' rounding (K terms of order 1) and the activation's on top
        torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=2 ** -8 * 0.05)
        prev = G.set_sched(1)  # a workgroup a tile of 256 rows
        try:
            assert torch.equal(got, f())
        finally:
            G.set_sched(prev)
