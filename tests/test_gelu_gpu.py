"""GELU of the elementwise kernel and of the tile GEMM's epilogue against 64-bit values over both tails."""
import pytest
import torch

pytestmark = pytest.mark.gpu
dev = "cuda"
bf = torch.bfloat16


def gelu64(z):
    return z * 0.5 * torch.erfc(-z / 2 ** 0.5)


@pytest.mark.parametrize("lo,hi", [(-9.0, -3.0), (-3.0, 3.0), (3.0, 40.0), (-1e-3, 1e-3)])
def test_bias_act_gelu(lo, hi):
    from githubrepostorag_amd.ops.elementwise import ACT_GELU, bias_act

    x = torch.linspace(lo, hi, 4096, device=dev).to(bf)[None]
    y, r = bias_act(x.clone(), None, ACT_GELU).double(), gelu64(x.double())
    # bf16 rounding of the result (half a unit in its last place of 8 bits, 2^-8) plus the fit's 3.8e-7
    assert ((y - r).abs() <= r.abs() * 2 ** -8 + 4e-7).all()


def test_bias_act_gelu_special():
    from githubrepostorag_amd.ops.elementwise import ACT_GELU, bias_act

    inf, nan = float("inf"), float("nan")
    x = torch.tensor([[inf, -inf, nan, 0.0, 3e38, -3e38, 100.0, -100.0]], device=dev).to(bf)
    y = bias_act(x.clone(), None, ACT_GELU).float().cpu()[0]
    assert y[0] == inf and y[1].isnan() and y[2].isnan()
    assert y[3:].tolist() == [0.0, x[0, 4].item(), 0.0, 100.0, 0.0]


@pytest.mark.parametrize("M", [256, 300])
def test_gemm_gelu_tails(M):
    from githubrepostorag_amd.ops import gemm as G

    # a product with one term a row and column: its pre-activation is exact in fp32
    K, N = 128, 256
    x = torch.zeros(M, K, device=dev, dtype=bf)
    w = torch.zeros(N, K, device=dev, dtype=bf)
    x[:, 5] = torch.linspace(-3, 3, M, device=dev).to(bf)
    w[:, 5] = torch.linspace(-3, 3, N, device=dev).to(bf)
    r = gelu64(x[:, 5].double()[:, None] * w[:, 5].double()[None])
    y = G.gemm(x, w, None, act=G.ACT_GELU, ksplit=1).double()
    assert ((y - r).abs() <= r.abs() * 2 ** -8 + 4e-7).all()
