"""Decode products whose column tiles are more than half the CUs and too few for all (ops/gemm.py dec_plan: their units dealt
evenly to every CU) against fp64: the narrowest and the widest such product of the chip, 1 to 128 rows, one 64-deep round of K and
several."""
import pytest
import torch

from githubrepostorag_amd.ops.gemm import EPI_SILU, _num_cus, dec_plan, gemm_decode, interleave_gate_up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [256, 1280])
@pytest.mark.parametrize("M", [1, 17, 64, 128])
@pytest.mark.parametrize("wide", [False, True])
def test_dealt(dev, wide, M, K):
    ncu = _num_cus()
    N = 128 * (4 * ncu // 5 if wide else ncu // 2 + 1)
    assert dec_plan(M, N, K)[3:] == (1, ncu)
    g = torch.Generator(device=dev).manual_seed(M + K)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    b = torch.randn(N, generator=g, device=dev).bfloat16()
    want = x.double() @ w.double().T + b.double()
    # the result's rounding to bf16's 8 bits, and fp32 sums of K products of about 1 / sqrt(K) each
    assert ((gemm_decode(x, w, b).double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all()


@pytest.mark.parametrize("M", [1, 33, 128])
@pytest.mark.parametrize("extra", [2, 48, 1024])
def test_dealt_gated(dev, extra, M):
    """SwiGLU over 5-wave workgroups of 1 - 5 units each, so that most have waves without one."""
    ncu, K = _num_cus(), 512
    N = 32 * (ncu + extra)
    assert dec_plan(M, N, K, True)[3:] == (1, ncu)
    g = torch.Generator(device=dev).manual_seed(M + extra)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    wg, wu = ((torch.randn(N // 2, K, generator=g, device=dev) * K ** -0.5).bfloat16() for _ in range(2))
    a, b = x.double() @ wg.double().T, x.double() @ wu.double().T
    want = a * torch.sigmoid(a) * b
    got = gemm_decode(x, interleave_gate_up(wg, wu), epi=EPI_SILU).double()
    # bf16's rounding of the result; fp32 sums and exponentials of numbers of about 1
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-5 * (1 + b.abs())).all()
