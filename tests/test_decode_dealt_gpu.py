"""Decode products whose column tiles are more than half the CUs and too few for all (ops/gemm.py dec_plan: their units dealt
evenly to every CU) against fp64: the narrowest and the widest such product of the chip, 1 to 128 rows, one 64-deep round of K and
several."""
import pytest
import torch

from githubrepostorag_amd.ops.gemm import (EPI_SILU, _num_cus, dec_glu_plan, dec_own_plan, dec_plan, dec_wide, gemm_decode, gemm_decode_glu,
                                          interleave_gate_up)
from githubrepostorag_amd.ops import gemm as G
from githubrepostorag_amd.ops import linear as L


@pytest.mark.gpu
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


@pytest.mark.gpu
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


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("K", [512, 1280])
@pytest.mark.parametrize("share", [0.01, 0.625])
def test_dealt_one_idle(dev, share, K, M):
    """4 - 5 units of 32 rows to 5 waves: the wave without one stores nothing."""
    ncu = _num_cus()
    N = 64 * int((2 + share / 2) * ncu)
    assert dec_plan(M, N, K, True) == (2, 5, 2, 1, ncu)
    g = torch.Generator(device=dev).manual_seed(M + K)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    wg, wu = ((torch.randn(N // 2, K, generator=g, device=dev) * K ** -0.5).bfloat16() for _ in range(2))
    a, b = x.double() @ wg.double().T, x.double() @ wu.double().T
    want = a * torch.sigmoid(a) * b
    got = gemm_decode(x, interleave_gate_up(wg, wu), epi=EPI_SILU).double()
    # bf16's rounding of the result; fp32 sums and exponentials of numbers of about 1
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-5 * (1 + b.abs())).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 64, 65, 128])
@pytest.mark.parametrize("width", [1.0625, 2.25, 2.5])
@pytest.mark.parametrize("kind", ["plain", "silu", "glu"])
def test_fine_units(dev, kind, width, M):
    """Units of 16 rows (8 gate and 8 up ones of a gated unit): 2 - 5 a workgroup, and the narrowest and widest such product."""
    ncu, K = _num_cus(), 320 if kind == "glu" else 256
    N = int(width * ncu) // 2 * 64
    plan = (-(-M // 16) if M <= 32 else 4 if M <= 64 else 8, 5, 1, 1, ncu)
    g = torch.Generator(device=dev).manual_seed(M + N)
    x = torch.randn(M, K + 8, generator=g, device=dev).bfloat16()[:, 8:]
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    z = x.double() @ w.double().T
    if kind == "plain":
        b = torch.randn(N, generator=g, device=dev).bfloat16()
        got, want, fp32 = gemm_decode(x, w, b, plan=plan), z + b.double(), 1e-5
    elif kind == "silu":
        b = torch.randn(N, generator=g, device=dev).bfloat16()
        a, u = (z + b.double()).chunk(2, 1)
        got = gemm_decode(x, interleave_gate_up(*w.chunk(2)), interleave_gate_up(*b[:, None].chunk(2))[:, 0].contiguous(), epi=EPI_SILU,
                          plan=plan)
        want, fp32 = a * torch.sigmoid(a) * u, 2e-5 * (1 + u.abs())
    else:
        a, u = z.chunk(2, 1)
        got = gemm_decode_glu(x, w, (*plan[:3], ncu), 1.5, 1.702, 1.0)
        a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5)
        want, fp32 = a * torch.sigmoid(1.702 * a) * (u + 1), 1e-4
    assert got.shape == want.shape
    # bf16's rounding of the result; fp32 sums and exponentials of numbers of about 1
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + fp32).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,K,taken", [(1, 8960, 256, True), (33, 8192, 512, True), (128, 4096, 256, True), (32, 4096, 256, False),
                                         (129, 8960, 256, False), (64, 8960, 320, False)])
def test_glu_linear_decode(dev, M, F, K, taken, monkeypatch):
    seen = []
    orig = G.gemm_decode_glu
    monkeypatch.setattr(G, "gemm_decode_glu", lambda *a: seen.append(1) or orig(*a))
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(2 * F, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    y = L.glu_linear(x, w, 7.0).double()
    assert bool(seen) == taken
    a, u = (x.double() @ w.double().T).chunk(2, 1)
    a, u = a.clamp(max=7.0), u.clamp(-7.0, 7.0)
    s = torch.sigmoid(1.702 * a)
    # two launches round gate and up as well: 2^-8 of each, times the unit's slopes
    slope = (s + 1.702 * a * s * (1 - s)).abs() * (u + 1).abs() * a.abs() + (a * s).abs() * u.abs()
    assert ((y - a * s * (u + 1)).abs() <= 2 ** -8 * ((a * s * (u + 1)).abs() + (0 if taken else 1.01) * slope) + 1e-4).all()
    seen.clear()
    with torch.enable_grad():  # where a gradient is asked for, the product goes the way it went
        L.glu_linear(x.requires_grad_(), w, 7.0)
    assert not seen


def test_rules(monkeypatch):
    monkeypatch.setattr(G, "_num_cus", lambda: 256)
    assert dec_plan(64, 17920, 1536, True) == (4, 5, 1, 1, 256)     # 560 units of 32: 3 at most, 1120 of 16: 5
    assert dec_plan(64, 37888, 3584, True) == (4, 5, 2, 1, 256)     # 1184: 5, 2368: 10
    assert dec_plan(100, 18944, 3584) == (8, 5, 1, 1, 256)
    assert dec_own_plan(64, 8192, 1536) == (4, 5, 1, 1, 256) and dec_plan(64, 8192, 1536) == (4, 4, 2, 3)
    assert dec_own_plan(64, 4096 - 128, 1536)[3] > 1 and dec_own_plan(64, 8192, 2560)[3] > 1 and dec_own_plan(32, 8192, 1536)[3] > 1
    assert dec_wide(1, 18944, 3584) and dec_wide(32, 18944, 3584) and dec_wide(16, 32768, 3584) and not dec_wide(17, 32768, 3584)
    assert not dec_wide(1, 152064, 3584) and not dec_wide(33, 18944, 3584) and not dec_wide(1, 8192, 1536)
    assert dec_glu_plan(1, 8960, 1536) == (1, 5, 1, 256) and dec_glu_plan(100, 18944, 3584) == (8, 5, 2, 256)
    assert dec_glu_plan(1, 3776, 3584) is None and dec_glu_plan(129, 18944, 3584) is None
    assert L.kernel_for(1, 18944, 3584) == "decode" and L.kernel_for(1, 18944, 3584, wide_ok=False) != "decode"
    for p, N in ((dec_plan(64, 17920, 1536, True), 17920), (dec_own_plan(64, 8192, 1536), 8192), (dec_plan(1, 18944, 3584), 18944)):
        assert -(-(N // 16) // p[4]) <= p[1]  # what the launcher takes


@pytest.mark.gpu
@pytest.mark.parametrize("N", [32 * 327691, 32 * 262149])
def test_dealt_many(dev, N):
    """More than 65536 workgroups that the units do not divide into: 65539 of 4 - 5 units, 65538 of 3 - 4."""
    K, gs = 64, 65539 if N == 32 * 327691 else 65538
    g = torch.Generator(device=dev).manual_seed(gs)
    x = torch.randn(2, K, generator=g, device=dev).bfloat16()
    w = torch.randn(N, K, generator=g, device=dev, dtype=torch.bfloat16)
    got = gemm_decode(x, w, plan=(1, 5, 2, 1, gs)).float()
    want = x.float() @ w.float().T
    # bf16's rounding of the result, and fp32 sums of 64 products of about 1 in another order
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 64 * 2 ** -23 * 16).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 64, 128])
@pytest.mark.parametrize("silu", [False, True])
def test_packed_takes_the_plan(dev, silu, M):
    """Packed weights with the product's own plan, also one in units of 16 rows, which only natural weights have."""
    ncu, K = _num_cus(), 512
    N = 64 * (9 * ncu // 8)  # 2.25 units of 32 a CU
    plan = dec_plan(M, N, K, silu)
    assert plan[2:] == (1, 1, ncu)
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    epi = EPI_SILU if silu else G.EPI_STORE
    packed = G.DecPacked(w, silu)
    want = gemm_decode(x, w, epi=epi, plan=G.dec_coarse(plan, N))  # the same sums in the same order
    assert torch.equal(gemm_decode(x, w, epi=epi, plan=plan, packed=packed), want)
    assert torch.equal(gemm_decode(x, w, epi=epi, packed=packed), want)


@pytest.mark.gpu
def test_packed_takes_the_own_plan(dev):
    """A plan with more workgroups than the product has units of 32 rows."""
    ncu, K, M = _num_cus(), 512, 64
    N = 64 * (3 * ncu // 8)  # 1.5 units of 16 a CU, 0.75 of 32
    plan = G.dec_own_plan(M, N, K)
    assert plan[1:] == (5, 1, 1, ncu) and G.dec_coarse(plan, N)[1:] == (5, 2, 1, N // 32)
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    assert torch.equal(gemm_decode(x, w, plan=plan, packed=G.DecPacked(w)), gemm_decode(x, w, plan=G.dec_coarse(plan, N)))
