"""The experts' grouped GEMM at decode's row counts (csrc/kernels/moe.hip moe_gemm_stream_kernel, and the 128-row tiles that
take over where the experts fill the chip) against a plain fp32 product per pair: row counts around the tiles of 16, 32 and 64
rows, none among them, contractions shorter than the waves' blocks, columns past the last whole tile."""
import math

import pytest
import torch

from githubrepostorag_amd.ops.moe import moe_experts

pytestmark = pytest.mark.gpu

FEW = [0, 1, 16, 17, 3, 0, 2, 5, 1, 2]           # at most 6 a mean expert
SOME = [0, 1, 32, 33, 31, 16, 40, 24]            # at most 26
MANY = [0, 64, 65, 20, 63, 33, 1]                # at most 48
EVEN = [13] * 16                                 # with 24 column tiles an expert: the 128-row tiles


@pytest.mark.parametrize("counts,W,F", [(c, W, F) for c in (FEW, SOME, MANY) for W, F in ((64, 128), (192, 64), (328, 392), (640, 1088))]
                         + [(EVEN, 64, 3072), ([1], 256, 512), ([0, 1, 0, 0], 448, 192)])
@pytest.mark.parametrize("unit,limit", [("glu", None), ("glu", 2.0), ("relu2", None)])
def test_moe_stream(counts, W, F, unit, limit):
    g = torch.Generator().manual_seed(W + F + len(counts))
    E, top = len(counts), 1 if sum(counts) % 2 else 2
    flat = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)] + [torch.tensor([-1, E])])
    flat = flat[torch.randperm(len(flat), generator=g)]
    flat = flat[: len(flat) // top * top]
    T = len(flat) // top
    ids = flat.view(T, top).to(torch.int32)
    h = torch.randn(T, W, generator=g).bfloat16()
    wgu = (torch.randn(E, F if unit == "relu2" else 2 * F, W, generator=g) * W ** -0.5).bfloat16()
    wd = (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16()
    kw = dict(unit=unit) if unit == "relu2" else dict(limit=limit, alpha=1.3 if limit else 1.0, shift=0.5 if limit else 0.0)
    wide = torch.zeros(T, W + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, :W] = h.cuda()
    got = moe_experts(wide[:, :W], ids.cuda(), wgu.cuda(), wd.cuda(), **kw).float().cpu()
    want = moe_experts(h, ids, wgu, wd, **kw).float()
    ok = (ids >= 0) & (ids < E)
    # both round the unit's output and the result to bf16 (2^-8 apart at most where fp32 sums of another order fall on
    # different sides); the second product averages the first rounding over F terms
    err = (got - want)[ok].abs().max() / want[ok].abs().max()
    assert err < 2 ** -7, err
    assert (got - want)[ok].norm() / want[ok].norm() < 5e-3


@pytest.mark.parametrize("rows", [1, 20, 60, 300])  # the stream, its larger tile, the 128-row and the 256-row tiles
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_infinite_gate(rows, dtype):
    """A gate whose sum leaves fp32 upwards gives an infinite unit."""
    W = F = 128
    h = torch.ones(rows, W, dtype=dtype, device="cuda")
    wgu = torch.full((1, 2 * F, W), 2.0 ** -7, dtype=dtype, device="cuda")
    wgu[0, 5] = 3e38
    wd = torch.ones(1, W, F, dtype=dtype, device="cuda")
    y = moe_experts(h, torch.zeros(rows, 1, dtype=torch.int32, device="cuda"), wgu, wd)
    assert (y == float("inf")).all()


def test_unit_in_fp32():
    """fp32 experts: gates down to -80 (each a product of one term, and the second matrix the identity, so that only the unit
    rounds: the exponential, sum, quotient and product by an ulp or half of 1.2e-7 each)."""
    n = W = F = 256
    g = torch.cat([torch.linspace(-80, -20, n // 2), torch.linspace(-20, 20, n // 2)])
    h = torch.zeros(n, W)
    h[:, 0], h[:, 1] = g, 1.0
    wgu = torch.zeros(1, 2 * F, W)
    wgu[0, :F, 0], wgu[0, F:, 1] = 1.0, torch.linspace(0.5, 3.0, F)
    y = moe_experts(h.cuda(), torch.zeros(n, 1, dtype=torch.int32, device="cuda"), wgu.cuda(), torch.eye(F)[None].cuda())
    want = (g.double() * torch.sigmoid(g.double()))[:, None] * wgu[0, F:, 1].double()
    err = (y[:, 0].double().cpu() - want).abs() / want.abs()
    assert err.max() < 5e-7, err.max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_unit_of_large_negative_gates(dtype):
    """Where e^-g leaves fp32 (g < -88.7) the unit is 0, as the quotient by infinity is; just above, a number below 1e-35."""
    g = torch.tensor([-86.0, -88.0, -88.5, -89.0, -90.0, -100.0, -128.0, -1e4, -1e30, 1.0])
    n, W, F = len(g), 128, 128
    h = torch.zeros(n, W, dtype=dtype)
    h[:, 0], h[:, 1] = g, 1.0
    wgu = torch.zeros(1, 2 * F, W, dtype=dtype)
    wgu[0, :F, 0], wgu[0, F:, 1] = 1.0, 2.0
    y = moe_experts(h.cuda(), torch.zeros(n, 1, dtype=torch.int32, device="cuda"), wgu.cuda(), torch.eye(F, dtype=dtype)[None].cuda())
    y = y[:, :F].float().cpu()
    assert (y[:-1].abs() < 1e-35).all() and ((y[-1] - 2 / (1 + math.exp(-1))).abs() < 2 ** -7).all()


@pytest.mark.parametrize("E", [63, 64, 65, 130])
def test_many_experts(E):
    """Row tiles of experts past the first 64, and of the last."""
    g = torch.Generator().manual_seed(E)
    W, F, T = 64, 64, 40
    ids = torch.randint(0, E, (T, 2), generator=g, dtype=torch.int32)
    ids[:20, 0] = E - 1
    h = torch.randn(T, W, generator=g).bfloat16()
    wgu, wd = ((torch.randn(E, n, 64, generator=g) / 8).bfloat16() for n in (2 * F, W))
    got = moe_experts(h.cuda(), ids.cuda(), wgu.cuda(), wd.cuda()).float().cpu()
    want = moe_experts(h, ids, wgu, wd).float()
    assert (got - want).abs().max() / want.abs().max() < 2 ** -7 and (got - want).norm() / want.norm() < 5e-3  # (as above)
