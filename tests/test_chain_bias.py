"""Plans that count on whole tiles of 192 or 128 rows (ops/gemm.py prefill_plan, wide_plan): only where the launcher has such tiles
(csrc/kernels/gemm_tile.hip chain_ok), which refuses a bias that is too wide for its LDS or not on 16 bytes."""
import pytest
import torch
import torch.nn.functional as F

from githubrepostorag_amd.ops import gemm as G
from githubrepostorag_amd.ops import linear as L
from githubrepostorag_amd.ops._lib import lib


def test_plans(monkeypatch):
    monkeypatch.setattr(G, "_NCU", [256])
    most = lib().grag_gemm_chain_bias()
    assert 8192 <= most < 18944
    x, w, wide = torch.empty(900, 64), torch.empty(most, 64), torch.empty(most + 8, 64)
    assert G.chain_fits(x, w, torch.empty(most)) and G.chain_fits(x, wide) and not G.chain_fits(x, wide, torch.empty(most + 8))
    b = torch.empty(most + 8, dtype=torch.bfloat16)
    assert G.chain_takes(x, w, b[:most]) and not G.chain_takes(x, w, b[4:most + 4]) and G.chain_fits(x, w, b[4:most + 4])
    out = torch.empty(900, most + 8, dtype=torch.bfloat16)
    assert G.chain_takes(x, w, None, out[:, 8:]) and not G.chain_takes(x, w, None, out[:, 4:most + 4])
    # 900 x 18944: 296 tiles of 256 rows fill half of two rounds, 370 of 192 rows two thirds
    assert G.wide_plan(900, 18944, 3584) == (1, 0) and G.wide_plan(900, 18944, 3584, False) is None
    assert L.kernel_for(900, 18944, 3584) == "tile_prefill" and L.kernel_for(900, 18944, 3584, chain_ok=False) == "library"
    assert G.wide_plan(2405, 18944, 3584, False) == (1, 0)  # full rounds of 256 rows
    # a streamed tail stays where whole tiles would have 256 rows
    assert G.prefill_plan(300, 37888, 3584, True) == G.schedule(300, 37888, 3584, True) == (1, 0)
    assert G.prefill_plan(300, 37888, 3584, True, False)[1] < 0 and G.schedule(300, 37888, 3584, True, False)[1] < 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,own", [(900, 18944, 3584, False), (1200, 14336, 2048, True), (2405, 18944, 3584, True)])
def test_plain(dev, monkeypatch, M, N, K, own):
    """A biased product outside the measured table, its fill that of the tiles that it gets."""
    g = torch.Generator(device=dev).manual_seed(M + N)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    x, w, b = r(M, K).bfloat16(), (r(N, K) * K ** -0.5).bfloat16(), r(N).bfloat16()
    took = []
    monkeypatch.setattr(G, "gemm", lambda *a, _f=G.gemm, **k: took.append(k) or _f(*a, **k))
    y = L.linear(x, w, b)
    assert bool(took) == own
    # the result's rounding to bf16's 8 bits (the library's before the bias is added as well), fp32 sums of K products
    torch.testing.assert_close(y.double(), x.double() @ w.double().T + b.double(), rtol=2 ** -7, atol=2 ** -7 * 0.05)


@pytest.mark.gpu
@pytest.mark.parametrize("at", [None, 0, 4])
def test_gated(dev, monkeypatch, at):
    """A gated unit's streamed tail: whole tiles of 128 rows without a bias; with one as swept, on 16 bytes or not."""
    if G._num_cus() != 256:
        pytest.skip("the table's streamed tails are those of 256 CUs")
    M, N, K = 300, 37888, 3584
    g = torch.Generator(device=dev).manual_seed(7)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    x, w = r(M, K).bfloat16(), (r(N, K) * K ** -0.5).bfloat16()
    b = None if at is None else r(N + 8).bfloat16()[at:at + N]
    took = []
    monkeypatch.setattr(G, "_launch", lambda *a, _f=G._launch: took.append(a[-2:]) or _f(*a))
    got = G.gemm_silu(x, w, b)
    assert len(took) == 1 and (took[0] == (1, 0)) == (at is None)
    z = x.double() @ w.double().T + (0 if b is None else b.double())
    gate, up = G.deinterleave_gate_up(z.T.contiguous())
    torch.testing.assert_close(got.double(), (F.silu(gate) * up).T, rtol=2 ** -8, atol=2 ** -8 * 0.05)
