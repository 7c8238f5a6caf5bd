"""minGRU over long portions (csrc/kernels/seqmix.hip, mingru_chunk_kernel): chunks of 32 tokens, eight of them fetched at a time, and
the chunks before folded eight at a time, against the recurrence in fp64."""
import pytest
import torch

from githubrepostorag_amd.ops.recurrent import mingru_scan
from test_pubulix import _meta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W", [1, 257, 512])
@pytest.mark.parametrize("lens", [(33,), (64, 7, 1), (289, 40, 65), (32 * 9, 32 * 8 + 1, 8), (3, 1000)])
def test_chunks(lens, W, dtype):
    g = torch.Generator().manual_seed(sum(lens) + W)
    rnd = lambda *s: torch.randn(*s, generator=g)
    T, n = sum(lens), len(lens)
    proj = rnd(T, 3 * W + 5).to(dtype)
    bz, bx, st = rnd(W) - 1, rnd(W), rnd(n + 1, W)
    ctx = [l + (9 if s % 2 == 0 else 0) for s, l in enumerate(lens)]  # (every second portion starts its sequence)
    slots = list(range(n, 0, -1))
    state = st.clone().cuda()
    y = mingru_scan(proj.cuda(), 2, 2 + W, 3 + 2 * W, bz.cuda(), bx.cuda(), state, _meta("cuda", lens, ctx, slots), W)
    x = proj.double()
    z, u, gate = torch.sigmoid(x[:, 2:2 + W] + bz), x[:, 2 + W:2 + 2 * W] + bx, torch.nn.functional.silu(x[:, 3 + 2 * W:3 + 3 * W])
    cand = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    at = 0
    for s, l in enumerate(lens):
        S = st[slots[s]].double() if ctx[s] > l else torch.zeros(W, dtype=torch.float64)
        want = []
        for t in range(at, at + l):
            S = (1 - z[t]) * S + z[t] * cand[t]
            want.append(S * gate[t])
        want = torch.stack(want)
        at += l
        # a state is a mean of what came before: each token adds a few roundings of it, of which the weights 1 - z forget those
        # before; a chunk's product and sum twice that.  64 ulp of the largest number, and the output's own rounding
        big = max(float(cand.abs().max()), float(st.abs().max()))
        assert (state[slots[s]].cpu().double() - S).abs().max() < 64 * 2 ** -24 * big
        tol = (64 * 2 ** -24 + (2 ** -8 if dtype == torch.bfloat16 else 0)) * big * float(gate.abs().max())
        assert (y[at - l:at].cpu().double() - want).abs().max() < tol
    assert torch.equal(state[0].cpu(), st[0])
