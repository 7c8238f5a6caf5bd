"""Selective scan: whole portions of one step are walked longest first, four tokens at a time, the step sizes' rows shared by a
workgroup's waves.  Each portion's output and state have to be those of a step of that portion alone, bit for bit; and the
rule that cuts portions into chunks."""
import pytest
import torch

from githubrepostorag_amd.ops import recurrent as R
from test_pubulix import _meta


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inner,N,rank", [(64, 16, 24), (70, 13, 130), (200, 16, 300), (33, 37, 3)])
@pytest.mark.parametrize("nseq", [1, 5, 64, 65])
def test_portions_are_those_of_a_step_alone(nseq, inner, N, rank, dtype, monkeypatch):
    monkeypatch.setattr(R, "CHAN_SCAN_WGS", 1)  # (never cut)
    g = torch.Generator().manual_seed(nseq + inner)
    lens = [int(n) for n in torch.randint(2, 120, (nseq,), generator=g)]
    if nseq > 2:
        lens[1], lens[2], lens[-1] = lens[0], 16, 17
    ctx = [n + (7 if s % 3 else 0) for s, n in enumerate(lens)]  # (every third portion starts its sequence)
    slots = torch.randperm(nseq, generator=g).tolist()
    width, T = rank + 2 * N, sum(lens)
    rnd = lambda *s: torch.randn(*s, generator=g)
    xc, proj, low = rnd(T, inner).to(dtype).cuda(), rnd(T, 2 * inner).to(dtype).cuda(), rnd(T, -(-width // 8) * 8).to(dtype).cuda()
    wdt = R.pad_step_matrix((rnd(inner, rank) / rank ** 0.5).to(dtype)).contiguous().cuda()
    dtb, A, skip = (rnd(inner) - 2).cuda(), -torch.exp(rnd(inner, N)).cuda(), rnd(inner).cuda()
    st = rnd(nseq, inner, N).cuda()
    run = lambda x, l, p, state, *m: R.selective_scan(x, l, wdt, rank, dtb, A, skip, p, inner, state, _meta("cuda", *m))
    before = st.clone()
    y = run(xc, low, proj, st, lens, ctx, slots)
    for s in sorted(range(nseq), key=lambda s: lens[s])[-6:] + [0]:
        at, to = sum(lens[:s]), sum(lens[:s + 1])
        mine = before.clone()
        want = run(xc[at:to].clone(), low[at:to].clone(), proj[at:to].clone(), mine, [lens[s]], [ctx[s]], [slots[s]])
        assert torch.equal(y[at:to], want) and torch.equal(st[slots[s]], mine[slots[s]]), s


def test_rule_for_chunks():
    for inner in (64, 1536, 3584, 8192):
        for nseq, tokens, longest in ((1, 65, 65), (1, 9000, 9000), (2, 300, 290), (8, 4000, 700), (16, 5000, 480), (40, 9000, 8000)):
            c = R._chan_chunk(nseq, longest, inner, tokens)
            assert c in (0, 64, 128, 256) and (c == 0 or c < longest)
    assert R._chan_chunk(8, 684, 3584, 4000) == 0 and R._chan_chunk(8, 684, 1536, 4000) == 64  # work of all against the longest
    assert R._chan_chunk(2, 2586, 3584, 5000) == 128 and R._chan_chunk(6, 576, 1536, 2000) == 64
    assert R._chan_chunk(1, 8192, 3584, 8192) == 256 and R._chan_chunk(1, 4000, 1536, 4000) == 128
