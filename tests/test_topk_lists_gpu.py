"""The flat scan's lists (csrc/kernels/topk.hip): merged over waves, workgroups and lanes, against the plain fp32 scan, at row
counts around a workgroup's share, both list lengths, every query tiling, and filters that leave fewer rows than asked for."""
import pytest
import torch

from githubrepostorag_amd.ops import topk
from githubrepostorag_amd.ops.topk import Predicate, score_topk, score_topk_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq", [1, 17, 65])
@pytest.mark.parametrize("k", [1, 16, 17, 32])
@pytest.mark.parametrize("N,d", [(1, 32), (128, 96), (129, 384), (4001, 768), (40000, 64)])
def test_flat_lists(N, d, k, nq, monkeypatch):
    monkeypatch.setattr(topk, "NQT4_MIN_ROWS", 4000)  # (the widest tiling at a testable size)
    g = torch.Generator().manual_seed(N + k + nq)
    X = torch.nn.functional.normalize(torch.randn(N, d, generator=g), dim=1).bfloat16().cuda()
    Q = torch.nn.functional.normalize(torch.randn(nq, d, generator=g), dim=1).bfloat16().cuda()
    col = torch.randint(0, max(2, N // 20), (N,), generator=g, dtype=torch.int32).cuda()
    for preds, begin in ((None, 0), ([Predicate(col, 1)], 0), (None, N // 3)):
        s, i = score_topk(X, Q, k, preds=preds, row_begin=begin)
        part = [Predicate(p.column[begin:], p.value) for p in preds] if preds else None
        ws, wi = score_topk_ref(X[begin:], Q, k, preds=part)
        wi = torch.where(wi >= 0, wi + begin, wi)
        assert s.shape == ws.shape and torch.equal(torch.isinf(s), torch.isinf(ws)) and torch.equal(i < 0, wi < 0)
        ok = wi >= 0
        # d exact products, summed in fp32 in another order: d / 2 ulp of scores below 1
        assert not ok.any() or (s - ws)[ok].abs().max() < d * 2 ** -24
        own = (X[i.clamp_min(0)].float() * Q[:, None].float()).sum(-1)  # the ids are rows of those scores
        assert not ok.any() or (own - s)[ok].abs().max() < 2 * d * 2 ** -24
        assert all(len(set(r[r >= 0].tolist())) == int((r >= 0).sum()) for r in i.cpu())
