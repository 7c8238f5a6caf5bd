"""The flat scan's tiles and the merge of its lists (csrc/kernels/topk.hip) against the fp32 scores: row counts around a wave's
and a workgroup's tile and more than one tile a wave, query counts around its tiles, list lengths, filters, equal scores."""
import pytest
import torch

from githubrepostorag_amd.ops import topk as T

pytestmark = pytest.mark.gpu


def _data(dev, rows, nq, d, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    # small whole numbers: every score is exact in bf16 products and fp32 sums, and many are equal
    X = torch.randint(-2, 3, (rows, d), generator=g, device=dev).bfloat16()
    Q = torch.randint(-2, 3, (nq, d), generator=g, device=dev).bfloat16()
    return X, Q, torch.randint(0, 3, (rows,), generator=g, device=dev, dtype=torch.int32)


@pytest.mark.parametrize("rows,nq,k,d", [
    (1, 1, 1, 32), (15, 16, 10, 96), (129, 17, 16, 768), (130, 3, 17, 64), (2049, 33, 32, 384), (40000, 5, 5, 224), (70001, 65, 10, 32),
    (70001, 20, 30, 160), (300000, 1, 32, 32), (600000, 70, 7, 64)])
@pytest.mark.parametrize("filt", [0, 1, 2])
def test_flat_scan(dev, rows, nq, k, d, filt):
    X, Q, col = _data(dev, rows, nq, d, rows + nq)
    alive = torch.ones(rows, dtype=torch.bool, device=dev)
    preds = bitmap = None
    if filt:
        preds = [T.Predicate(col, 1)]
        alive = col == 1
    if filt == 2:  # two columns and an allow-bitmap
        preds.append(T.Predicate(col * 3 + 4, 4, T.OP_BITAND))
        keep = torch.rand(rows, device=dev) < 0.5
        pad = torch.zeros(-rows % 32, dtype=torch.bool, device=dev)
        bits = torch.cat([keep, pad]).view(-1, 32).long() << torch.arange(32, device=dev)
        bitmap = bits.sum(1).to(torch.int64).bitwise_and(0xFFFFFFFF).to(torch.uint32).view(torch.int32)
        alive = alive & keep & (((col * 3 + 4) & 4) != 0)
    s, ids = T.score_topk(X, Q, k, preds=preds, bitmap=bitmap)
    full = (Q.float() @ X.float().T).masked_fill(~alive, float("-inf"))
    want = torch.cat([full, full.new_full((nq, max(0, k - rows)), float("-inf"))], 1).topk(k, 1).values
    assert torch.equal(s, want)  # (exact sums)
    there = ids >= 0
    assert torch.equal(there, want > float("-inf"))
    assert torch.equal(full.gather(1, ids.clamp_min(0))[there], s[there])
    for row in ids.tolist():
        row = [i for i in row if i >= 0]
        assert len(set(row)) == len(row)


@pytest.mark.parametrize("n,k", [(1, 4), (2, 32), (17, 17), (18, 17), (32, 32), (33, 32), (255, 10), (257, 1), (1024, 32), (1000, 17)])
def test_merge_orders_ties_by_list(dev, n, k):
    """Lists of equal and of missing values: the best k by value, then list, then place."""
    g = torch.Generator(device=dev).manual_seed(n + k)
    nq, G = 3, 16
    ps = torch.randint(0, 4, (n * G, k), generator=g, device=dev).float().sort(1, descending=True).values
    ps[torch.rand(n * G, device=dev, generator=g) < 0.3] = float("-inf")
    pi = torch.arange(n * G * k, device=dev).view(-1, k)
    out_s, out_i = torch.empty(nq, k, device=dev), torch.empty(nq, k, dtype=torch.long, device=dev)
    T.call("grag_topk_lists_merge", T.ptr(ps), T.ptr(pi), n, G, nq, k, T.ptr(out_s), T.ptr(out_i))
    for q in range(nq):
        v, i = ps[q::G].reshape(-1).cpu(), pi[q::G].reshape(-1).cpu()
        order = sorted(range(len(v)), key=lambda e: (-v[e].item(), e))[:k]
        order += [None] * (k - len(order))
        assert out_s[q].tolist() == [float("-inf") if e is None else v[e].item() for e in order]
        assert out_i[q].tolist() == [-1 if e is None or v[e] == float("-inf") else i[e].item() for e in order]
