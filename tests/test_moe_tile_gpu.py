"""The experts' grouped GEMM on 256 x 256 tiles (csrc/kernels/moe.hip moe_gemm_tile_kernel) against a plain fp32 product per
pair: experts of unequal row counts around the tile's quadrants (none, 1, 64, 65, 256, 257 rows), columns past the last whole
tile, pairs that name no expert."""
import pytest
import torch

from githubrepostorag_amd.ops.moe import moe_experts

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 64, 65, 128, 200, 256, 257, 300, 513]


@pytest.mark.parametrize("unit,limit,W,F", [("glu", None, 192, 192), ("glu", 2.0, 320, 448), ("relu2", None, 448, 320),
                                           ("glu", None, 128, 128)])
def test_moe_tile(unit, limit, W, F):
    g = torch.Generator().manual_seed(W + F)
    E, top = len(COUNTS), 2
    flat = torch.cat([torch.full((n,), e) for e, n in enumerate(COUNTS)] + [torch.tensor([-1, E, E + 3, -1])])
    flat = flat[torch.randperm(len(flat), generator=g)]
    T = len(flat) // top
    ids = flat[:T * top].view(T, top).to(torch.int32)
    h = torch.randn(T, W + 8, generator=g).bfloat16()[:, :W]  # rows of a wider matrix
    wgu = (torch.randn(E, F if unit == "relu2" else 2 * F, W, generator=g) * W ** -0.5).bfloat16()
    wd = (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16()
    kw = dict(unit=unit) if unit == "relu2" else dict(limit=limit, alpha=1.3 if limit else 1.0, shift=0.5 if limit else 0.0)
    wide = torch.zeros(T, W + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, :W] = h.cuda()
    got = moe_experts(wide[:, :W], ids.cuda(), wgu.cuda(), wd.cuda(), **kw).float().cpu()
    want = moe_experts(h.contiguous(), ids, wgu, wd, **kw).float()
    ok = (ids >= 0) & (ids < E)
    # both round the unit's output and the result to bf16 (2^-8 apart at most where fp32 sums of another order fall on
    # different sides); the second product averages the first rounding over F terms
    err = (got - want)[ok].abs().max() / want[ok].abs().max()
    assert err < 2 ** -7, err
    assert (got - want)[ok].norm() / want[ok].norm() < 4e-3


@pytest.mark.parametrize("T,W,E,extra,groups,score,dtype", [
    (129, 1536, 16, 1, 4, "softmax", torch.bfloat16), (143, 40, 16, 0, 1, "sigmoid", torch.bfloat16),
    (200, 520, 30, 2, 5, "softmax", torch.float32), (161, 8, 64, 0, 8, "sigmoid", torch.bfloat16),
    (130, 3592, 63, 1, 1, "softmax", torch.float32),
    (128, 2056, 16, 1, 4, "softmax", torch.bfloat16), (1, 8, 3, 0, 1, "sigmoid", torch.bfloat16),
    (64, 2048, 64, 1, 8, "softmax", torch.float32), (65, 6152, 17, 0, 1, "softmax", torch.bfloat16),
    (127, 5128, 200, 1, 8, "sigmoid", torch.float32), (64, 2060, 16, 1, 4, "softmax", torch.bfloat16)])
def test_router(T, W, E, extra, groups, score, dtype):
    """Token counts of steps (matrix cores) and of decode rows (a wave a row) against the plain fp32 router: widths that end
    inside a wave's step, one that is no multiple of 8, rows past a tile or a round of waves."""
    from githubrepostorag_amd.ops.moe import moe_route

    g = torch.Generator().manual_seed(T + W)
    h = torch.randn(T, W, generator=g).to(dtype)
    wr = torch.randn(E + (extra == 1), W, generator=g) * 2 * W ** -0.5
    identity = extra if extra == 2 else 0
    kw = dict(score=score, identity=identity, corr=torch.randn(E, generator=g) * 0.01 if groups == 1 else None)
    top = min(E, 4)
    ids, wts, third = moe_route(h.cuda(), wr.cuda(), E, top, groups, max(1, groups // 2), **{
        k: v.cuda() if torch.is_tensor(v) else v for k, v in kw.items()})
    want_ids, want_wts, want_third = moe_route(h, wr, E, top, groups, max(1, groups // 2), **kw)
    # logits differ by the order of W fp32 terms: sqrt(W) 2^-24 of their size 2, through a softmax of slope <= 1
    tol = 2e-6 + 2 * W ** 0.5 * 2 ** -24
    same = ids.cpu() == want_ids
    assert same.float().mean() > 0.995  # (a tie within the tolerance may fall either way)
    assert ((wts.cpu() - want_wts).abs()[same] < tol).all()
    if third is not None:
        ok = same.all(1)
        assert ((third.cpu() - want_third).abs()[ok] < 4 * tol).all()
