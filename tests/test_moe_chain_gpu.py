"""The experts' grouped GEMM as chains of tiles (csrc/kernels/moe.hip moe_gemm_chain_kernel) against fp64 products per pair:
more tiles than CUs, so that workgroups go on from expert to expert, over experts without rows, with ragged last tiles of
1 to 256 rows and a ragged last column tile, at the fewest K steps (5) and odd counts."""
import pytest
import torch
import torch.nn.functional as F

from githubrepostorag_amd.ops.moe import moe_experts

pytestmark = pytest.mark.gpu
COUNTS = [0, 1300, 0, 0, 1, 700, 255, 256, 257, 1024, 65, 0, 513, 2000, 128, 300]


@pytest.mark.parametrize("unit,W,width", [("glu", 320, 2120), ("relu2", 448, 4104), ("glu", 1024, 1352), ("clamped", 576, 2048)])
def test_chain(dev, unit, W, width):
    g = torch.Generator(device=dev).manual_seed(W)
    E, top = len(COUNTS), 2
    flat = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(COUNTS)])
    flat = torch.cat([flat, torch.full((len(flat) % top,), -1, dtype=torch.int32)])
    ids = flat[torch.randperm(len(flat), generator=torch.Generator().manual_seed(1))].view(-1, top).to(dev)
    T = ids.shape[0]
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    h = r(T, W).bfloat16()
    wgu = (r(E, width if unit == "relu2" else 2 * width, W) * W ** -0.5).bfloat16()
    wd = (r(E, W, width) * width ** -0.5).bfloat16()
    kw = {"glu": {}, "relu2": dict(unit="relu2"), "clamped": dict(limit=1.0, alpha=1.702, shift=1.0)}[unit]
    got = moe_experts(h, ids, wgu, wd, **kw)
    for e in range(E):
        t, k = torch.where(ids == e)
        if not len(t):
            continue
        v = h[t].double() @ wgu[e].double().T
        if unit == "relu2":
            u = v.clamp_min(0) ** 2
        else:
            a, b = v.chunk(2, 1)
            u = F.silu(a) * b if unit == "glu" else a.clamp(max=1) * torch.sigmoid(1.702 * a.clamp(max=1)) * (b.clamp(-1, 1) + 1)
        want = u @ wd[e].double().T
        # the unit's output and the result are rounded to bf16 (2^-9 each), the first averaged over ``width`` terms
        assert (got[t, k].double() - want).norm() / want.norm() < 4e-3, e
        assert (got[t, k].double() - want).abs().max() < 2 ** -7 * want.abs().max(), e
