"""Sums over more than 16 split-K planes (csrc/kernels/common.h plane_acc4: passes of 16, then the rest) in plane order, bit for bit:
the boundary norm's residual stream at the last plane of a pass and one past it, in both of its kernels."""
import pytest
import torch

from githubrepostorag_amd.ops._lib import call, ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [16, 17, 18, 32, 33, 41])
@pytest.mark.parametrize("T,H", [(1, 1536), (16, 1536), (17, 2304)])
def test_plane_order(dev, S, T, H):
    g = torch.Generator(device=dev).manual_seed(S)
    planes = torch.randn(S, T, H, generator=g, device=dev)
    res = torch.randn(T, H, generator=g, device=dev).bfloat16()
    w = torch.randn(H, generator=g, device=dev).bfloat16()
    want = res.float()
    for p in planes:
        want = want + p
    want = want.bfloat16()
    out = torch.empty_like(res)
    call("grag_splitk_add_rmsnorm", ptr(planes), S, ptr(res), ptr(w), ptr(out), T, H, 1e-6)
    assert torch.equal(res, want)
    h = want.double()
    y = h * torch.rsqrt(h.pow(2).mean(1, keepdim=True) + 1e-6) * w.double()
    assert ((out.double() - y).abs() <= 2 ** -8 * 1.01 * y.abs()).all()  # the result's rounding to bf16, and fp32's
