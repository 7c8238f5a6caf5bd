"""Row passes of the hybrid layers in wide accesses (dynamic-tanh residual, gated RMSNorm of wide groups, rotary + K/V store
with value norms) at the edges of their forms, against the fp32 CPU paths of the same operations."""
import pytest
import torch

pytestmark = pytest.mark.gpu
dev = "cuda"
bf = torch.bfloat16


def rnd(g, *s):
    return torch.randn(*s, generator=g)


@pytest.mark.parametrize("T,H", [(1, 4), (1023, 36), (8192, 36), (4098, 1028), (3, 3584), (5, 6)])
@pytest.mark.parametrize("post,rows,vec,pre", [(1, 1, 1, 1), (1, 0, 0, 1), (0, 0, 1, 0), (0, 1, 0, 1), (1, 0, 1, 0), (0, 0, 0, 1)])
def test_dyt_residual(T, H, post, rows, vec, pre):
    from githubrepostorag_amd.ops.norm import dyt_residual

    g = torch.Generator().manual_seed(T + H)
    r, y = rnd(g, T, H), rnd(g, T, H).to(bf) * 3
    tri = lambda a: (a, rnd(g, H), rnd(g, H))
    po, pr = tri(0.7), tri(-1.3)
    ar, av = rnd(g, T, H), rnd(g, H)
    on = lambda t: t if t is None else (t[0], t[1].to(dev), t[2].to(dev))
    r1 = r.clone().to(dev)
    h = dyt_residual(r1, y.to(dev) if post else None, on(po if post else None), ar.to(dev) if rows else None,
                     av.to(dev) if vec else None, on(pr if pre else None))
    x = r.double()
    if post:
        x = x + torch.tanh(po[0] * y.double()) * po[1].double() + po[2].double()
    x = x + (ar.double() if rows else 0) + (av.double() if vec else 0)
    # a handful of fp32 roundings of terms of a few units
    assert (r1.cpu().double() - x).abs().max() <= 4e-6
    if pre:
        o = torch.tanh(pr[0] * x) * pr[1].double() + pr[2].double()
        assert ((h.cpu().double() - o).abs() <= o.abs() * 2 ** -8 + 4e-5).all()  # bf16 rounding of the result
    else:
        assert h is None


def test_dyt_residual_special():
    from githubrepostorag_amd.ops.norm import dyt_residual

    inf, nan = float("inf"), float("nan")
    y = torch.tensor([[inf, -inf, nan, 0.0, 1e-30, -1e30, 1e30, 0.02]], device=dev)
    r = torch.zeros_like(y)
    one, zero = torch.ones(8, device=dev), torch.zeros(8, device=dev)
    dyt_residual(r, y, (1.0, one, zero), out_dtype=torch.float32)
    v = r.cpu()[0]
    assert v[2].isnan() and v[[0, 1, 3, 5, 6]].tolist() == [1.0, -1.0, 0.0, -1.0, 1.0]
    assert abs(v[4].item() - 1e-30) < 1e-36 and abs(v[7].item() - 0.0199973340) < 1e-8


@pytest.mark.parametrize("N,groups", [(260, 1), (512, 1), (516, 1), (1032, 2), (3584, 1), (4100, 1), (8192, 1), (8196, 1), (7168, 8)])
@pytest.mark.parametrize("gate,first", [("silu", False), ("sigmoid", False), ("silu", True)])
@pytest.mark.parametrize("dtype", [bf, torch.float32])
def test_gated_rmsnorm_wide(N, groups, gate, first, dtype):
    from githubrepostorag_amd.ops.recurrent import gated_rmsnorm

    g = torch.Generator().manual_seed(N)
    T = 3
    x, w, p = rnd(g, T, N), rnd(g, N), rnd(g, T, N + 8).to(dtype)
    for goff, weight in ((4, w), (3, None)):  # aligned columns, and not
        o, ref = torch.empty(T, N + 4, dtype=dtype, device=dev), torch.empty(T, N)
        gated_rmsnorm(x.to(dev), None if weight is None else w.to(dev), p.to(dev), goff, 1e-5, o[:, 4:], 1.7, groups, gate, first)
        gated_rmsnorm(x, weight, p.float(), goff, 1e-5, ref, 1.7, groups, gate, first)
        # bf16 rounding of the result; fp32: the sums' and the exponential's roundings
        tol = (2 ** -8 if dtype == bf else 4e-6) * ref.abs() + 1e-6
        assert ((o[:, 4:].float().cpu() - ref).abs() <= tol).all()


@pytest.mark.parametrize("d,vd,rd,H,G", [(16, 32, 16, 3, 1), (128, 128, 128, 4, 2), (64, 128, 32, 2, 1), (128, 64, 0, 2, 2), (256, 256, 64, 1, 1)])
@pytest.mark.parametrize("T", [1, 37])
def test_rope_store_value_norm(d, vd, rd, H, G, T):
    from githubrepostorag_amd.ops.elementwise import rope_table, rope_vnorm_store

    g = torch.Generator().manual_seed(d + vd + T)
    ld = (H + G) * d + G * vd + 8
    p, pos = rnd(g, T, ld).to(bf), torch.randint(0, 90, (T,), generator=g).int()
    p[0, (H + G) * d:] = 0  # a value of zero: eps alone under the root
    tab = rope_table(90, rd, 1e4) if rd else None
    slots = torch.randperm(T + 16, generator=g)[:T].int()
    slots[T // 2] = -1
    outs = []
    for dv in ("cpu", dev):
        kc, vc = torch.zeros(4, G, 16, d, dtype=bf, device=dv), torch.zeros(4, G, 16, vd, dtype=bf, device=dv)
        q = rope_vnorm_store(p.to(dv), 0, H * d, (H + G) * d, pos.to(dv), None if tab is None else tab.to(dv), slots.to(dv), kc, vc,
                             H, G, d, vd, rd, 1e-6)
        outs.append([t.float().cpu() for t in (q, kc, vc)])
    for a, b in zip(*outs):
        # both round once from fp32: half a unit each way, plus a rotation's cancellation in fp32
        assert ((a - b).abs() <= a.abs() * 2 ** -7 + 1e-5).all()


@pytest.mark.parametrize("T,H,S", [(1, 8, 1), (3, 1032, 7), (300, 64, 9), (2, 3584, 17)])
def test_dyt_residual_splitk(T, H, S):
    """The planes of a deferred split-K product in place of its sum."""
    from githubrepostorag_amd.ops.gemm import SplitKPartial
    from githubrepostorag_amd.ops.norm import dyt_residual

    g = torch.Generator().manual_seed(T + H)
    planes, r = rnd(g, S, T, H).to(dev), rnd(g, T, H)
    po, pr, av = (0.7, rnd(g, H), rnd(g, H)), (0.9, rnd(g, H), rnd(g, H)), rnd(g, H)
    on = lambda t: (t[0], t[1].to(dev), t[2].to(dev))
    r1 = r.clone().to(dev)
    h = dyt_residual(r1, SplitKPartial(planes, S, T, H, bf), on(po), None, av.to(dev), on(pr))
    x = r.double() + torch.tanh(po[0] * planes.double().sum(0).cpu()) * po[1].double() + po[2].double() + av.double()
    # a handful of fp32 roundings of terms of a few units, S of them in the sum
    assert (r1.cpu().double() - x).abs().max() <= 4e-6 + S * 1e-6
    o = torch.tanh(pr[0] * x) * pr[1].double() + pr[2].double()
    assert ((h.cpu().double() - o).abs() <= o.abs() * 2 ** -8 + 4e-5 + S * 4e-6).all()


def test_dyt_residual_splitk_unaligned():
    """Norm vectors that lie at no multiple of 16 bytes (views of one buffer), as with a product that was summed before."""
    from githubrepostorag_amd.ops.gemm import SplitKPartial
    from githubrepostorag_amd.ops.norm import dyt_residual

    T, H, S = 5, 128, 3
    g = torch.Generator(device="cuda").manual_seed(3)
    planes = torch.randn(S * T * H, generator=g, device="cuda")
    flat = torch.randn(4 * H + 1, generator=g, device="cuda")
    w1, b1, w2, b2 = flat[1:].view(4, H)
    x = torch.randn(T, H, generator=g, device="cuda")
    r1, r2 = x.clone(), x.clone()
    h1 = dyt_residual(r1, SplitKPartial(planes, S, T, H, torch.bfloat16), (0.7, w1, b1), pre=(0.9, w2, b2))
    h2 = dyt_residual(r2, planes.view(S, T, H).sum(0).bfloat16(), (0.7, w1, b1), pre=(0.9, w2, b2))
    assert torch.equal(r1, r2) and torch.equal(h1, h2)
