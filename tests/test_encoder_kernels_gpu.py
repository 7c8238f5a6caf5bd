"""Encoder kernels at the edges of their tiles: LayerNorm with a wave a row, attention over packed ragged rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
dev = "cuda"
bf = torch.bfloat16


@pytest.mark.parametrize("H", [8, 504, 512, 520, 768, 1024, 1032])
@pytest.mark.parametrize("T", [1, 4, 7])
@pytest.mark.parametrize("bias,res", [(True, True), (False, True), (True, False), (False, False)])
def test_layernorm_rows(H, T, bias, res):
    from githubrepostorag_amd.ops import norm as N

    g = torch.Generator(device=dev).manual_seed(H * 10 + T)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(bf)
    x, ga, be = rnd(T, H), rnd(H), rnd(H)
    b, r = rnd(H) if bias else None, rnd(T, H) if res else None
    v = x.double() + (b.double() if bias else 0) + (r.double() if res else 0)
    ref = torch.nn.functional.layer_norm(v, (H,), ga.double(), be.double(), 1e-12)
    y = N.layernorm(x, ga, be, 1e-12, bias=b, residual=r).double()
    # bf16 rounding of the result, and fp32 sums of H terms of at most a few units
    assert ((y - ref).abs() <= ref.abs() * 2 ** -8 + 2e-5).all()
    if res:
        r1 = r.clone()
        y = N.add_layernorm(x, ga, be, 1e-12, r1, bias=b).double()
        s = ((x.float() + (b.float() if bias else 0)) + r.float()).to(bf)
        assert torch.equal(r1, s)
        ref = torch.nn.functional.layer_norm(s.double(), (H,), ga.double(), be.double(), 1e-12)
        assert ((y - ref).abs() <= ref.abs() * 2 ** -8 + 2e-5).all()


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lens", [[1, 63, 64, 65], [17, 128, 129, 2, 200], [15, 16, 3], [5, 70, 64, 1, 130, 20, 3, 65, 33] * 2])
def test_varlen_attention_edges(D, causal, lens):
    from githubrepostorag_amd.ops.attention import varlen_attention, varlen_attention_ref

    H = 3
    st = torch.tensor([0] + lens).cumsum(0).int().to(dev)
    sl = torch.tensor(lens).int().to(dev)
    q = torch.randn(int(st[-1]), 3 * H * D, generator=torch.Generator(device=dev).manual_seed(D), device=dev).to(bf)
    q[:, : H * D] *= 3  # some rows' softmax close to one key
    y = varlen_attention(q, st, sl, max(lens), H, D, D ** -0.5, causal).float().cpu()
    r = varlen_attention_ref(q.float().cpu(), st.cpu(), H, D, D ** -0.5, causal)
    # weights and result rounded to bf16 of 8 bits (2^-8 of a value at most, each, relative to the largest value a row can hold)
    assert (y - r).abs().max() <= 2 * 2 ** -8 * q[:, 2 * H * D:].float().abs().max().item() + 1e-5
