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


@pytest.mark.parametrize("H,G", [(4, 2), (8, 8)])  # row tiles dealt one by one, and by sequence
def test_paged_prefill_of_uneven_sequences(H, G):
    from githubrepostorag_amd.ops.attention import AttnMetadata, paged_attention, paged_attention_ref

    g = torch.Generator(device="cuda").manual_seed(G)
    D, BS, lens = 32, 16, [700, 3, 64, 65, 1, 130, 17, 5, 300, 40, 9]
    q0 = [0]
    for n in lens:
        q0.append(q0[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    nb = [-(-n // BS) for n in lens]
    bt = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    for i, n in enumerate(nb):
        bt[i, :n] = torch.arange(n) + sum(nb[:i])
    q = torch.randn(q0[-1], H, D, generator=g, device="cuda").bfloat16()
    kc, vc = (torch.randn(sum(nb), G, BS, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    m = AttnMetadata(q_start=i32(q0), ctx_len=i32(lens), block_tables=bt.cuda(), slot_mapping=None, max_q_len=max(lens),
                     num_seqs=len(lens), num_tokens=q0[-1])
    got = paged_attention(q, kc, vc, m, D ** -0.5).float()
    want = paged_attention_ref(q.float(), kc.float(), vc.float(), m, D ** -0.5).reshape(q0[-1], -1).float()
    # the weights and the result are rounded to bf16: 2^-8 of the result and of the values that the weights sum
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 4 * 2 ** -8).all()
    assert (got - want).norm() / want.norm() < 5e-3
