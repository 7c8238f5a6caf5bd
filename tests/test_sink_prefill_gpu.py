"""The row-packed prefill attention (csrc/kernels/sink_prefill.hip) against the plain fp32 attention: row counts around its
128-row workgroups and 16-row groups, cached tokens before the portion, and every visibility form and score option."""
import pytest
import torch

from githubrepostorag_amd.ops.attention import AttnMetadata, sink_attention

pytestmark = pytest.mark.gpu

FORMS = {
    "causal": {}, "window": dict(window=70), "narrow": dict(window=3), "kept": dict(window=65, keep=20),
    "kept_far": dict(window=40, keep=130), "block": dict(chunk=100), "block_kept": dict(chunk=64, keep=5),
    "capped": dict(window=128, softcap=2.0),
}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("D,H,G,lens,past", [
    (128, 28, 4, [37, 16, 300], [0, 61, 0]), (128, 4, 4, [257], [5]), (64, 12, 2, [129, 1, 64], [200, 0, 63]),
    (64, 6, 1, [43], [400]), (128, 14, 2, [1], [0]), (64, 16, 8, [130] * 19 + [3], [0, 70] * 10),
    (128, 12, 4, [140] * 29 + [17], [0, 75, 3] * 10)])  # the last two: 128-row workgroups
def test_sink_prefill(D, H, G, lens, past, form):
    g = torch.Generator().manual_seed(D + sum(lens) + len(form))
    BS = 16
    lens, past = (lens, past) if max(lens) >= 16 else (lens + [16], past + [9])  # (the kernel's least)
    ctx = [n + p for n, p in zip(lens, past)]
    q0 = [0]
    for n in lens:
        q0.append(q0[-1] + n)
    width = -(-max(ctx) // BS)
    nb = 1 + sum(-(-c // BS) for c in ctx)
    order = (torch.randperm(nb - 1, generator=g) + 1).tolist()
    bt = torch.zeros(len(ctx), width, dtype=torch.int32)
    for i, c in enumerate(ctx):
        for j in range(-(-c // BS)):
            bt[i, j] = order.pop()
    T = q0[-1]
    q = torch.randn(T, H, D, generator=g).bfloat16()
    kc, vc = (torch.randn(nb, G, BS, D, generator=g).bfloat16() for _ in range(2))
    for i, c in enumerate(ctx):  # what lies behind a sequence's end must not matter
        if c % BS:
            kc[bt[i, c // BS], :, c % BS:] = float("nan")
            vc[bt[i, c // BS], :, c % BS:] = float("nan")
    kw = dict(FORMS[form])
    sinks = None if form in ("narrow", "block") else torch.randn(H, generator=g)
    if form in ("block", "kept"):
        kw.update(head_scale=torch.linspace(-1.5, 1.5, H), head_gate=torch.randn(T, H + 3, generator=g).bfloat16()[:, 1:H + 1])
    i32 = lambda v, dev: torch.tensor(v, dtype=torch.int32, device=dev)

    def run(dev):
        m = AttnMetadata(q_start=i32(q0, dev), ctx_len=i32(ctx, dev), block_tables=bt.to(dev), slot_mapping=None,
                         max_q_len=max(lens), num_seqs=len(ctx), num_tokens=T)
        out = torch.zeros(T, H * D + 8, dtype=torch.bfloat16 if dev == "cuda" else torch.float32, device=dev)
        k = {a: b.to(dev) if torch.is_tensor(b) else b for a, b in kw.items()}
        sink_attention(q.to(dev), kc.to(dev), vc.to(dev), m, D ** -0.5, None if sinks is None else sinks.to(dev),
                       out[:, :H * D], 0.7, **k)
        return out.float().cpu()

    got, want = run("cuda"), run("cpu")
    assert not want.isnan().any()
    assert torch.equal(got[:, H * D:], torch.zeros(T, 8))
    # the result's own rounding to bf16 is 2^-9; the weights reach the sums with 16 bits
    err = (got - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 2e-4).all(), err.max()


@pytest.mark.parametrize("scale", [-0.11, 0.0])
@pytest.mark.parametrize("form", ["causal", "window", "block_kept", "capped"])
def test_scale_of_any_sign(form, scale):
    """The scale is the caller's number: a negative one turns the order of the scores, with 0 every key weighs the same."""
    g = torch.Generator().manual_seed(len(form))
    D, H, G, n, past, BS = 64, 6, 2, 130, 70, 16
    nb = -(-(n + past) // BS)
    q = torch.randn(n, H, D, generator=g).bfloat16()
    kc, vc = (torch.randn(nb, G, BS, D, generator=g).bfloat16() for _ in range(2))
    sinks = torch.randn(H, generator=g)

    def run(dev):
        i32 = dict(dtype=torch.int32, device=dev)
        m = AttnMetadata(q_start=torch.tensor([0, n], **i32), ctx_len=torch.tensor([n + past], **i32),
                         block_tables=torch.arange(nb, **i32).view(1, nb), slot_mapping=None, max_q_len=n, num_seqs=1, num_tokens=n)
        out = torch.empty(n, H * D, dtype=torch.bfloat16 if dev == "cuda" else torch.float32, device=dev)
        return sink_attention(q.to(dev), kc.to(dev), vc.to(dev), m, scale, sinks.to(dev), out, **FORMS[form]).float().cpu()

    got, want = run("cuda"), run("cpu")
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-4).all()  # (as above)
