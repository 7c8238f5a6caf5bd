"""The prefill attention's workgroups (csrc/kernels/sink_prefill.hip: 128 rows, or 64 by one or two teams of waves) against the
plain fp32 attention: portions that end at and beside their edges and those of the waves, cached tokens before some, walks whose
last tile is one key, and caps met by the power series and by tanhf."""
import pytest
import torch

from githubrepostorag_amd.ops._lib import lib
from githubrepostorag_amd.ops.attention import AttnMetadata, sink_attention, sink_attention_ref

pytestmark = pytest.mark.gpu

FORMS = {"causal": {}, "window": dict(window=150), "kept": dict(window=90, keep=70), "block": dict(chunk=200),
         "cap_low": dict(softcap=3.0), "cap_high": dict(window=300, softcap=60.0)}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("D,H,G,lens,past", [
    (64, 24, 8, [640, 33, 1, 705, 128, 321], [0, 31, 64, 0, 1, 0]), (128, 28, 4, [1100, 16, 577, 64], [5, 0, 0, 63])])
def test_rows(dev, D, H, G, lens, past, form):
    assert shape(D, H, G, lens, past, form) == (1 if D == 64 else 2)  # one team of 64 rows, 128 rows
    check(dev, D, H, G, lens, past, form)


def shape(D, H, G, lens, past, form):
    kw, width = FORMS[form], -(-max(n + p for n, p in zip(lens, past)) // 16)
    return lib().grag_sink_prefill_shape(D, len(lens), sum(lens), max(lens), H // G, G, kw.get("chunk", 0), kw.get("window", 0), width)


def check(dev, D, H, G, lens, past, form):
    g = torch.Generator(device=dev).manual_seed(D + len(form))
    BS, ctx, T = 16, [n + p for n, p in zip(lens, past)], sum(lens)
    q0 = torch.tensor([0] + lens).cumsum(0)
    width, nb = -(-max(ctx) // BS), sum(-(-c // BS) for c in ctx)
    perm, bt, at = torch.randperm(nb, generator=torch.Generator().manual_seed(1)), torch.zeros(len(ctx), width, dtype=torch.int32), 0
    for i, c in enumerate(ctx):
        n = -(-c // BS)
        bt[i, :n], at = perm[at:at + n].int(), at + n
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    q, kc, vc, sinks = r(T, H, D).bfloat16(), r(nb, G, BS, D).bfloat16(), r(nb, G, BS, D).bfloat16(), r(H)
    for i, c in enumerate(ctx):  # what lies behind a sequence's end must not matter
        if c % BS:
            kc[bt[i, c // BS], :, c % BS:] = float("nan")
            vc[bt[i, c // BS], :, c % BS:] = float("nan")
    i32 = lambda v: torch.as_tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    m = AttnMetadata(q_start=i32(q0), ctx_len=i32(ctx), block_tables=bt.to(dev), slot_mapping=None, max_q_len=max(lens),
                     num_seqs=len(ctx), num_tokens=T)
    kw = dict(FORMS[form])
    if form == "block":
        kw["head_scale"] = torch.linspace(-1.2, 1.4, H, device=dev)
    got = sink_attention(q, kc, vc, m, D ** -0.5, sinks, **kw).view(T, H, D).float()
    want = sink_attention_ref(q, kc, vc, m, D ** -0.5, sinks, kw.get("head_scale"), kw.get("chunk", 0), kw.get("window", 0),
                              kw.get("softcap", 0.0), kw.get("keep", 0)).float()
    assert not want.isnan().any()
    # the result's own rounding to bf16 is 2^-9; the weights reach the sums with 16 bits
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-4).all(), (got - want).abs().max()


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("D,H,G,lens,past,teams", [
    (128, 12, 2, [300, 1, 65, 16], [0, 63, 1500, 700], 2), (64, 6, 1, [64, 1, 65], [900, 0, 0], 2), (64, 14, 2, [16], [0], 1),
    (64, 6, 1, [64, 65], [64, 0], 1)])
def test_two_teams(dev, D, H, G, lens, past, teams, form):
    """Few rows: two teams of waves on a walk's tiles, of which one may have none, or none that a row sees; one team for the
    shortest walks."""
    assert shape(D, H, G, lens, past, form) == 2 - teams
    check(dev, D, H, G, lens, past, form)
