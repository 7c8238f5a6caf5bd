"""Decode sink attention on the matrix cores (csrc/kernels/sink_decode.hip) against the plain fp32 attention: lengths around
tiles, blocks and the 1024 keys of a table window, key splits and none, every option it takes."""
import pytest
import torch

from githubrepostorag_amd.ops.attention import AttnMetadata, sink_attention, sink_attention_ref

pytestmark = pytest.mark.gpu
dev = "cuda"
LENS = [1, 15, 16, 17, 31, 32, 33, 64, 65, 257, 1024, 1025, 2111]


def step(lens, H, G, D, nsplit, split_len, seed=0, BS=16):
    g = torch.Generator(device=dev).manual_seed(seed + D + H)
    n = len(lens)
    nb = sum(-(-x // BS) for x in lens)
    order = torch.randperm(nb, generator=torch.Generator().manual_seed(seed)) + 1
    bt, a = torch.full((n, -(-max(lens) // BS) + 1), nb + 7, dtype=torch.int32), 0  # entries past a sequence name no block
    for i, x in enumerate(lens):
        k = -(-x // BS)
        bt[i, :k] = order[a:a + k]
        a += k
    kc, vc = (torch.randn(nb + 1, G, BS, D, generator=g, device=dev).bfloat16() for _ in range(2))
    for i, x in enumerate(lens):  # slots past a sequence's end hold no numbers
        if x % BS:
            kc[bt[i, x // BS], :, x % BS:] = float("nan")
            vc[bt[i, x // BS], :, x % BS:] = float("inf")
    i32 = dict(dtype=torch.int32, device=dev)
    m = AttnMetadata(q_start=torch.arange(n + 1, **i32), ctx_len=torch.tensor(lens, **i32), block_tables=bt.to(dev), slot_mapping=None,
                     max_q_len=1, num_seqs=n, num_tokens=n, is_decode=True, num_splits=nsplit, split_len=split_len,
                     part_o=torch.full((nsplit * n * H * D,), float("nan"), device=dev),
                     part_ml=torch.full((nsplit * n * H * 2,), float("nan"), device=dev))
    q = torch.randn(n, H, D, generator=g, device=dev).bfloat16() * 2
    return q, kc, vc, m, g


@pytest.mark.parametrize("H,G,D", [(14, 2, 128), (16, 1, 64), (20, 1, 128), (3, 3, 64)])
@pytest.mark.parametrize("splits", [(1, 0), (5, 448), (34, 64)])
@pytest.mark.parametrize("opts", [{}, dict(window=100), dict(window=1500), dict(chunk=1100), dict(softcap=5.0),
                                  dict(window=40, softcap=3.0, scales=True), dict(scales=True, gate=True), dict(sinks=False)])
def test_sink_decode(H, G, D, splits, opts):
    check(LENS, H, G, D, splits, opts)


@pytest.mark.parametrize("H,G,D", [(28, 4, 128), (12, 4, 64)])
@pytest.mark.parametrize("n,splits", [(64, (4, 512)), (129, (1, 0)), (129, (3, 704))])  # one and two waves, also of eight and more tiles
@pytest.mark.parametrize("opts", [{}, dict(window=700), dict(chunk=1100, softcap=5.0), dict(scales=True, gate=True)])
def test_many_parts(H, G, D, n, splits, opts):
    check([(i * 397 + 61) % 2048 + 1 for i in range(n)], H, G, D, splits, opts)


def check(lens, H, G, D, splits, opts):
    q, kc, vc, m, g = step(lens, H, G, D, *splits)
    opts = dict(opts)
    sinks = torch.randn(H, generator=g, device=dev) * 2 if opts.pop("sinks", True) else None
    if opts.pop("scales", False):
        opts["head_scale"] = torch.randn(H, generator=g, device=dev)
    gate = torch.randn(len(lens), H, generator=g, device=dev).bfloat16() if opts.pop("gate", False) else None
    y = sink_attention(q, kc, vc, m, D ** -0.5, sinks, out_scale=1.5, head_gate=gate, **opts).float().view(len(lens), H, D)
    kf, vf = kc.float().nan_to_num(0, 0, 0), vc.float().nan_to_num(0, 0, 0)
    s = sinks if sinks is not None else torch.full((H,), float("-inf"), device=dev)
    r = sink_attention_ref(q.float(), kf, vf, m, D ** -0.5, s, **opts).float().view(len(lens), H, D) * 1.5
    if gate is not None:
        r = r * torch.sigmoid(gate.float())[:, :, None]
    # bf16 rounding of the result (2^-8 of it), and 16-bit weights of a sum that is at most the largest value
    assert ((y - r).abs() <= r.abs() * 2 ** -8 + 1.5 * 5 * 2 ** -15).all()
