"""The decode waves' walk over the cache's tiles (csrc/kernels/attention.hip DecodeWalk) against fp32 attention: contexts that end
beside a tile, a block and a window of 64 blocks, blocks of a size that is no power of two, one key, every ring, and walks that
start behind a shared prefix of an odd number of blocks, whose tiles lie across the windows."""
import numpy as np
import pytest
import torch

from githubrepostorag_amd.ops import attention as A

pytestmark = pytest.mark.gpu


def batch(dev, rows, nb, H, G, D, BS, seed):
    """rows: (block ids, keys).  What lies behind a row's end is not a number."""
    g = torch.Generator(device=dev).manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    q, kc, vc = r(len(rows), H, D), r(nb, G, BS, D), r(nb, G, BS, D)
    bt = torch.zeros(len(rows), max(len(ids) for ids, _ in rows), dtype=torch.int32)
    for i, (ids, n) in enumerate(rows):
        bt[i, :len(ids)] = torch.tensor(ids)
        if n % BS:
            kc[ids[-1], :, n % BS:] = float("nan")
            vc[ids[-1], :, n % BS:] = float("nan")
    m = A.AttnMetadata(q_start=torch.arange(len(rows) + 1, dtype=torch.int32, device=dev), block_tables=bt.to(dev),
                       ctx_len=torch.tensor([n for _, n in rows], dtype=torch.int32, device=dev), slot_mapping=None, max_q_len=1,
                       num_seqs=len(rows), num_tokens=len(rows), is_decode=True)
    return q, kc, vc, m


def check(q, kc, vc, m, got):
    want = A.paged_attention_ref(q.float(), kc, vc, m, q.shape[2] ** -0.5)
    size = A.paged_attention_ref(q.float(), kc, vc.abs(), m, q.shape[2] ** -0.5)
    # the weights and the result are rounded to bf16's 8 bits: at most 2^-8 of each; 1.05 for fp32's sums and exponents
    assert ((got.reshape(want.shape).float() - want).abs() <= 1.05 * 2 ** -8 * (want.abs() + size)).all()


def split(m, H, D, dev, n, most):
    if n:
        m.num_splits, m.split_len = -(-most // n), n
        m.part_o = torch.empty(m.num_splits * m.num_seqs * H * D, device=dev)
        m.part_ml = torch.empty(m.num_splits * m.num_seqs * H * 2, device=dev)


@pytest.mark.parametrize("D,H,G", [(128, 28, 4), (64, 6, 1), (32, 8, 2)])
@pytest.mark.parametrize("BS", [16, 48])
@pytest.mark.parametrize("n", [0, 256])
def test_walk(dev, D, H, G, BS, n):
    lens = [1, 15, 16, 33, 64 * BS - 1, 64 * BS, 64 * BS + 1, 64 * BS + 17, 100 * BS + 5]
    perm = torch.randperm(sum(-(-c // BS) for c in lens), generator=torch.Generator().manual_seed(D)).tolist()
    nb, rows = len(perm), []
    for c in lens:
        rows.append((perm[:-(-c // BS)], c))
        perm = perm[-(-c // BS):]
    q, kc, vc, m = batch(dev, rows, nb, H, G, D, BS, D + BS)
    split(m, H, D, dev, n, max(lens))
    A.decode_counters(dev)
    got = {}
    for code in (1, 3, 7, 8, 11, 12) + ((22, 24) if D > 32 else ()):
        m.extra = {"decode_nw": code}
        got[code] = A.paged_attention(q, kc, vc, m, D ** -0.5)
        check(q, kc, vc, m, got[code])
    # the rings of 32-key tiles differ in their loads alone: another kernel would sum in another order
    assert all(torch.equal(got[3], got[c]) for c in (7, 8, 11, 12))


@pytest.mark.parametrize("n", [0, 4096])
def test_wide_table(dev, n):
    """A table of more than 2048 blocks, which the 8-wave prefill kernel does not take: the decode kernel all the same."""
    D, H, G, BS = 64, 6, 2, 16
    lens, nb, rows = [2049 * BS, 2050 * BS - 3, 300], 0, []
    for c in lens:
        rows.append((list(range(nb, nb + -(-c // BS))), c))
        nb += -(-c // BS)
    q, kc, vc, m = batch(dev, rows, nb, H, G, D, BS, 5)
    split(m, H, D, dev, n, max(lens))
    got = {}
    for code in (3, 11, 12):
        m.extra = {"decode_nw": code}
        got[code] = A.paged_attention(q, kc, vc, m, D ** -0.5)
        check(q, kc, vc, m, got[code])
    assert torch.equal(got[3], got[11]) and torch.equal(got[3], got[12])


@pytest.mark.parametrize("D,H", [(64, 32), (128, 17), (64, 80), (32, 33)])
@pytest.mark.parametrize("n", [0, 256])
def test_more_heads_than_a_wave_has_columns(dev, D, H, n):
    """Past 16 query heads a kv head: several workgroups of the one-wave kernel a row, by the default choice and every code."""
    lens, nb, rows = [1, 77, 600], 0, []
    for c in lens:
        rows.append((list(range(nb, nb + -(-c // 16))), c))
        nb += -(-c // 16)
    q, kc, vc, m = batch(dev, rows, nb, H, 1, D, 16, H)
    split(m, H, D, dev, n, max(lens))
    for code in (None, 1, 2, 3, 7, 8, 11, 12):
        m.extra = {} if code is None else {"decode_nw": code}
        check(q, kc, vc, m, A.paged_attention(q, kc, vc, m, D ** -0.5, out=torch.full((3, H * D), 9.0, device=dev).bfloat16()))


@pytest.mark.parametrize("blocks", [9, 63, 67])
@pytest.mark.parametrize("n", [0, 512])
def test_behind_a_prefix(dev, blocks, n):
    D, H, G, BS = 128, 28, 4, 16
    pre, at, rows = list(range(blocks)), blocks, []
    for own in (1040, 77, 1205):  # keys behind the prefix
        k = -(-own // BS)
        rows.append((pre + list(range(at, at + k)), blocks * BS + own))
        at += k
    q, kc, vc, m = batch(dev, rows, at, H, G, D, BS, blocks)
    split(m, H, D, dev, n, max(c for _, c in rows))
    found, spans, _ = A.prefix_groups(m.block_tables.cpu().numpy(), np.array([c for _, c in rows]), BS, H // G)
    assert found.tolist() == [blocks * BS] * 3
    part, items, _ = A.cascade_layout(found, spans, A.cascade_items(3))
    i32 = lambda v: torch.from_numpy(v).to(dev)  # noqa: E731
    m.cascade = A.Cascade(pre_len=i32(found), pre_part=i32(part), items=i32(items.reshape(-1)), planes=8,
                          pre_o=torch.empty(8 * 3 * H * D, device=dev), pre_ml=torch.empty(8 * 3 * H * 2, device=dev))
    for code in (1, 3, 12):
        m.extra = {"decode_nw": code}
        check(q, kc, vc, m, A.paged_attention(q, kc, vc, m, D ** -0.5))


@pytest.mark.parametrize("seqs,takes", [(25, True), (26, False)])  # 200 and 208 parts in all
def test_few_parts_take_the_merging_kernel(dev, seqs, takes):
    D, H, G = 128, 28, 4
    lens = [257 + 9 * i for i in range(seqs)]
    nb, rows = 0, []
    for c in lens:
        rows.append((list(range(nb, nb + -(-c // 16))), c))
        nb += -(-c // 16)
    q, kc, vc, m = batch(dev, rows, nb, H, G, D, 16, seqs)
    split(m, H, D, dev, 256, 512)
    assert A.decode_mw_takes(m, G) == takes
    check(q, kc, vc, m, A.paged_attention(q, kc, vc, m, D ** -0.5))
    assert int(A.decode_counters(dev)[: seqs * G].abs().sum()) == 0


@pytest.mark.parametrize("n", [0, 128])
def test_rows_of_any_alignment(dev, n):
    """The merging kernel's output rows at strides and offsets that no 8-byte store takes; 3, 9 and 17 parts."""
    D, H, G = 64, 14, 2
    lens, nb, rows = [300, 1100, 2100], 0, []
    for c in lens:
        rows.append((list(range(nb, nb + -(-c // 16))), c))
        nb += -(-c // 16)
    q, kc, vc, m = batch(dev, rows, nb, H, G, D, 16, n)
    split(m, H, D, dev, n, max(lens))
    m.extra = {"decode_nw": 24}
    A.decode_counters(dev)
    out = torch.zeros(3, H * D + 3, dtype=torch.bfloat16, device=dev)
    check(q, kc, vc, m, A.paged_attention(q, kc, vc, m, D ** -0.5, out=out[:, 1:H * D + 1]))
    assert not out[:, 0].any() and not out[:, H * D + 1:].any()


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("code", [3, 24])
def test_infinite_values(dev, parts, code):
    """An infinite value in the last part stays an infinity of its sign: parts that are not there add nothing."""
    D, H, G = 64, 6, 2
    rows = [(list(range(8 * parts)), 128 * parts)]
    q, kc, vc, m = batch(dev, rows, 8 * parts, H, G, D, 16, parts)
    vc[-1, :, :, 5], vc[-1, :, :, 6] = float("inf"), float("-inf")
    split(m, H, D, dev, 128 if parts > 1 else 0, 128 * parts)
    m.extra = {"decode_nw": code}
    got = A.paged_attention(q, kc, vc, m, D ** -0.5).view(H, D).float()
    assert (got[:, 5] == float("inf")).all() and (got[:, 6] == float("-inf")).all()
    assert got[:, [d for d in range(D) if d not in (5, 6)]].isfinite().all()
