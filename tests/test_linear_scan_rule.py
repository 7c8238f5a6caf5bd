"""Which kernels a prompt step of the linear recurrences runs (ops/recurrent.py _scan_taken): the side that was measured faster."""
from types import SimpleNamespace

import pytest
import torch

from githubrepostorag_amd.ops import recurrent
from githubrepostorag_amd.ops.attention import AttnMetadata

RAGGED = [1900, 600, 1500, 300, 1700, 1292, 900]
# dtype, SiLU, lens, heads, d, vd, us of the matrix-core scan and of the one-pass kernels
MEASURED = [
    ("f32", False, [64] * 64, 28, 16, 16, 153, 54), ("f32", False, RAGGED, 28, 8, 8, 370, 100), ("f32", False, [8] * 64, 28, 128, 128, 376, 108),
    ("f32", False, [20] * 30, 12, 8, 8, 25, 21), ("bf16", True, RAGGED, 28, 33, 65, 886, 552), ("bf16", True, [24] * 64, 28, 96, 96, 320, 199),
    ("bf16", False, [64] * 64, 28, 8, 8, 43, 36), ("bf16", True, [64] * 64, 28, 16, 32, 147, 65),
    ("f32", False, RAGGED, 28, 128, 128, 1335, 2014), ("f32", True, [1187], 12, 64, 64, 57, 281), ("bf16", True, [64] * 64, 28, 96, 96, 370, 481),
    ("bf16", False, RAGGED, 4, 48, 48, 54, 246), ("bf16", True, [1187], 12, 33, 65, 63, 160), ("bf16", False, [64], 4, 8, 8, 16, 28),
    ("bf16", True, RAGGED, 28, 128, 128, 677, 2159), ("bf16", True, [1187], 12, 128, 128, 54, 517), ("bf16", False, RAGGED, 28, 128, 128, 214, 2057),
    ("bf16", True, [30] * 20, 28, 128, 128, 75, 175), ("bf16", False, [16] * 64, 28, 128, 128, 65, 180), ("bf16", False, [8] * 4, 12, 128, 128, 14, 51),
]


@pytest.mark.parametrize("dtype,act,lens,H,d,vd,scan,passes", MEASURED)
def test_rule(dtype, act, lens, H, d, vd, scan, passes, monkeypatch):
    monkeypatch.setattr(recurrent, "lib", lambda: SimpleNamespace(grag_linear_scan_max_dim=lambda: 128))
    m = AttnMetadata(q_start=None, ctx_len=None, block_tables=None, slot_mapping=None, max_q_len=max(lens), num_seqs=len(lens),
                     num_tokens=sum(lens))
    x = torch.empty(2, H * (2 * d + vd), dtype=torch.float32 if dtype == "f32" else torch.bfloat16)
    exact = recurrent._scan_exact(x, (0, H * d, 2 * H * d), d, vd)
    assert recurrent._scan_taken(m, sum(lens), H, d, vd, act or dtype == "f32", exact) == (scan < passes)


# longest portion, tokens, portions, heads, d, vd, operands in three parts, us by chunks a part
CUTS = [(914, 1500, 2, 8, 64, 128, True, {1: 89, 2: 65, 3: 84, 4: 106, 8: 192, 15: 253}),
        (551, 800, 2, 28, 16, 16, True, {1: 67, 2: 53, 3: 69, 4: 87, 9: 122}),
        (800, 800, 1, 12, 128, 128, False, {1: 33, 2: 26, 3: 30, 4: 35, 6: 46, 8: 59, 13: 62}),
        (8192, 8192, 1, 12, 128, 128, True, {1: 646, 2: 320, 3: 297, 4: 231, 6: 246, 8: 264, 16: 274, 32: 530, 128: 1427}),
        (3094, 4096, 2, 28, 128, 128, False, {1: 354, 2: 155, 3: 118, 4: 114, 6: 111, 8: 98, 12: 130, 16: 113, 49: 225}),
        (8192, 8192, 1, 80, 16, 64, False, {1: 1107, 2: 559, 4: 419, 8: 384, 12: 421, 16: 453, 24: 422, 32: 514, 128: 1125})]


@pytest.mark.parametrize("max_q,tokens,nseq,H,d,vd,split,us", CUTS)
def test_cut(max_q, tokens, nseq, H, d, vd, split, us):
    """A portion's cut within 1.15 of the best that was measured."""
    part = recurrent._scan_part(max_q, tokens, nseq, H * -(-vd // 64), split, d)
    assert part % 64 == 0 and us[min(part // 64, max(us))] <= 1.15 * min(us.values())


def test_exact_rows():
    x = torch.empty(4, 400, dtype=torch.bfloat16)
    ok = recurrent._scan_exact
    assert ok(x, (0, 64, 128), 64, 64) and ok(x, (0, 4, 8), 32, 128, 16) and ok(x[:, 4:], (0, 4, 8), 128, 64)
    assert not (ok(x.float(), (0, 64, 128), 64, 64) or ok(x, (0, 64, 128), 64, 65) or ok(x, (0, 64, 128), 48, 64) or ok(x, (0, 2, 8), 64, 64)
                or ok(x[:, 1:], (0, 4, 8), 64, 64) or ok(x, (0, 4, 8), 64, 64, 20) or ok(torch.empty(4, 401, dtype=torch.bfloat16), (0, 4, 8), 64, 64))
