"""The order in which the matrix-core scan deals its workgroups (csrc/kernels/linscan.hip scan_item): a step's portions
give, bit for bit, what each gives alone, whatever their lengths and number."""
import pytest
import torch

from githubrepostorag_amd.ops import recurrent
from githubrepostorag_amd.ops.attention import AttnMetadata

pytestmark = pytest.mark.gpu
H, D, VD = 3, 32, 64
# equal lengths, empty portions among others, lengths of whole parts and one more or less, rising and falling ones, 63 - 65 and
# 130 portions (up to 64 are sorted)
LENS = [[64, 64, 64], [0, 130, 0, 64, 1, 0], [128, 127, 129, 256, 255, 257], list(range(5, 400, 41)), list(range(400, 5, -41)),
        [1 + 37 * i % 211 for i in range(63)], [1 + 37 * i % 211 for i in range(64)], [1 + 37 * i % 211 for i in range(65)],
        [1 + 53 * i % 190 for i in range(130)]]


def _run(proj, decay, state, lens, slots, part, monkeypatch):
    q = [0]
    for n in lens:
        q.append(q[-1] + n)
    t = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    m = AttnMetadata(q_start=t(q), ctx_len=t([n + 1 for n in lens]), block_tables=None, slot_mapping=None, max_q_len=max(lens),
                     num_seqs=len(lens), num_tokens=q[-1], state_slots=t(slots))
    monkeypatch.setattr(recurrent, "_scan_taken", lambda *a: True)
    monkeypatch.setattr(recurrent, "_scan_part", lambda *a: part)
    return recurrent.decay_attention(proj, 0, H * D, 2 * H * D, decay, state, m, H, D, VD, act=False)


@pytest.mark.parametrize("part", [64, 128, 1 << 20])
@pytest.mark.parametrize("lens", LENS, ids=lambda v: f"{len(v)}x{max(v)}")
def test_portions_together_and_alone(dev, lens, part, monkeypatch):
    g = torch.Generator(device=dev).manual_seed(sum(lens))
    proj = torch.randn(sum(lens), H * (2 * D + VD), generator=g, device=dev).bfloat16()
    decay = torch.tensor([0.9, 0.99, 0.5], device=dev)
    start = torch.randn(len(lens), H, D, VD, generator=g, device=dev)
    together, apart = start.clone(), start.clone()
    out = _run(proj, decay, together, lens, list(range(len(lens))), part, monkeypatch)
    row = 0
    for i, n in enumerate(lens):
        if n:
            assert torch.equal(out[row:row + n], _run(proj[row:row + n], decay, apart, [n], [i], part, monkeypatch))
        row += n
    assert torch.equal(together, apart)
