"""Decay attention, one token per sequence (csrc/kernels/seqmix.hip decay_step_kernel), against the plain fp32 recurrence: head
sizes around the row groups, fresh and kept states, empty portions, rotation."""
import pytest
import torch

from githubrepostorag_amd.ops.attention import AttnMetadata
from githubrepostorag_amd.ops.elementwise import rope_table
from githubrepostorag_amd.ops.recurrent import decay_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,vd", [(128, 128), (64, 64), (8, 4), (10, 36), (17, 128), (128, 64), (256, 64), (33, 256), (64, 256), (256, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rope", [False, True])
def test_decay_step(d, vd, dtype, rope):
    g = torch.Generator().manual_seed(d * 3 + vd)
    H, n = 3, 5
    rd = d // 2 // 2 * 2 if rope else 0
    proj = torch.randn(n, H * (2 * d + vd) + 5, generator=g).to(dtype)
    state = torch.randn(n + 2, H, d, vd, generator=g)
    decay = torch.tensor([1.0, 0.97, 0.5])
    slots = torch.tensor([4, 0, 2, 6, 1], dtype=torch.int32)
    i32 = dict(dtype=torch.int32)
    lens = [1, 9, 40, 1, 77]  # of 1: the state starts from zero, whatever the slot holds
    tab = rope_table(100, rd, 1e4) if rope else None
    got = []
    for dev in ("cpu", "cuda"):
        m = AttnMetadata(q_start=torch.arange(n + 1, **i32).to(dev), ctx_len=torch.tensor(lens, **i32).to(dev), block_tables=None,
                         slot_mapping=None, max_q_len=1, num_seqs=n, num_tokens=n, is_decode=True, state_slots=slots.to(dev))
        st = state.clone().to(dev)
        kw = dict(rope=tab.to(dev), positions=torch.tensor([x - 1 for x in lens], **i32).to(dev)) if rope else {}
        o = decay_attention(proj.to(dev), 0, H * d, 2 * H * d, decay.to(dev), st, m, H, d, vd, k_scale=0.7, **kw)
        got.append((o.float().cpu().view(n, H, vd), st.cpu()))
    (o0, s0), (o1, s1) = got
    # one fp32 multiply-add an element; d terms of a few units a sum
    assert (s0 - s1).abs().max() <= 4e-6
    assert (o0 - o1).abs().max() <= 2e-6 * d ** 0.5 * 8
