"""Causal convolution in four-channel accesses (csrc/kernels/ssm.hip causal_conv_vec_kernel) and its pool update, against the plain
form: portions around a token tile and shorter than the window, several in a step, fewer taps than the window, unaligned
weights, channels past a block."""
import pytest
import torch

from githubrepostorag_amd.ops.attention import AttnMetadata
from githubrepostorag_amd.ops.recurrent import causal_conv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,past", [([1, 2, 3], [5, 1, 0]), ([7, 8, 9, 1], [0, 4, 2, 0]), ([16, 17, 2], [9, 0, 1]), ([40], [3])])
@pytest.mark.parametrize("C,taps", [(8, 4), (1028, 4), (1024, 3), (12, 2), (20, 1), (36, 7)])
@pytest.mark.parametrize("dtype,shift", [(torch.bfloat16, 0), (torch.float32, 0), (torch.bfloat16, 1)])
def test_causal_conv(lens, past, C, taps, dtype, shift):
    g = torch.Generator().manual_seed(C + taps + sum(lens))
    n, T = len(lens), sum(lens)
    proj = torch.randn(T, C + 16, generator=g).to(dtype)
    w = torch.randn(C * taps + shift, generator=g)[shift:].view(C, taps)
    b = torch.randn(C, generator=g)
    cs = torch.randn(n + 2, taps - 1, C, generator=g).to(dtype)
    slots = torch.randperm(n + 2, generator=g)[:n].int()
    q = [0]
    for x in lens:
        q.append(q[-1] + x)
    got = []
    for dev in ("cpu", "cuda"):
        i32 = dict(dtype=torch.int32, device=dev)
        m = AttnMetadata(q_start=torch.tensor(q, **i32), ctx_len=torch.tensor([x + p for x, p in zip(lens, past)], **i32), block_tables=None,
                         slot_mapping=None, max_q_len=max(lens), num_seqs=n, num_tokens=T, state_slots=slots.to(dev))
        pool = cs.clone().to(dev)
        wd = torch.empty(C * taps + shift, device=dev)[shift:].view(C, taps).copy_(w)
        o = causal_conv(proj.to(dev), 4, wd, b.to(dev), pool, m)
        got.append((o.float().cpu(), pool.float().cpu()))
    (o0, s0), (o1, s1) = got
    assert torch.equal(s0, s1)
    # bf16: each rounds its result once (2^-8 of it); the sum of taps fp32 terms and the exponential
    assert ((o0 - o1).abs() <= o0.abs() * (2 ** -7 if dtype == torch.bfloat16 else 2e-6) + 4e-6).all()


@pytest.mark.parametrize("n", [65535 * 8, 65535 * 8 + 1])
def test_longest_portions(n):
    """Portions up to and past the most token tiles of the four-channel form."""
    g = torch.Generator(device="cuda").manual_seed(1)
    C, taps = 8, 4
    x = torch.randn(n, C, generator=g, device="cuda")
    w = torch.randn(C, taps, generator=g, device="cuda")
    pool = torch.randn(1, taps - 1, C, generator=g, device="cuda")
    before = torch.cat([pool[0], x])
    i32 = dict(dtype=torch.int32, device="cuda")
    m = AttnMetadata(q_start=torch.tensor([0, n], **i32), ctx_len=torch.tensor([n + 9], **i32), block_tables=None, slot_mapping=None,
                     max_q_len=n, num_seqs=1, num_tokens=n, state_slots=torch.zeros(1, **i32))
    y = causal_conv(x, 0, w, None, pool, m)
    want = torch.nn.functional.silu(sum(before[j:j + n] * w[:, j] for j in range(taps)))
    assert ((y - want).abs() <= 2e-6 * want.abs() + 4e-6).all() and torch.equal(pool[0], x[-(taps - 1):])
