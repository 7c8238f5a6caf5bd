"""The ticket words of the decode attention that merges its parts in the launch (ops/attention.py _decode_tickets): whose they are,
and the numbers where two streams of one thread launch it side by side."""
from types import SimpleNamespace

import pytest
import torch

from githubrepostorag_amd.ops import attention as A
from githubrepostorag_amd.ops import gemm as G

SEQS, H, KV, D = 24, 28, 4, 128  # 24 sequences of 300 keys in two parts: 192 parts in all


def step(dev, num_splits=2):
    lens = [300 + i for i in range(SEQS)]
    width = -(-max(lens) // 16)
    return A.AttnMetadata(q_start=torch.arange(SEQS + 1, dtype=torch.int32, device=dev),
                          ctx_len=torch.tensor(lens, dtype=torch.int32, device=dev),
                          block_tables=torch.arange(SEQS * width, dtype=torch.int32, device=dev).view(SEQS, width), slot_mapping=None,
                          max_q_len=1, num_seqs=SEQS, num_tokens=SEQS, is_decode=True, num_splits=num_splits, split_len=256,
                          part_o=torch.empty(num_splits * SEQS * H * D, device=dev),
                          part_ml=torch.empty(num_splits * SEQS * H * 2, device=dev))


@pytest.fixture
def launches(monkeypatch):
    """A host that records the launches and makes none: f(stream) -> (entry point, its tickets' address)."""
    at, seen = [0], []
    cpu = torch.device("cpu")
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: SimpleNamespace(cuda_stream=at[0]))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(G._Workspace, "scratch", lambda self, name, dev, make: (
        self.owner() if self.owner() is not None else thread).setdefault(name, make(cpu)))
    monkeypatch.setattr(A, "call", lambda name, *a: seen.append((name, a[-3])))
    thread = {}
    q = SimpleNamespace(shape=(SEQS, H, D), is_cuda=True, device=cpu, dtype=torch.bfloat16, stride=lambda i: H * D, data_ptr=lambda: 0)
    kc = torch.empty(SEQS * 19, KV, 16, 1, dtype=torch.bfloat16).expand(-1, -1, -1, D)

    def launch(stream):
        at[0] = stream
        A.paged_attention(q, kc, kc, step(cpu), D ** -0.5)
        return seen[-1]

    yield launch
    getattr(G.WS._tls, "tickets", {}).clear()


def test_streams_of_one_thread_share_no_words(launches):
    (n1, t1), (n2, t2), (n3, t3) = launches(1), launches(2), launches(1)
    assert n1 == n2 == n3 == "grag_paged_decode_mw" and t1 == t3 != t2
    own, other = {}, {}
    with G.WS.owned_by(own):  # (an owner runs on one stream at a time)
        a, b = launches(1)[1], launches(2)[1]
    with G.WS.owned_by(other):
        c = launches(1)[1]
    assert a == b == own["decode_tickets"].data_ptr() and c not in (a, t1, t2)


@pytest.mark.gpu
def test_two_streams_of_one_thread(dev):
    g = torch.Generator(device=dev).manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    work, wait = [], torch.cuda.current_stream()
    for _ in range(2):
        m = step(dev)
        q, kc, vc = r(SEQS, H, D), r(m.block_tables.numel(), KV, 16, D), r(m.block_tables.numel(), KV, 16, D)
        s = torch.cuda.Stream()
        s.wait_stream(wait)
        work.append((s, (q, kc, vc, m, D ** -0.5), []))
    for _ in range(200):  # side by side: neither stream waits for the other
        for s, args, out in work:
            with torch.cuda.stream(s):
                out.append(A.paged_attention(*args))
    torch.cuda.synchronize()
    for _, (q, kc, vc, m, scale), out in work:
        want = A.paged_attention_ref(q.float(), kc, vc, m, scale).reshape(SEQS, -1)
        size = A.paged_attention_ref(q.float(), kc, vc.abs(), m, scale).reshape(SEQS, -1)
        for o in out:  # the weights and the result are rounded to bf16's 8 bits; 1.05 for fp32's sums and exponents
            assert ((o.float() - want).abs() <= 1.05 * 2 ** -8 * (want.abs() + size)).all()
