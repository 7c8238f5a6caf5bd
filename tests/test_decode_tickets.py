"""The ticket words of the decode attention that merges its parts in the launch (ops/attention.py _decode_tickets): whose they are,
and the numbers where two streams of one thread launch it side by side."""
from types import SimpleNamespace

import pytest
import torch

from githubrepostorag_amd.ops import _lib
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


def test_a_capture_takes_the_words_only_of_an_owner_that_has_them(monkeypatch):
    m, own = step(torch.device("cpu")), {}
    assert A.decode_mw_takes(m, KV)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert not A.decode_mw_takes(m, KV)
    with G.WS.owned_by(own):
        assert not A.decode_mw_takes(m, KV)
        own["decode_tickets"] = {0: torch.zeros(1)}
        assert A.decode_mw_takes(m, KV)


@pytest.mark.gpu
@pytest.mark.parametrize("owned", [False, True])
def test_first_captured(dev, owned):
    """No eager step before the capture, in a thread that has none of the words."""
    import threading

    _lib.lib()
    got, failed = [], []

    def body():
        try:
            torch.cuda.set_device(dev)
            g = torch.Generator(device=dev).manual_seed(3)
            m = step(dev)
            q, kc, vc = (torch.randn(n, *s, generator=g, device=dev).bfloat16() for n, s in (
                (SEQS, (H, D)), (m.block_tables.numel(), (KV, 16, D)), (m.block_tables.numel(), (KV, 16, D))))
            graph, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
            torch.cuda.synchronize()
            owner = {}
            with torch.cuda.stream(s):
                if owned:
                    with G.WS.owned_by(owner), torch.cuda.graph(graph, stream=s):
                        got.append(A.paged_attention(q, kc, vc, m, D ** -0.5))
                else:
                    with torch.cuda.graph(graph, stream=s):
                        got.append(A.paged_attention(q, kc, vc, m, D ** -0.5))
                for _ in range(3):
                    got[0].zero_()
                    graph.replay()
            torch.cuda.synchronize()
            want = A.paged_attention_ref(q.float(), kc, vc, m, D ** -0.5).reshape(SEQS, -1)
            size = A.paged_attention_ref(q.float(), kc, vc.abs(), m, D ** -0.5).reshape(SEQS, -1)
            assert ((got[0].float() - want).abs() <= 1.05 * 2 ** -8 * (want.abs() + size)).all()
        except BaseException as e:  # raised by the test's own thread
            failed.append(e)

    t = threading.Thread(target=body)
    t.start()
    t.join(100)
    assert not t.is_alive() and got
    if failed:
        raise failed[0]


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
