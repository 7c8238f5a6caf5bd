"""The small-tile GEMM (csrc/kernels/gemm_pair.hip): every tile shape and epilogue against the 256 x 256 tile's results, bit
for bit, and the fp64 product within the rounding of the bf16 result; layouts; the products that linear() gives to it."""
import pytest
import torch
import torch.nn.functional as F

from githubrepostorag_amd.ops import gemm as G
from githubrepostorag_amd.ops import linear as L

# one row and column tile part, edges of 64 and 128 rows and of 64, 128 and 192 columns, one, two, three and many K steps
SIZES = [(1, 8, 128), (64, 64, 128), (65, 72, 192), (127, 192, 256), (129, 200, 320), (300, 1000, 768), (257, 448, 64)]


def _mk(dev, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    return r(M, K).bfloat16(), (r(N, K) * K ** -0.5).bfloat16(), r(N).bfloat16()


# half an ulp of bf16 (2^-9) of the value; fp32 sums of K terms of order 1 / sqrt(K) and the activation's rounding on top
TOL = dict(rtol=2 ** -8, atol=2 ** -8 * 0.05)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", range(4))
@pytest.mark.parametrize("M,N,K", SIZES)
def test_epilogues(dev, M, N, K, shape):
    x, w, b = _mk(dev, M, N, K)
    for bias in (None, b):
        ref = x.double() @ w.double().T + (0 if bias is None else bias.double())
        for act, fn in ((G.ACT_NONE, lambda t: t), (G.ACT_GELU, F.gelu), (G.ACT_GELU_TANH, lambda t: F.gelu(t, approximate="tanh"))):
            got = G.gemm_pair(x, w, bias, shape, act=act)
            torch.testing.assert_close(got.double(), fn(ref), **TOL)
            if K >= 128:
                assert torch.equal(got, G.gemm(x, w, bias, act=act, ksplit=1, sk=0))
        if N % 64 == 0:
            got = G.gemm_pair(x, w, bias, shape, G.EPI_SILU)
            gate, up = G.deinterleave_gate_up(ref.T.contiguous())
            torch.testing.assert_close(got.double(), (F.silu(gate) * up).T, **TOL)
            if K >= 128:
                assert torch.equal(got, G.gemm_silu(x, w, bias, ksplit=1, sk=0))
    if N % 16 == 0:
        got = G.gemm_pair(x, w, None, shape, G.EPI_GLU, glu=(7.0, 1.702, 1.0))
        gate, up = (x.double() @ w.double().T).chunk(2, 1)
        gate = gate.clamp(max=7.0)
        torch.testing.assert_close(got.double(), gate * torch.sigmoid(1.702 * gate) * (up.clamp(-7, 7) + 1), **TOL)


@pytest.mark.gpu
def test_layouts(dev):
    """A column slice of a wider input, one row for all (stride 0), a result between other columns and rows."""
    x, w, b = _mk(dev, 200, 328, 256)
    wide = torch.randn(200, 512, device=dev).bfloat16()
    want = G.gemm_pair(wide[:, 128:384].contiguous(), w, b, 3)
    for shape in range(4):
        assert torch.equal(G.gemm_pair(wide[:, 128:384], w, b, shape), want)
        assert torch.equal(G.gemm_pair(x[:1].expand(200, 256), w, b, shape), G.gemm_pair(x[:1], w, b, shape).expand(200, 328))
        big = torch.full((202, 352), 7.0, dtype=torch.bfloat16, device=dev)
        G.gemm_pair(wide[:, 128:384], w, b, shape, out=big[1:201, 8:336])
        assert torch.equal(big[1:201, 8:336], want)
        big[1:201, 8:336] = 7.0
        assert bool((big == 7.0).all())


def test_rule(monkeypatch):
    monkeypatch.setattr(G, "_NCU", [256])
    assert [G.pair_plan(M, 768, 768) for M in (20, 33, 300, 2688, 2752)] == [None, 3, 3, 3, None]  # 504, 516 tiles
    assert [G.pair_plan(M, 3072, 768, True) for M in (1, 300, 1136, 1752, 4200)] == [3, 3, 2, 1, None]
    assert G.pair_plan(300, 3072, 1088) is None and G.pair_plan(300, 22016, 4096, True) is None  # deep
    assert G.pair_fills(24000, 768, 768) and not G.pair_fills(12000, 2304, 768) and not G.pair_fills(21504, 768, 768)
    # rows, width, depth, library and owned us (the latter in tiles of 192 rows at 900, 1187, 1641 x 18944 and 2405 x 8192); runs of one
    # side differ by 2 %
    for M, N, K, lib, own in [(2405, 18944, 3584, 365, 237), (4000, 18944, 3584, 502, 387), (1641, 18944, 3584, 207, 192),
                              (900, 18944, 3584, 134, 126), (1187, 8192, 1536, 30.9, 32.1), (1641, 8192, 1536, 40.1, 40.4),
                              (2405, 8192, 1536, 59.4, 59.7), (1632, 10752, 1536, 71.1, 61.2), (2594, 12288, 6144, 326, 315)]:
        assert (G.wide_plan(M, N, K) is not None) == (own < 1.02 * lib), (M, N, K)
    assert G.wide_plan(4000, 3584, 3584) is None  # a measured shape keeps its rows


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,kind,shape", [(40, 768, 768, "pair", 3), (300, 2304, 768, "pair", 3), (700, 18944, 1536, "tile_prefill", None),
                                              (8000, 2304, 768, "tile_prefill", 0)])
def test_linear(dev, monkeypatch, M, N, K, kind, shape):
    """Plain products that linear() runs here, with a gradient on the library's."""
    x, w, b = _mk(dev, M, N, K)
    took = []
    monkeypatch.setattr(G, "gemm_pair", lambda *a, _f=G.gemm_pair, **k: took.append(a[3]) or _f(*a, **k))
    assert L.kernel_for(M, N, K) == kind
    assert torch.equal(L.linear(x, w, b), G.gemm(x, w, b, ksplit=1, sk=0)) and took == ([] if shape is None else [shape])
    ref = x.double() @ w.double().T + b.double()
    torch.testing.assert_close(L.linear(x, w, b).double(), ref, **TOL)
    w.requires_grad_(True)
    y = L.linear(x, w, b)
    y.sum().backward()
    assert w.grad is not None and w.grad.shape == w.shape


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,shape", [(2944, 1024, 1024, 3), (640, 1024, 4096, 3), (2900, 1024, 4096, 2), (6528, 1024, 1024, 1),
                                         (2150, 2048, 1536, 0), (10880, 1024, 4096, None)])
def test_linear_of_a_bucket_that_stays_owned(dev, monkeypatch, M, N, K, shape):
    """Measured products that keep the owned kernels: the tile of the bucket's row, bit for bit the 256 x 256 tile's; a gradient
    on the library's."""
    x, w, b = _mk(dev, M, N, K)
    monkeypatch.setattr(G, "gemm_pair", lambda *a, _f=G.gemm_pair, **k: took.append(a[3]) or _f(*a, **k))
    took = []
    y = L.linear(x, w, b)
    assert took == ([] if shape is None else [shape]) and torch.equal(y, G.gemm(x, w, b, ksplit=1, sk=0))
    torch.testing.assert_close(y.double(), x.double() @ w.double().T + b.double(), **TOL)
    w.requires_grad_(True)
    assert L.linear(x, w, b).requires_grad


@pytest.mark.gpu
def test_captured_without_an_eager_step(dev):
    """A product that has no slab can be captured before any eager one."""
    x, w, b = _mk(dev, 100, 3072, 768)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    assert G.capture_ok(x.device, 100, 3072, 768, act=G.ACT_GELU)
    with G.WS.owned_by({}), torch.cuda.graph(g):
        y = G.gemm(x, w, b, act=G.ACT_GELU)
    for _ in range(3):
        x.normal_()
        g.replay()
        assert torch.equal(y, G.gemm(x, w, b, act=G.ACT_GELU))


@pytest.mark.parametrize("at", [0, 4])
def test_gate_up_captured_with_a_bias_at_any_address(monkeypatch, at):
    """A bias that the small tiles refuse (no multiple of 8 bytes), in a capture whose slab was not sized: the library's branch
    and no K parts.  (On a host that launches nothing.)"""
    from types import SimpleNamespace

    M, F, K = 300, 1536, 2048  # K parts without the small tiles
    b = torch.zeros(2 * F + 8).bfloat16()[at // 2:][:2 * F]
    w = torch.empty(2 * F, 1).bfloat16().expand(2 * F, K)
    x = SimpleNamespace(shape=(M, K), is_cuda=True, device=torch.device("cpu"), dtype=torch.bfloat16, stride=lambda i: K if i == 0 else 1,
                        data_ptr=lambda: 0)
    monkeypatch.setattr(G, "_NCU", [256])
    monkeypatch.setattr(G, "supported", lambda *a: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert G.pair_plan(M, 2 * F, K, True) is not None and G.schedule(M, 2 * F, K, True)[0] > 1
    took = []
    monkeypatch.setattr(torch.nn.functional, "linear", lambda *a: took.append("library") or torch.zeros(M, 2 * F).bfloat16())
    monkeypatch.setattr(G, "gemm_silu", lambda *a: took.append("pair" if G.pair_takes(*a) else "parts"))
    with G.WS.owned_by({}):
        G.mlp_gate_up(x, w, b)
    assert took == (["library"] if at else ["pair"])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,other", [(100, 768, 768, "decode"), (256, 768, 1024, "decode"), (700, 768, 768, "library")])
@pytest.mark.parametrize("at", [8, 4, 2])
def test_linear_with_a_bias_at_any_address(dev, monkeypatch, M, N, K, other, at):
    """What the small tiles refuse goes to the kernel that the shape has without them; a bias at 8 bytes they take."""
    x, w, b = _mk(dev, M, N, K)
    b = torch.cat([b[: at // 2], b])[at // 2:]
    assert L.kernel_for(M, N, K) == "pair" and L.kernel_for(M, N, K, pair_ok=False) == other
    took = []
    for name in ("gemm_pair", "gemm_decode", "gemm"):
        monkeypatch.setattr(G, name, lambda *a, _f=getattr(G, name), _n=name, **k: took.append(_n) or _f(*a, **k))
    y = L.linear(x, w, b)
    assert took == (["gemm_pair"] if at == 8 else ["gemm_decode"] if other == "decode" else [])
    torch.testing.assert_close(y.double(), x.double() @ w.double().T + b.double(), **TOL)


@pytest.mark.gpu
@pytest.mark.parametrize("K,takes", [(768, True), (1024, True), (1088, False)])
def test_rounds_of_small_tiles(dev, K, takes):
    """Short contractions of more tiles than CUs go in small tiles up to three of them a CU: 255, 258, 288 and 291 tiles on 256 CUs, the
    last two of 768 and 776 small ones."""
    if G._num_cus() != 256:
        pytest.skip("the row counts are those of 256 CUs")
    assert [G.pair_fills(t * 256, 768, K) for t in (85, 86, 96, 97)] == [False, takes, takes, False]
    x, w, b = _mk(dev, 86 * 256 - 7, 768, K)
    assert torch.equal(G.gemm(x, w, b), G.gemm(x, w, b, ksplit=1, sk=0))


@pytest.mark.parametrize("M,N,K,act,chain,takes", [
    (42419, 384, 384, False, True, True), (32768, 384, 384, False, True, False), (50611, 384, 384, False, True, False),  # (three a CU)
    (50611, 384, 384, True, True, True), (50611, 384, 448, True, True, False), (66000, 384, 384, True, True, False),  # (four with GELU)
    (300, 36864, 768, False, True, False), (300, 36864, 768, True, True, True), (1600, 10752, 512, False, True, True),  # (few rows)
    (68787, 128, 256, False, True, True), (68787, 128, 320, False, True, False),  # (a deep column)
    (27000, 768, 768, False, True, False), (27000, 768, 768, False, False, True), (28000, 768, 768, False, False, False)])  # (no chains)
def test_lines_of_small_tiles(monkeypatch, M, N, K, act, chain, takes):
    monkeypatch.setattr(G, "_NCU", [256])
    assert G.pair_fills(M, N, K, act, chain) == takes


@pytest.mark.gpu
@pytest.mark.parametrize("at,took", [(0, 0), (4, 1)])
def test_small_tiles_without_chains(dev, monkeypatch, at, took):
    """A bias at an address that chains do not take: small tiles up to 0.62 of the rounds, and the same results."""
    if G._num_cus() != 256:
        pytest.skip("the row counts are those of 256 CUs")
    x, w, b = _mk(dev, 97 * 256, 768, 192)
    b = torch.cat([b, b[:at]])[at:] if at else b
    calls, pair = [], G.gemm_pair
    monkeypatch.setattr(G, "gemm_pair", lambda *a, **k: calls.append(1) or pair(*a, **k))
    y = G.gemm(x, w, b)
    assert len(calls) == took
    torch.testing.assert_close(y.double(), x.double() @ w.double().T + b.double(), **TOL)
