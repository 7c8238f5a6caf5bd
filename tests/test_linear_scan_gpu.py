"""The matrix-core scan of the decay linear attention and of the state-space mixer (csrc/kernels/linscan.hip) against the
recurrences written out in 64 bits: sizes around its tiles (64 tokens, 64 columns, 32 rows), portions cut into parts,
carried states, every form of its operands."""
import pytest
import torch

from githubrepostorag_amd.ops import recurrent
from githubrepostorag_amd.ops.attention import AttnMetadata

pytestmark = pytest.mark.gpu
# Both sides sum the same terms; B is the same recurrence over their absolute values.  fp32 sums of up to 64 + 128 terms
# round by at most (64 + 128) / 2 ulp of 6e-8 of B in the worst order, and the weights 2^(L_t - L_s) carry a few ulp more.
TOL = 1.2e-5


@pytest.fixture(autouse=True)
def _scan(monkeypatch):
    """The kernels of this file, whatever the rule would take."""
    monkeypatch.setattr(recurrent, "_scan_taken", lambda *a: True)


def _meta(lens, past, dev):
    q = [0]
    for n in lens:
        q.append(q[-1] + n)
    t = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    return AttnMetadata(q_start=t(q), ctx_len=t([n + p for n, p in zip(lens, past)]), block_tables=None, slot_mapping=None,
                        max_q_len=max(lens), num_seqs=len(lens), num_tokens=q[-1],
                        state_slots=t([len(lens) - 1 - i for i in range(len(lens))])), q


def _walk(a, k, v, q, S):
    """S_t = a_t S + k_t v_t^T, o_t = S_t^T q_t over [n, H, ...] float64."""
    out = []
    for t in range(q.shape[0]):
        S = a[t][:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out), S


def _check(got, want, bound, what):
    worst = ((got.double().cpu() - want).abs() / (bound + 1e-30)).max().item()
    assert worst < TOL, f"{what}: {worst:.2e} of the bound"


CASES = [
    # lens, past, H, d, vd, dtype, act, rope dims, part
    ([64], [0], 2, 128, 128, torch.bfloat16, False, 0, 64),
    ([65, 8, 130], [0, 7, 3], 3, 128, 64, torch.bfloat16, True, 0, 1 << 20),
    ([200, 63, 1], [0, 5, 0], 2, 24, 40, torch.bfloat16, False, 0, 64),
    ([300, 129], [0, 9], 2, 128, 128, torch.bfloat16, True, 0, 128),
    ([257], [4], 3, 33, 65, torch.bfloat16, True, 22, 64),
    ([190, 64], [0, 1], 2, 100, 70, torch.float32, False, 0, 64),
    ([130], [0], 1, 17, 9, torch.float32, True, 6, 64),
    ([9], [2], 2, 5, 3, torch.bfloat16, False, 0, 64),
    # the sizes of 32, 64 and 128 rows that are compiled for themselves
    ([130, 64], [0, 5], 3, 32, 64, torch.bfloat16, False, 0, 64),
    ([257, 33], [3, 0], 2, 32, 128, torch.bfloat16, True, 16, 128),
    ([100, 129], [0, 7], 2, 64, 128, torch.bfloat16, False, 0, 1 << 20),
    ([300], [9], 3, 64, 64, torch.bfloat16, True, 64, 64),
    ([191, 20], [0, 30], 2, 64, 64, torch.bfloat16, True, 0, 1 << 20),
    ([140, 65], [11, 0], 2, 128, 64, torch.bfloat16, True, 64, 64),
    ([200], [0], 2, 128, 128, torch.bfloat16, False, 40, 128),
]


@pytest.mark.parametrize("lens,past,H,d,vd,dtype,act,rd,part", CASES)
def test_decay_scan(lens, past, H, d, vd, dtype, act, rd, part, monkeypatch):
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(sum(lens) + d)
    m, qs = _meta(lens, past, dev)
    T = qs[-1]
    monkeypatch.setattr(recurrent, "_scan_part", lambda *a: part)
    pad = 0 if d % 4 == 0 else 3  # odd sizes go with rows that are not aligned
    proj = torch.randn(T, H * (2 * d + vd) + pad, generator=g).to(dtype)
    decay = torch.tensor([1.0, 0.0, -0.97][:H] if d < 64 else [0.996, 0.05, 0.75][:H])
    state = torch.randn(len(lens) + 1, H, d, vd, generator=g)
    rope = torch.randn(512, rd, generator=g) if rd else None
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(lens, past)]).to(torch.int32)
    ks = 0.3
    st = state.to(dev)
    got = recurrent.decay_attention(proj.to(dev), 0, H * d, 2 * H * d, decay.to(dev), st, m, H, d, vd, act=act,
                                    positions=pos.to(dev) if rd else None, rope=rope.to(dev) if rd else None, k_scale=ks)
    x = proj.double()
    f = torch.nn.functional.silu if act else (lambda t: t)
    q, k = (f(x[:, o:o + H * d]).view(T, H, d) for o in (0, H * d))
    v = f(x[:, 2 * H * d:2 * H * d + H * vd]).view(T, H, vd)

    def rot(t):
        if not rd:
            return t
        c, s = (rope.double()[pos.long()][:, None, o:o + rd // 2] for o in (0, rd // 2))
        u, w = t[..., :rd // 2], t[..., rd // 2:rd]
        return torch.cat([u * c - w * s, w * c + u * s, t[..., rd:]], -1)

    q, k = rot(q), rot(k) * ks
    for i, (a, b) in enumerate(zip(qs, qs[1:])):
        slot = len(lens) - 1 - i
        lam = decay.double().expand(b - a, H)
        S0 = state[slot].double() if past[i] else torch.zeros(H, d, vd, dtype=torch.float64)
        o, S = _walk(lam, k[a:b], v[a:b], q[a:b], S0)
        bo, bS = _walk(lam.abs(), k[a:b].abs(), v[a:b].abs(), q[a:b].abs(), S0.abs())
        _check(got[a:b].view(-1, H, vd), o, bo, "outputs")
        _check(st[slot], S, bS, "state")
    assert torch.equal(st[len(lens)].cpu(), state[len(lens)])


SSM = [
    # lens, past, H, G, N, P, dtype, part
    ([64, 70], [0, 3], 4, 1, 128, 64, torch.bfloat16, 1 << 20),
    ([300, 65, 8], [0, 0, 11], 6, 2, 128, 64, torch.bfloat16, 64),
    ([193], [5], 6, 2, 12, 8, torch.bfloat16, 128),
    ([129, 128], [0, 2], 3, 3, 50, 67, torch.float32, 64),
    ([130, 64], [0, 4], 4, 2, 32, 64, torch.bfloat16, 64),
    ([257], [3], 2, 1, 64, 64, torch.bfloat16, 128),
    ([66, 190], [0, 1], 2, 1, 64, 128, torch.bfloat16, 1 << 20),
]


@pytest.mark.parametrize("lens,past,H,G,N,P,dtype,part", SSM)
def test_state_space_scan(lens, past, H, G, N, P, dtype, part, monkeypatch):
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(sum(lens) + N)
    m, qs = _meta(lens, past, dev)
    T = qs[-1]
    monkeypatch.setattr(recurrent, "_scan_part", lambda *a: part)
    xbc = torch.randn(T, H * P + 2 * G * N, generator=g).to(dtype)
    proj = (2 * torch.randn(T, H + 5, generator=g)).to(dtype)
    dtb, alog, skip = torch.randn(H, generator=g), torch.linspace(-2.0, 3.0, H), torch.randn(H, generator=g)
    state = torch.randn(len(lens) + 1, H, N, P, generator=g)
    st = state.to(dev)
    got = recurrent.ssm_scan(xbc.to(dev), proj.to(dev), 2, dtb.to(dev), alog.to(dev), skip.to(dev), st, m, H, G, N, P)
    x = xbc.double()
    v = x[:, :H * P].view(T, H, P)
    Bm, Cm = (x[:, H * P + o * G * N:H * P + (o + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for o in (0, 1))
    dt = torch.nn.functional.softplus(proj.double()[:, 2:2 + H] + dtb.double(), threshold=60.0)
    a = torch.exp(-torch.exp(alog.double()) * dt)
    k = Bm * dt[:, :, None]
    for i, (s, e) in enumerate(zip(qs, qs[1:])):
        slot = len(lens) - 1 - i
        S0 = state[slot].double() if past[i] else torch.zeros(H, N, P, dtype=torch.float64)
        o, S = _walk(a[s:e], k[s:e], v[s:e], Cm[s:e], S0)
        bo, bS = _walk(a[s:e], k[s:e].abs(), v[s:e].abs(), Cm[s:e].abs(), S0.abs())
        extra = skip.double()[:, None] * v[s:e]
        _check(got[s:e].view(-1, H, P), o + extra, bo + extra.abs(), "outputs")
        _check(st[slot], S, bS, "state")


def _walk32(a, k, v, q, S):
    """_walk in the kernels' own 32 bits."""
    out = []
    for t in range(q.shape[0]):
        S = a[t][:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out), S


def _same(got, want, what):
    """Infinite, no number and finite in the same places, and the finite numbers close to each other."""
    assert torch.equal(got.isnan(), want.isnan()), f"{what}: NaN"
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[got.isinf()], want[want.isinf()]), f"{what}: inf"
    f = want.isfinite()
    # (positive terms alone: no sum cancels, so TOL holds relative to the result, and the reference is a 32-bit one)
    assert ((got[f] - want[f]).abs() <= 2 * TOL * want[f].abs() + 1e-30).all(), what


@pytest.mark.parametrize("part", [64, 1 << 20])
@pytest.mark.parametrize("d,vd,dtype,act", [(128, 64, torch.bfloat16, False), (128, 128, torch.bfloat16, True), (24, 40, torch.bfloat16, False),
                                            (64, 64, torch.bfloat16, True), (20, 70, torch.float32, True)])
def test_numbers_past_the_products(d, vd, dtype, act, part, monkeypatch):
    """Infinities, NaN and numbers at the end of the range in v, k, q and the carried state: a token sees those of the tokens
    before it and of itself, in their own columns, and no other."""
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(d + vd)
    H, lens, past = 7, [200, 140], [0, 3]
    m, qs = _meta(lens, past, dev)
    T = qs[-1]
    monkeypatch.setattr(recurrent, "_scan_part", lambda *a: part)
    q, k, v = (torch.rand(T, H, n, generator=g) + 0.1 for n in (d, d, vd))
    state = torch.rand(3, H, d, vd, generator=g)
    inf = float("inf")
    v[70, 0, 5] = inf
    v[qs[1] + 10, 1, 3], v[qs[1] + 40, 1, 3], v[qs[1] + 90, 1, 2] = inf, -inf, float("nan")
    k[130, 2, 7] = inf
    q[100, 3, 2] = inf
    state[0, 4, 2, 6], state[0, 4, 1, 1] = inf, 3.4e38  # (the second sequence's slot)
    q[:, 4] *= 2.0 ** -9
    v[150, 5, 0], q[:, 5] = 3.38e38, q[:, 5] * 2.0 ** -9
    v[33, 6, 1], k[34, 6, 2] = (-inf, -3e38) if act else (inf, 1e30)
    proj = torch.cat([t.reshape(T, -1) for t in (q, k, v)], 1).to(dtype)
    decay = torch.tensor([0.996, 0.75, 0.5, 1.0, 0.9, 0.95, 0.8])
    st = state.to(dev)
    got = recurrent.decay_attention(proj.to(dev), 0, H * d, 2 * H * d, decay.to(dev), st, m, H, d, vd, act=act, k_scale=0.5)
    got = got.float().cpu().view(T, H, vd)
    x = proj.float()
    f = (lambda t: t / (1 + torch.exp(-t))) if act else (lambda t: t)
    q, k = (f(x[:, o:o + H * d]).view(T, H, d) for o in (0, H * d))
    v = f(x[:, 2 * H * d:]).view(T, H, vd)
    for i, (a, b) in enumerate(zip(qs, qs[1:])):
        S0 = state[1 - i] if past[i] else torch.zeros(H, d, vd)
        o, S = _walk32(decay.expand(b - a, H), k[a:b] * 0.5, v[a:b], q[a:b], S0)
        for h in range(H):
            _same(got[a:b, h], o[:, h], f"outputs of sequence {i}, head {h}")
            _same(st[1 - i, h].cpu(), S[h], f"state of sequence {i}, head {h}")


@pytest.mark.parametrize("part", [64, 1 << 20])
@pytest.mark.parametrize("N,P,dtype", [(128, 64, torch.bfloat16), (32, 128, torch.bfloat16), (12, 8, torch.float32)])
def test_state_space_past_the_products(N, P, dtype, part, monkeypatch):
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(N + P)
    H, n = 4, 150
    m, _ = _meta([n], [5], dev)
    monkeypatch.setattr(recurrent, "_scan_part", lambda *a: part)
    x, B, C = torch.rand(n, H, P, generator=g) + 0.1, torch.rand(n, N, generator=g) + 0.1, torch.rand(n, N, generator=g) + 0.1
    dt = torch.rand(n, H, generator=g)
    x[70, 0, 5], x[100, 1, 2], dt[80, 2] = float("inf"), float("nan"), float("inf")
    xbc, proj = torch.cat([x.reshape(n, -1), B, C], 1).to(dtype), dt.to(dtype)
    dtb, alog, skip = torch.zeros(H), torch.linspace(-2.0, 0.0, H), torch.rand(H, generator=g)
    state = torch.rand(1, H, N, P, generator=g)
    st = state.to(dev)
    got = recurrent.ssm_scan(xbc.to(dev), proj.to(dev), 0, dtb.to(dev), alog.to(dev), skip.to(dev), st, m, H, 1, N, P)
    got = got.float().cpu().view(n, H, P)
    f = xbc.float()
    v, B, C = f[:, :H * P].view(n, H, P), f[:, H * P:H * P + N], f[:, H * P + N:]
    dt = torch.nn.functional.softplus(proj.float() + dtb)
    o, S = _walk32(torch.exp(-torch.exp(alog) * dt), B[:, None] * dt[:, :, None], v, C[:, None].expand(n, H, N), state[0])
    o = o + skip[:, None] * v
    for h in range(H):
        _same(got[:, h], o[:, h], f"outputs of head {h}")
        _same(st[0, h].cpu(), S[h], f"state of head {h}")


@pytest.mark.parametrize("d,vd,dtype", [(1, 70, torch.float32), (128, 64, torch.float32), (32, 64, torch.bfloat16), (128, 128, torch.bfloat16)])
def test_all_parts_of_an_operand(d, vd, dtype):
    """Outputs of one term each, so that nothing averages an operand's error away: k q v with a decay of 0, and S q of the carried
    state alone.  fp32 operands, or SiLU of bf16.  Three roundings of 2^-24 and products left out below 2^-24 of each of the
    two products; SiLU adds 2 ulp an operand.  An operand without its third part is off by 2^-17."""
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(d + vd)
    n, H, act = 130, 2, dtype == torch.bfloat16
    m, _ = _meta([n], [6], dev)
    q, k, v = torch.zeros(n, H, d), torch.zeros(n, H, d), 1 + torch.rand(n, H, vd, generator=g)
    q[..., 0], k[..., 0] = 1 + torch.rand(n, H, generator=g), 1 + torch.rand(n, H, generator=g)
    k[:, 1] = 0
    state = torch.zeros(1, H, d, vd)
    state[:, 1, 0] = 1 + torch.rand(vd, generator=g)
    proj = torch.cat([t.reshape(n, -1) for t in (q, k, v)], 1).to(dtype)
    st = state.to(dev)
    got = recurrent.decay_attention(proj.to(dev), 0, H * d, 2 * H * d, torch.tensor([0.0, 1.0], device=dev), st, m, H, d, vd, act=act)
    got = got.double().cpu().view(n, H, vd)
    x = proj.double()
    x = torch.nn.functional.silu(x) if act else x
    q, k, v = x[:, :H * d].view(n, H, d)[..., 0], x[:, H * d:2 * H * d].view(n, H, d)[..., 0], x[:, 2 * H * d:].view(n, H, vd)
    want = torch.stack([(q * k)[:, 0, None] * v[:, 0], q[:, 1, None] * state[0, 1, 0].double()], 1)
    assert ((got - want).abs() / want).max() < (9 + (6 if act else 0)) * 2.0 ** -24


@pytest.mark.parametrize("e", [-108, -90, -60, -30, -8, 0, 9, 17])
@pytest.mark.parametrize("which", ["q", "k", "v", "state"])
def test_parts_at_all_exponents(which, e):
    """test_all_parts_of_an_operand with one operand of 2^e to 2^(e + 1), from the least that has all its parts (the third of 2^-108 is
    2^-124, of lesser numbers it goes below 2^-126 and is 0) to the largest that the products take (the state: 2^58)."""
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(e + 200)
    n, H, d, vd = 70, 2, 128, 64
    m, _ = _meta([n], [6], dev)
    e = 58 if which == "state" and e == 17 else e
    up = 15 if e < -60 else 0  # (the others, so that the result is a normal number)
    x = {c: (1 + torch.rand(n, H, w, generator=g)) * 2.0 ** (e if c == which else up) for c, w in (("q", 1), ("k", 1), ("v", vd))}
    q, k = torch.zeros(n, H, d), torch.zeros(n, H, d)
    q[..., :1], k[..., :1] = x["q"], x["k"]
    k[:, 1] = 0
    state = torch.zeros(1, H, d, vd)
    state[:, 1, 0] = (1 + torch.rand(vd, generator=g)) * 2.0 ** (e if which == "state" else up)
    st = state.to(dev)
    proj = torch.cat([t.reshape(n, -1) for t in (q, k, x["v"])], 1).to(dev)
    got = recurrent.decay_attention(proj, 0, H * d, 2 * H * d, torch.tensor([0.0, 1.0], device=dev), st, m, H, d, vd, act=False)
    got = got.double().cpu().view(n, H, vd)
    q, k, v = (x[c].double() for c in "qkv")
    want = torch.stack([q[:, 0] * k[:, 0] * v[:, 0], q[:, 1] * state[0, 1, 0].double()], 1)
    assert ((got - want).abs() / want).max() < 9 * 2.0 ** -24
