"""Which decode attention kernel a step takes (ops/attention.py)."""
import pytest

from githubrepostorag_amd.ops import attention as A
from githubrepostorag_amd.ops._lib import lib


@pytest.mark.skipif(not A._DEC_AUTO or A._DEC_NT != "auto", reason="rules switched off by the environment")
def test_ring_by_rows_and_waves(monkeypatch):
    assert (A.DECODE_NS3_ROWS, A.DECODE_NS3_WAVES) == (512, 1280)
    # 28 / 4 heads: 192 sequences in 2 parts, 128 in 2, 83 in 4
    assert [A.decode_variant(2, 2048, 1536), A.decode_variant(2, 1024, 1024), A.decode_variant(4, 512, 1328)] == [12, 11, 11]
    for rows, code in ((0, 11), (769, 11), (768, 12)):  # GRAG_DECODE_NS3_ROWS: 0 switches the 3-stage ring off
        monkeypatch.setattr(A, "DECODE_NS3_ROWS", rows)
        assert A.decode_variant(2, 2048, 1536) == code
    monkeypatch.setattr(A, "DECODE_NS3_WAVES", 0)
    assert A.decode_variant(2, 2048, 1536) == 11


def test_rules_by_the_device(monkeypatch):
    """A quarter of the CUs: a quarter of the parts that a launch's rules count."""
    from types import SimpleNamespace

    from githubrepostorag_amd.ops import gemm as G

    monkeypatch.setattr(G.WS, "scratch_ok", lambda name: True)
    meta = lambda n: SimpleNamespace(num_seqs=n, num_splits=2, cascade=None)  # noqa: E731
    for ncu, most in ((256, 25), (64, 6)):
        monkeypatch.setattr(G, "_NCU", [ncu])
        assert A.decode_mw_takes(meta(most), 4) and not A.decode_mw_takes(meta(most + 1), 4)


# D, parts, us of 1 / 2 / 4 waves
@pytest.mark.parametrize("D,parts,us", [(128, 1024, (36.5, 40.1, 45.4)), (128, 640, (20.5, 23.6, 24.9)), (128, 384, (20.0, 16.9, 19.3)),
                                        (128, 332, (7.0, 5.8, 8.8)), (128, 32, (13.8, 11.5, 10.8)), (64, 1024, (34.6, 33.7, 36.5)),
                                        (64, 768, (15.0, 13.3, 13.4)), (64, 1024, (17.8, 17.5, 20.0))])
def test_waves_of_a_hybrid_decode_part(D, parts, us):
    assert us[(1, 2, 4).index(lib().grag_sink_decode_waves(D, parts))] <= 1.02 * min(us)


def test_waves_of_any_parts():
    assert [lib().grag_sink_decode_waves(D, n) for D in (64, 128) for n in (1, 1 << 20)] == [4, 1, 4, 1]


def test_every_number_of_waves_is_tested():
    """The parts of tests/test_sink_decode_gpu.py test_many_parts (4 kv heads), for heads of 128 and 64."""
    took = [[lib().grag_sink_decode_waves(D, 4 * n * k) for n, k in ((64, 4), (129, 1), (129, 3))] for D in (128, 64)]
    assert took == [[1, 2, 1], [2, 4, 1]]
