"""Which decode attention kernel a step takes (ops/attention.py)."""
import pytest

from githubrepostorag_amd.ops import attention as A


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
