"""The grouped GEMM's chains with the experts' row counts that make their tiles 192 and 128 rows (csrc/kernels/moe.hip moe_chain):
last tiles of one row, one past a wave's first quadrant and half, and all but one; and, at widths where both products are chains, with
counts for each of 256, 192 and 128 rows, the number of rows that the kernel finds (grag_moe_chain_rows) asked for."""
import ctypes

import pytest
import test_moe_chain_gpu as chain

from githubrepostorag_amd.ops._lib import lib
from githubrepostorag_amd.ops.gemm import _num_cus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit,W,width", [("glu", 320, 2120), ("relu2", 448, 4104), ("clamped", 576, 2048)])
@pytest.mark.parametrize("counts", [[192] * 11 + [1, 49, 97, 145, 191], [192, 384] * 8, [128] * 12 + [1, 33, 65, 127], [128, 97] * 8])
def test_chain_rows(dev, counts, unit, W, width, monkeypatch):
    monkeypatch.setattr(chain, "COUNTS", counts)
    chain.test_chain(dev, unit, W, width)


@pytest.mark.parametrize("unit", ["glu", "relu2", "clamped"])
@pytest.mark.parametrize("rows,counts", [(256, [256] * 11 + [1, 65, 129, 193, 255]), (192, [192] * 11 + [1, 49, 97, 145, 191]),
                                         (128, [128] * 12 + [1, 33, 65, 127])])
def test_each_number_of_rows(dev, rows, counts, unit, monkeypatch):
    """Both products of every unit, a ragged last column tile in each."""
    W = width = 2624
    E, n = len(counts), -(-sum(counts) // 2) * 2
    took = [lib().grag_moe_chain_rows((ctypes.c_int * E)(*counts), E, n, N, K, kind, _num_cus())
            for N, K, kind in ((width, W, 3 if unit == "relu2" else 1), (W, width, 0))]
    assert 0 not in took and (_num_cus() != 256 or took == [rows, rows])
    monkeypatch.setattr(chain, "COUNTS", counts)
    chain.test_chain(dev, unit, W, width)
