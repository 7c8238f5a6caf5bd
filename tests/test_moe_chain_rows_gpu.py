"""The grouped GEMM's chains with the experts' row counts that make their tiles 192 and 128 rows (csrc/kernels/moe.hip moe_chain):
last tiles of one row, one past a wave's first quadrant and half, and all but one."""
import pytest
import test_moe_chain_gpu as chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit,W,width", [("glu", 320, 2120), ("relu2", 448, 4104), ("clamped", 576, 2048)])
@pytest.mark.parametrize("counts", [[192] * 11 + [1, 49, 97, 145, 191], [192, 384] * 8, [128] * 12 + [1, 33, 65, 127], [128, 97] * 8])
def test_chain_rows(dev, counts, unit, W, width, monkeypatch):
    monkeypatch.setattr(chain, "COUNTS", counts)
    chain.test_chain(dev, unit, W, width)
