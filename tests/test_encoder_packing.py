"""BertEncoder.encode_ids packs ragged batches as the explicit tensors would: empty, over-long and tuple entries."""
import numpy as np
import pytest
import torch

from githubrepostorag_amd.models.configs import EncoderConfig
from githubrepostorag_amd.models.encoder import BertEncoder


@pytest.mark.parametrize("batch", [[[3]], [[1, 2, 3], [], [7] * 40, (4, 5)], [[5, 6.0, True]], [[np.int64(4), 2], (1, torch.tensor(8))]])
def test_packing(batch):
    cfg = EncoderConfig("t", vocab_size=50, hidden_size=32, num_layers=1, num_heads=2, intermediate_size=64, max_position=16)
    enc = BertEncoder(cfg, device="cpu", dtype=torch.float32)
    seen = {}
    fwd = enc.forward
    enc.forward = lambda *a: seen.update(a=a) or fwd(*a)
    out = enc.encode_ids(batch, want_bf16=False)
    ids, pos, start, length, most, _ = seen["a"]
    lens = [max(1, min(len(x), 16)) for x in batch]
    assert length.tolist() == lens and start.tolist() == [sum(lens[:i]) for i in range(len(lens) + 1)] and most == max(lens)
    assert ids.tolist() == [int(t) for x, n in zip(batch, lens) for t in (x[:n] if x else [0])]
    assert pos.tolist() == [i for n in lens for i in range(n)]
    assert all(t.dtype == torch.int32 for t in (ids, pos, start, length)) and out.shape[0] == len(batch)


def test_not_whole_numbers_refused():
    cfg = EncoderConfig("t", vocab_size=50, hidden_size=32, num_layers=1, num_heads=2, intermediate_size=64, max_position=16)
    enc = BertEncoder(cfg, device="cpu", dtype=torch.float32)
    for bad in ([["a"]], [[None]], [[1 << 40]], [["12"]], [["1", 2]], [("3", 4, 5)], [[b"12", 3]], [[np.float32(2.5)]]):
        with pytest.raises((TypeError, ValueError, RuntimeError, OverflowError)):
            enc.encode_ids(bad)
