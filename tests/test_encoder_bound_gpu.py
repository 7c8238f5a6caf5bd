"""The encoder's layers with their kernels chosen once (models/encoder.py _layers_bound) against the ops one by one, bit for
bit: from one short sequence to several rounds of tiles, a weight that is laid out differently, inside a captured graph."""
import pytest
import torch

from githubrepostorag_amd.models.configs import encoder_config
from githubrepostorag_amd.models.encoder import BertEncoder

pytestmark = pytest.mark.gpu


def _batch(dev, lens, H):
    g = torch.Generator(device=dev).manual_seed(sum(lens))
    h = torch.randn(sum(lens), H, generator=g, device=dev).bfloat16()
    start = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=dev)
    return h, start, torch.tensor(lens, dtype=torch.int32, device=dev), max(lens)


@pytest.fixture(scope="module")
def enc():
    e = BertEncoder(encoder_config("bge-base-en-v1.5"), seed=3)
    e.layers = e.layers[:3]
    return e


@pytest.mark.parametrize("lens", [[5], [33], [20, 60, 7], [190] * 6, [300] * 9, [400] * 22, [500] * 50], ids=lambda v: str(sum(v)))
def test_same_as_one_by_one(dev, enc, lens):
    args = _batch(dev, lens, 768)
    with torch.inference_mode():
        assert torch.equal(enc._layers_bound(*args), enc._layers(*args))


def test_weights_laid_out_differently(dev, enc):
    args = _batch(dev, [100, 30], 768)
    with torch.inference_mode():
        want = enc._layers(*args)
        L = enc.layers[1]
        kept = L.o_w, L.f1_w
        try:
            L.o_w = torch.cat([L.o_w, L.o_w], 1)[:, :768]            # rows of a wider tensor
            flat = torch.empty(L.f1_w.numel() + 1, dtype=torch.bfloat16, device=dev)
            L.f1_w = flat[1:].view_as(L.f1_w).copy_(L.f1_w)          # an address that is no multiple of 16
            got = enc._layers_bound(*args)
            torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -6, atol=2 ** -6)
        finally:
            L.o_w, L.f1_w = kept


def test_captured(dev, enc):
    args = _batch(dev, [64, 64], 768)
    with torch.inference_mode():
        want = enc._layers_bound(*args)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = enc._layers_bound(*args)
        for _ in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
