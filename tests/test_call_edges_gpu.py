"""Edges of the operators' calls: empty batches, k-tile scales together with slices, rotation tables off the 8-byte grid, what the step
driver's accessors show, and the exact forms of the normalising store."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402


def e4m3(x):
    return x.to(torch.float8_e4m3fn).view(torch.uint8)


def randn(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen)


def test_packed_delta_of_an_empty_batch_is_zero():
    """no live rows: zeros, whatever lies in the rows beyond (e4m3, pad rows that nobody vouches for)"""
    print("case delta of an empty batch", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(1)
    rows, src, grad = 256, 256, 384
    b = L.MatMulBuffers(L.E4M3, rows, src, grad)
    x, dy = e4m3(randn(gen, rows, src) * 8), e4m3(randn(gen, rows, grad) * 8)
    for n in (0, 1):
        b.delta.fill_(77)
        b.delta_tile_scale.fill_(-1)
        b.backprop_delta(n, x, None, dy, L.E4M3)
        torch.cuda.synchronize()
        assert bool(b.delta.any()) == (n > 0) and bool(b.delta_tile_scale.any()) == (n > 0)
