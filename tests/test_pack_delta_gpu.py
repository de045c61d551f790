"""Sum of the slices of a delta and its packing: the slices are added in their order whatever number of rows and slices a launch requests
together, so bytes and scales are the bits of the same operations done here one slice after the other."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# both sides of 32 MB of slices (one row and eight slices at a time up to there), of two slices and eight; rows off the groups of two and four
@pytest.mark.parametrize("rows,cols,splits", [(1, 128, 1), (129, 128, 2), (131, 256, 3), (257, 384, 5), (5, 128, 8), (130, 256, 9), (67, 512, 32), (4096, 512, 4),
                                              (4097, 512, 4), (2049, 512, 8), (1027, 256, 33), (3, 1024, 2)])
def test_slices_are_added_in_order(rows, cols, splits):
    print("case pack delta", rows, cols, splits, flush=True)
    check(rows, cols, splits)


def test_many_slices_beyond_the_memory_side_cache():
    print("case pack delta, 257 MB", flush=True)
    check(4115, 1024, 16)


def check(rows, cols, splits):
    from tscale2_amd import lib as L
    L.load()
    r = np.random.default_rng(rows + splits)
    part = (r.standard_normal((splits, rows, cols)) * np.exp(r.standard_normal((splits, rows, 1)))).astype(np.float32)
    part[:, rows // 2] = 0  # a row of zeros: scale zero
    total = np.zeros((rows, cols), np.float32)
    for s in range(splits):
        total = total + part[s]
    alpha, mult = np.float32(0.03), np.float32(1.7)
    scale = np.float32(alpha * mult)
    d = torch.full((rows, cols), 3, dtype=torch.int8, device="cuda")
    ts = torch.full((cols // 128, rows), -1.0, device="cuda")
    L.call("ts2_pack_delta", torch.from_numpy(part.reshape(splits * rows, cols)).cuda(), splits, C.c_int64(rows * cols * 4), rows, cols, float(alpha),
           torch.tensor([float(mult)], device="cuda"), d, ts)
    torch.cuda.synchronize()
    tiles = total.reshape(rows, cols // 128, 128)
    discr = (np.abs(tiles).max(2) * scale / np.float32(127)).astype(np.float32)
    assert np.array_equal(ts.cpu().numpy().T, discr)
    with np.errstate(divide="ignore"):
        inv = np.where(discr > 0, np.float32(1) / discr, np.float32(0)).astype(np.float32)
    want = np.clip(np.rint(tiles * scale * inv[:, :, None]), -128, 127).astype(np.int8).reshape(rows, cols)
    assert np.array_equal(d.cpu().numpy(), want)
