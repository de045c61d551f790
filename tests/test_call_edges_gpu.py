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


@pytest.mark.parametrize("k,splits", [(2048, 4), (2048, 2), (3072, 2), (4608, 3)])
def test_stored_slices_with_k_tile_scales_hold_their_own_part_of_the_contraction(k, splits):
    """int8 with one scale per 512 contraction elements, the contraction cut into stored slices: slab i is the sum over slice i (whole
    k-tiles, ceil(tiles / splits) of them).  int32 sums are exact; per k-tile one fp32 product and one fp32 addition are left."""
    print("case k-tile scales and slices", k, splits, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(k + splits)
    m, n, kt = 256, 256, 512
    a, b = [torch.randint(-127, 128, (d, k), device="cuda", generator=gen, dtype=torch.int8) for d in (m, n)]
    scale = torch.rand(k // kt, device="cuda", generator=gen) + 0.5
    c = torch.full((splits * m, n), 9.0, device="cuda")
    L.load().gemm_nt(a, b, c, L.I8, L.F32, k_tile_scale=scale, k_tile=kt, split_k=splits, split_slab_bytes=m * n * 4, m=m, n=n)
    per = -(-(k // kt) // splits) * kt
    for i in range(splits):
        want, mag = torch.zeros((m, n), device="cuda", dtype=torch.float64), 0
        for t in range(i * per, min((i + 1) * per, k), kt):
            p = (a[:, t:t + kt].double() @ b[:, t:t + kt].double().t()) * scale[t // kt].double()
            want, mag = want + p, mag + p.abs()
        assert bool(((c[i * m:(i + 1) * m].double() - want).abs() <= (per // kt + 2) * 2.0 ** -24 * mag).all()), i


@pytest.mark.parametrize("mode", [L.E4M3, L.I8])
def test_normalised_forward_of_an_empty_batch_is_zero(mode):
    print("case normalised forward of an empty batch", mode, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(2)
    rows, src, dst = 256, 256, 384
    x, w = [e4m3(randn(gen, r, src) * 8) if mode == L.E4M3 else (randn(gen, r, src) * 30).to(torch.int8) for r in (rows, dst)]
    res = torch.full((rows, dst), 7, dtype=torch.int16, device="cuda")
    scale, raw = torch.full((dst // 128, rows), 7.0, device="cuda"), torch.empty((rows, dst), device="cuda")
    L.call("ts2_matmul_forward_norm_rope", mode, 0, rows, src, dst, x, w, 0.01, None, 1, 1 / 24, None, res, scale, raw)
    torch.cuda.synchronize()
    assert not bool(res.any()) and not bool(scale.any())


def two_launches(mode, n, rows, src, dst, x, w, normalize, vec, rope, res, scale, raw):
    L.call("ts2_matmul_forward", mode, n, rows, src, dst, x, w, 1.0, None, raw, L.F32, 0)
    L.call("ts2_row_tile_normalize_rope", n, rows, raw, L.F32, 1.0, normalize, vec, rope, res, scale)


@pytest.mark.parametrize("rows,dst", [(256, 256), (4096, 1664)])
@pytest.mark.parametrize("offset,pitch", [(1, 128), (0, 129)])
def test_rotation_tables_off_the_eight_byte_grid(rows, dst, offset, pitch):
    """a table at any fp32 address and stride is taken by the product and the stand-alone pass where the fused store cannot read it"""
    print("case rotation table alignment", rows, dst, offset, pitch, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    src, n = 128, rows - 5
    x, w = [torch.randint(-1, 2, (r, src), device="cuda", generator=gen).float() for r in (rows, dst)]
    x8, w8 = e4m3(x), e4m3(w)
    flat = randn(gen, rows * pitch + offset)
    rope = flat[offset:].view(rows, pitch)[:, :128]
    new = lambda: (torch.zeros((rows, dst), dtype=torch.int16, device="cuda"), torch.zeros((dst // 128, rows), device="cuda"))  # noqa: E731
    raw = torch.empty((rows, dst), device="cuda")
    (got, gs), (want, ws) = new(), new()
    two_launches(L.E4M3, n, rows, src, dst, x8, w8, 1, 1 / 24, rope, want, ws, raw)
    L.call("ts2_matmul_forward_norm_rope", L.E4M3, n, rows, src, dst, x8, w8, 1.0, None, 1, 1 / 24, rope, got, gs, raw)
    torch.cuda.synchronize()
    assert torch.equal(gs, ws) and torch.equal(got, want)


@pytest.mark.parametrize("mode", [L.E4M3, L.I8])
@pytest.mark.parametrize("rows,src,dst", [(256, 384, 256), (1024, 128, 1152), (2048, 2048, 1536), (4096, 256, 1664), (8192, 256, 1024), (16384, 1024, 1152)])
def test_normalised_store_rounds_like_the_stand_alone_pass(mode, rows, src, dst):
    """below the large tile's range: sums of squares of small whole numbers are exact in any order, so what is left is one division, one
    square root, one product and one reciprocal in fp32 - the fused store has to give the very bits of product + pass"""
    print("case normalised store", mode, rows, src, dst, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(rows + dst)
    n = rows - 3
    x, w = [torch.randint(-1, 2, (r, src), device="cuda", generator=gen) for r in (rows, dst)]
    x8, w8 = [e4m3(t.float()) if mode == L.E4M3 else t.to(torch.int8) for t in (x, w)]
    new = lambda: (torch.zeros((rows, dst), dtype=torch.int16, device="cuda"), torch.zeros((dst // 128, rows), device="cuda"))  # noqa: E731
    raw = torch.empty((rows, dst), device="cuda")
    for table in (None, randn(gen, rows, 128), randn(gen, rows, 130)[:, :128]):  # (rows on 16 bytes, rows on 8)
        (got, gs), (want, ws) = new(), new()
        two_launches(mode, n, rows, src, dst, x8, w8, 1, 1 / 24, table, want, ws, raw)
        L.call("ts2_matmul_forward_norm_rope", mode, n, rows, src, dst, x8, w8, 1.0, None, 1, 1 / 24, table, got, gs, raw)
        torch.cuda.synchronize()
        assert torch.equal(gs, ws)
        if table is None:
            assert torch.equal(got, want)
        else:  # (the rotation may contract its products differently: one step of bf16)
            a, b = got.view(torch.bfloat16).double(), want.view(torch.bfloat16).double()
            assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -20 * b.abs().max()).all())
