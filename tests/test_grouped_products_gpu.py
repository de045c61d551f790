"""The products and quantisers that the step driver launches for several matrices at once, called through the library's own symbols
(csrc/internal.h: C++ linkage, no part of the C ABI): int8 k-tile quantiser without a transpose, deltas from operands as they lie, sums of int8
products with row scales of their own, several separately stored products, one delta per expert.  Operands are column blocks of wider
arrays, and rows beyond the batch hold what must not be read.

Bounds: int32 sums are exact.  Per term of a sum (a k-tile, a product) the kernels convert to fp32, scale and add: 4 roundings of 2^-24 on
no more than the sum of the terms' magnitudes.  e4m3 and bf16 products: test_gemm_slice_gpu.py.  A packed value is off by half a step."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402

EPS = 2.0 ** -24
# symbol and kinds of arguments: i int, l int64, f float, m ts2_mat of a 2-D tensor, p device pointer (1-D tensor or none), a host array
DELTA_ROWS = "_Z12Ts2DeltaRowsiiiiiPK7ts2_matS1_PKfiifS3_PflS1_S1_Pv", "iiiiimmpiifpplmm"
QUANT_TILE_ROWS = "_Z16Ts2QuantTileRowsiiiiPK7ts2_matS1_PKPKfPKjS3_PfPv", "iiiiaaaapp"
SUM_I8 = "_Z18Ts2BackpropGroupI8iiiiiPK7ts2_matPKPKfS1_S3_S5_S1_iiPv", "iiiiiaaaaamii"
EXPERT_DELTAS = "_Z19Ts2GroupedDeltaRowsiiiiPKiPK7ts2_matS3_fPKfS3_lS3_lPv", "iiiipmmfpmlml"
FORWARD_GROUP = "_Z15Ts2ForwardGroupiiiiiiPK7ts2_matPKS1_fPKPKfifiS1_S1_S3_Pv", "iiiiiimafaifimaa"


def run(function, *args):
    """a call whose arguments are of the kinds its symbol takes: a tensor of another rank would be passed as a pointer to something else"""
    name, kinds = function
    assert len(kinds) == len(args)
    for kind, a in zip(kinds, args):
        dims = a.dim() if isinstance(a, torch.Tensor) else None
        assert {"i": isinstance(a, int), "l": isinstance(a, C.c_int64), "f": isinstance(a, float), "m": dims == 2, "p": a is None or dims == 1,
                "a": isinstance(a, C.Array)}[kind], (name, kinds, kind, type(a), dims)
    L.call(name, *args)


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def block(rows, cols, dtype, left=128, right=256):
    """a column block of a wider array of ones"""
    return torch.ones((rows, left + cols + right), dtype=dtype, device="cuda")[:, left:left + cols]


def int8(rows, cols, gen):
    b = block(rows, cols, torch.int8)
    b.copy_(torch.randint(-127, 128, (rows, cols), device="cuda", generator=gen, dtype=torch.int8))
    return b


def mats(tensors):
    return (L.Mat * len(tensors))(*[L.mat(t) for t in tensors])


def pointers(tensors):
    return (C.c_void_p * len(tensors))(*[None if t is None else t.data_ptr() for t in tensors])


def mat_pointers(ms):
    return (C.POINTER(L.Mat) * len(ms))(*[C.pointer(m) if m is not None else None for m in ms])


@pytest.mark.parametrize("n,rows,k_tile", [(1, 128, 128), (500, 512, 512), (700, 1536, 512), (1024, 1024, 256)])
@pytest.mark.parametrize("width", [128, 384, 1032])
@pytest.mark.parametrize("dither", [False, True])
def test_k_tile_quantiser_without_the_transpose(n, rows, k_tile, width, dither):
    """the very bytes and scales of the transposing quantiser, per source"""
    print("case k-tile quantiser", n, rows, k_tile, width, dither, flush=True)
    gen = generator(n + width)
    count = 3
    src = []
    for i in range(count):
        s = block(rows, width, torch.bfloat16)
        s.copy_(torch.randn((rows, width), device="cuda", generator=gen) * 10.0 ** (i - 1))
        if k_tile < rows:
            s[:k_tile] = 0  # a tile of zeros
        src.append(s)
    raw = [s.view(torch.int16) for s in src]
    seeds = [(17 + i if dither else 0) for i in range(count)]
    top = [torch.zeros(rows, device="cuda") for _ in range(count)]
    for t, s in zip(top, src):
        t[:n] = s[:n].float().abs().amax(1)
    dst = [block(rows, width, torch.int8) for _ in range(count)]
    scale = torch.zeros((count, rows // k_tile), device="cuda")
    run(QUANT_TILE_ROWS, count, n, rows, k_tile, mats(raw), mats(dst), pointers(top), (C.c_uint32 * count)(*seeds), None, scale.view(-1))
    for i in range(count):
        tile_max, tile_scale = torch.zeros(rows // k_tile, device="cuda"), torch.zeros(rows // k_tile, device="cuda")
        out = torch.zeros((-(-width // 128) * 128, rows), dtype=torch.int8, device="cuda")
        L.call("ts2_tile_absmax", n, raw[i], L.BF16, None, k_tile, tile_max, 1)
        if width % 128 == 0:
            L.call("ts2_transpose_quant_dither", n, rows, raw[i], L.BF16, None, tile_max, k_tile, None, out, L.I8, tile_scale, C.c_uint32(seeds[i]))
            assert torch.equal(dst[i], out.t()[:, :width]) and torch.equal(scale[i], tile_scale)
        else:  # (a width the transposing quantiser does not take: by its contract)
            ts = torch.where(tile_max > 0, tile_max / torch.full_like(tile_max, 127), torch.ones_like(tile_max))
            assert torch.equal(scale[i], ts) and not bool(dst[i][n:].any())
            far = (dst[i][:n].float() * ts.repeat_interleave(k_tile)[:n, None] - src[i][:n].float()).abs()
            assert bool((far <= (1.0 if dither else 0.5001) * ts.repeat_interleave(k_tile)[:n, None]).all())


def packed_ok(delta, tile_scale, want, err):
    step = tile_scale.t().repeat_interleave(128, 1).double()
    return bool(((delta.double() * step - want).abs() <= err + step * 0.5001).all()) and bool(delta.any())


@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("src,width,count", [(128, 128, 1), (384, 128, 2), (256, 384, 2)])
def test_int8_delta_from_rows(tiles, src, width, count):
    """`count` gradients side by side, each with k-tile scales of its own; more than four k-tiles go as stored slices that are packed"""
    print("case int8 delta", tiles, src, width, count, flush=True)
    gen = generator(tiles + src)
    k_tile = 256
    rows, grad = tiles * k_tile, count * width
    x, g = int8(rows, src, gen), int8(rows, grad, gen)
    scale = torch.rand((count, tiles), device="cuda", generator=gen) + 0.1
    factor = torch.full((1,), 0.25, device="cuda")
    partial = torch.zeros(3 * grad * src, device="cuda")
    delta, ts = block(grad, src, torch.int8), torch.zeros((src // 128, grad), device="cuda")
    run(DELTA_ROWS, L.I8, rows - 3, rows, src, grad, x, g, scale.view(-1), k_tile, width, 0.5, factor, partial, C.c_int64(partial.numel()), delta, ts)
    want, mag = 0, 0
    for t in range(tiles):
        part = slice(t * k_tile, (t + 1) * k_tile)
        p = (g[part].double().t() @ x[part].double()) * scale[:, t].double().repeat_interleave(width)[:, None] * 0.125
        want, mag = want + p, mag + p.abs()
    assert packed_ok(delta, ts, want, (tiles + 4) * 4 * EPS * mag)


@pytest.mark.parametrize("mode", [L.E4M3, L.BF16])
@pytest.mark.parametrize("n,rows", [(1, 128), (127, 128), (129, 256), (300, 512), (1500, 1536)])
def test_delta_from_rows_stops_at_the_last_live_one(mode, n, rows):
    """rows beyond the batch hold NaN: widths off the 256 grid go to the kernel for few tiles, which does not read them"""
    print("case live rows", mode, n, rows, flush=True)
    gen = generator(n)
    src, grad = 256, 384
    data = []
    for w in (src, grad):
        v = torch.randn((rows, w), device="cuda", generator=gen)
        v[n:] = float("nan")
        t = v.bfloat16().view(torch.int16) if mode == L.BF16 else (v * 16).to(torch.float8_e4m3fn).view(torch.uint8)
        b = block(rows, w, t.dtype)
        b.copy_(t)
        data.append(b)
    x, g = data
    partial = torch.zeros(8 * grad * src, device="cuda")
    delta, ts = block(grad, src, torch.int8), torch.zeros((src // 128, grad), device="cuda")
    run(DELTA_ROWS, mode, n, rows, src, grad, x, g, None, 0, 0, 0.5, None, partial, C.c_int64(partial.numel()), delta, ts)
    real = [t[:n].contiguous().view(torch.bfloat16 if mode == L.BF16 else torch.float8_e4m3fn).double() * 1.0 for t in (x, g)]
    want, mag = 0.5 * real[1].t() @ real[0], 0.5 * real[1].abs().t() @ real[0].abs()
    assert packed_ok(delta, ts, want, 2e-4 * want.abs().max() if mode == L.E4M3 else (n + 8) * EPS * mag)


@pytest.mark.parametrize("rows,src", [(256, 128), (1024, 384), (4096, 1280), (4096, 1408), (2176, 2560)])
@pytest.mark.parametrize("count", [1, 2, 3, 4])
@pytest.mark.parametrize("c_type,add", [(L.F32, 0), (L.F32, 1), (L.BF16, 0), (L.BF16, 1)])
def test_sum_of_int8_products(rows, src, count, c_type, add):
    """fp32, stored: beyond 64 tiles of 256x128 that tile; else up to 640 workgroups of the kernel for few tiles, beyond it (2176 rows, off the tile's grid) the
    128x128 tile's sum.  bf16 or added: the kernel for few tiles, beyond it one product after the other"""
    print("case int8 sum", rows, src, count, c_type, add, flush=True)
    gen = generator(rows + src + count)
    grad, n = 384, rows - 29
    g8, w8 = [int8(rows, grad, gen) for _ in range(count)], [int8(src, grad, gen) for _ in range(count)]
    rs = [torch.rand(rows, device="cuda", generator=gen) + 0.5 for _ in range(count)]
    factor = [None if i == 1 else torch.full((1,), 0.5 + i, device="cuda") for i in range(count)]
    alpha = [0.01 * (i + 1) for i in range(count)]
    c0 = torch.randn((rows, src), device="cuda", generator=gen) * 10
    c0 = c0 if c_type == L.F32 else c0.bfloat16()
    c = c0.clone()
    run(SUM_I8, count, n, rows, src, grad, mats(g8), pointers(rs), mats(w8), (C.c_float * count)(*alpha), pointers(factor),
        c if c_type == L.F32 else c.view(torch.int16), c_type, add)
    want = c0.double() if add else torch.zeros_like(c0, dtype=torch.float64)
    mag = want.abs()
    bf16 = torch.zeros_like(mag)
    for i in range(count):
        f = torch.tensor(alpha[i], dtype=torch.float32).double().item() * (1.0 if factor[i] is None else 0.5 + i)
        p = (g8[i].double() @ w8[i].double().t()) * (rs[i].double()[:, None] * f)
        want, mag = want + p, mag + p.abs()
        bf16 = bf16 + 2.0 ** -8 * want.abs()  # (one product after the other rounds after each)
    err = (count + 2) * 4 * EPS * mag + (bf16 if c_type == L.BF16 else 0)
    assert bool(((c.double() - want).abs() <= err)[:n].all())
    assert torch.equal(c[n:], c0[n:]) if add else not bool(c[n:].any())


@pytest.mark.parametrize("mode", [L.E4M3, L.I8])
@pytest.mark.parametrize("rows,n,dst", [(128, 1, 128), (512, 500, 256), (1024, 900, 640)])
def test_separately_stored_products_equal_single_calls(mode, rows, n, dst):
    """the four products of an attention layer in one launch: the bits of four calls"""
    print("case separate products", mode, rows, n, dst, flush=True)
    gen = generator(rows + dst)
    src, vec = 384, 1 / 24
    x, *w = [(torch.randn((r, src), device="cuda", generator=gen) * 16) for r in (rows, dst, dst, dst, dst)]
    x, *w = [t.to(torch.float8_e4m3fn).view(torch.uint8) if mode == L.E4M3 else t.to(torch.int8) for t in (x, *w)]
    rope = torch.randn((rows, 128), device="cuda", generator=gen)
    factor = [torch.full((1,), 0.5 + i, device="cuda") if i < 3 else None for i in range(4)]
    new = lambda: ([torch.full((rows, dst), 7, dtype=torch.int16, device="cuda") for _ in range(4)],  # noqa: E731
                   [torch.full((dst // 128, rows), 7.0, device="cuda") for _ in range(4)])
    (got, gs), (want, ws) = new(), new()
    normalize, rotate = 1 | 4, 1 | 2
    wm, sm = [L.mat(t) for t in w], [L.mat(t) for t in gs]
    run(FORWARD_GROUP, mode, 4, n, rows, src, dst, x, mat_pointers(wm), 0.01, pointers(factor), normalize, vec, rotate, rope, mats(got),
        mat_pointers([m if (normalize >> i) & 1 else None for i, m in enumerate(sm)]))
    raw = torch.empty((rows, dst), device="cuda")
    for i in range(4):
        L.call("ts2_matmul_forward_norm_rope", mode, n, rows, src, dst, x, w[i], 0.01, factor[i], (normalize >> i) & 1, vec,
               rope if (rotate >> i) & 1 else None, want[i], ws[i] if (normalize >> i) & 1 else None, raw)
        assert torch.equal(got[i], want[i]) and torch.equal(gs[i], ws[i])


@pytest.mark.parametrize("offsets", [[0, 128], [0, 0, 384, 512], [0, 128, 128, 896, 1024]])
def test_one_delta_per_expert(offsets):
    """contraction-major operands cut into expert groups, empty ones among them, on the kernel for few tiles"""
    print("case expert deltas", offsets, flush=True)
    gen = generator(len(offsets))
    rows, m, n, groups = offsets[-1], 384, 128, len(offsets) - 1
    a, b = block(rows, m, torch.uint8), block(rows, n, torch.uint8)
    for t in (a, b):
        t.copy_((torch.randn(tuple(t.shape), device="cuda", generator=gen) * 16).to(torch.float8_e4m3fn).view(torch.uint8))
    c, ts = torch.full((groups * m, n), 7, dtype=torch.int8, device="cuda"), torch.full((groups, n // 128, m), 7.0, device="cuda")
    off = torch.tensor(offsets, dtype=torch.int32, device="cuda")
    run(EXPERT_DELTAS, rows, n, m, groups, off, b, a, 0.5, None, c, C.c_int64(m * n), ts.view(groups * (n // 128), m), C.c_int64(m * (n // 128) * 4))
    for i in range(groups):
        part = slice(offsets[i], offsets[i + 1])
        d, s = c[i * m:(i + 1) * m], ts[i]
        if offsets[i] == offsets[i + 1]:
            assert not bool(d.any()) and not bool(s.any())
            continue
        ra, rb = [t[part].contiguous().view(torch.float8_e4m3fn).double() for t in (a, b)]
        want = 0.5 * ra.t() @ rb
        assert packed_ok(d, s, want, 2e-4 * want.abs().max())
