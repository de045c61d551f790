"""The 256x128 kernel for products of medium size (ts2_gemm_args.tileConfig bit 18) against fp64 products of the same 8-bit values, with the bounds of
the kernel for few tiles: contractions of one step to more than its pipeline holds, every result it writes, sums of two to four int8 products."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_gemm_slice_gpu import bound, operand, product, real  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402

TALL = 262144
SUM_I8 = "_Z18Ts2BackpropGroupI8iiiiiPK7ts2_matPKPKfS1_S3_S5_S1_iiPv"


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 9])
@pytest.mark.parametrize("t", [L.I8, L.E4M3])
@pytest.mark.parametrize("m,n", [(256, 128), (768, 384)])
def test_stored_and_accumulated(t, steps, m, n):
    print("case tall", t, steps, m, n, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(steps)
    k = 128 * steps
    a, b, want, mag = product(t, m, n, k, False, gen)
    lib = L.load()
    live = m - 37
    rs = torch.rand(m, device="cuda", generator=gen) + 0.5
    scale = 0.25 * rs.double()[:, None]
    want, tol = want * scale, bound(t, k, mag, want) * scale + 2.0 ** -22 * (want * scale).abs()
    for ct, dt in ((L.F32, torch.float32), (L.BF16, torch.int16)):
        c = torch.full((m, n), 7, dtype=dt, device="cuda")
        lib.gemm_nt(a, b, c, t, ct, row_scale=rs, alpha=0.25, m_live=live, tile_config=TALL)
        got = (c.view(torch.bfloat16) if ct == L.BF16 else c).double()
        assert bool(((got - want).abs() <= tol + (2.0 ** -8 * want.abs() if ct == L.BF16 else 0))[:live].all()) and not bool(got[live:].any())
    c0 = torch.randn((m, n), device="cuda", generator=gen)  # rows beyond the live ones keep what they held
    c = c0.clone()
    lib.gemm_nt(a, b, c, t, L.F32, row_scale=rs, alpha=0.25, m_live=live, epilogue=L.EPI_ADD, tile_config=TALL)
    w = want + c0.double()
    assert bool(((c.double() - w).abs() <= tol + 2.0 ** -23 * w.abs())[:live].all()) and torch.equal(c[live:], c0[live:])


@pytest.mark.parametrize("t", [L.I8, L.E4M3])
@pytest.mark.parametrize("normalize,rotate", [(True, True), (True, False), (False, True)])
def test_normalised_rows(t, normalize, rotate):
    print("case tall norm", t, normalize, rotate, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(4)
    m, n, k = 512, 384, 384
    a, b, want, mag = product(t, m, n, k, False, gen)
    rope = torch.randn((m, 128), device="cuda", generator=gen) if rotate else None
    c = torch.zeros((m, n), dtype=torch.int16, device="cuda"); ts = torch.zeros((n // 128, m), device="cuda")
    live = m - 5
    L.load().gemm_nt(a, b, c, t, L.BF16, alpha=0.5, epilogue=L.EPI_ROW_TILE_NORM, normalize=normalize, vec_scale=1 / 24, tile_scale=ts, rope=rope,
                     tile_config=TALL, m_live=live)
    v = (want * 0.5).view(m, n // 128, 128)
    e = 0.5 * bound(t, k, mag, want).amax()
    sc = v.pow(2).mean(-1).sqrt() / 24 if normalize else torch.ones_like(v[..., 0])
    if normalize:
        assert bool(((ts.t().double() - sc).abs() <= e / 24 + 1e-6 * sc)[:live].all()) and not bool(ts[:, live:].any())
    x = v / sc[..., None]
    p = rope.double().view(m, 1, 64, 2) if rotate else torch.tensor([1.0, 0.0], device="cuda").double().expand(m, 1, 64, 2)
    x = x.view(m, n // 128, 64, 2)
    w = torch.stack([x[..., 0] * p[..., 0] - x[..., 1] * p[..., 1], x[..., 1] * p[..., 0] + x[..., 0] * p[..., 1]], -1).reshape(m, n)
    far = (2 * (e / sc)[..., None, None] * (1 + x.abs().amax(-1, keepdim=True) / 24) * p.abs().amax(-1, keepdim=True)).expand(-1, -1, 64, 2).reshape(m, n)
    rad = (x.abs() * p.abs().amax(-1, keepdim=True)).sum(-1, keepdim=True).expand(-1, -1, -1, 2).reshape(m, n)
    got = c.view(torch.bfloat16).double()
    assert bool(((got - w).abs() <= 2.0 ** -8 * w.abs() + 1e-6 * rad + far)[:live].all()) and not bool(got[live:].any())


# 256 x 128 tiles from 65 on, one and three steps of K, and a count off the rounds of the chip; rows off its grid keep the 128x128 kernel
@pytest.mark.parametrize("count", [2, 3, 4])
@pytest.mark.parametrize("rows,cols,k", [(3328, 640, 128), (8448, 256, 384), (16640, 512, 256), (8320, 384, 384)])
def test_sums(count, rows, cols, k):
    print("case tall sum", count, rows, cols, k, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(count)
    g, w = [operand(L.I8, rows, k, gen) for _ in range(count)], [operand(L.I8, cols, k, gen) for _ in range(count)]
    rs = [torch.rand(rows, device="cuda", generator=gen) for _ in range(count)]
    f = [torch.rand(1, device="cuda", generator=gen) for _ in range(count)]
    live = rows - 3
    c = torch.full((rows, cols), 7.0, device="cuda")
    gm, wm, cm = (L.Mat * count)(*[L.mat(x) for x in g]), (L.Mat * count)(*[L.mat(x) for x in w]), L.mat(c)
    ptrs = lambda ts: (C.c_void_p * count)(*[x.data_ptr() for x in ts])  # noqa: E731
    lib = L.load()
    assert getattr(lib.dll, SUM_I8)(count, live, rows, cols, k, gm, ptrs(rs), wm, (C.c_float * count)(*[0.5] * count), ptrs(f), C.byref(cm), L.F32, 0, lib.stream()) == 0
    want, size = 0, 0
    for i in range(count):
        part = (real(L.I8, g[i]) @ real(L.I8, w[i]).t()) * (0.5 * f[i].double() * rs[i].double()[:, None])
        want, size = want + part, size + part.abs()
    # exact int32 sums; a conversion, a product of two factors and an addition each
    assert bool(((c.double() - want).abs() <= 5 * 2.0 ** -24 * count * size)[:live].all()) and not bool(c[live:].any())


# operands whose sums are exact: what is left is a fused multiply-add per element, the same in every kernel
@pytest.mark.parametrize("t", [L.I8, L.E4M3])
@pytest.mark.parametrize("row_scale", [True, False])
def test_accumulates_with_one_rounding(t, row_scale):
    print("case tall one rounding", t, row_scale, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(8)
    m, n, k = 512, 384, 640
    a, b = operand(t, m, k, gen), operand(t, n, k, gen)
    rs = torch.rand(m, device="cuda", generator=gen) + 0.5 if row_scale else None
    factor = torch.full((1,), 0.37, device="cuda")
    c0 = torch.randn((m, n), device="cuda", generator=gen) * 100
    got, few = c0.clone(), c0.clone()
    for c, config in ((got, TALL), (few, 65536)):
        L.load().gemm_nt(a, b, c, t, L.F32, row_scale=rs, alpha=0.3, alpha_ptr=factor, epilogue=L.EPI_ADD, tile_config=config, m_live=m - 9)
    assert torch.equal(got, few)


# int8 sums are exact, so that the rows have the bits of a stored product that the stand-alone pass normalises; of a rotation's two products either may
# be fused with their sum: an fp32 unit of the larger, a bf16 unit of the result at most
@pytest.mark.parametrize("normalize,rotate", [(True, True), (True, False), (False, True)])
def test_normalised_rows_are_the_passes(normalize, rotate):
    print("case tall norm bits", normalize, rotate, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    m, n, k, live = 768, 640, 512, 700
    a, b = operand(L.I8, m, k, gen), operand(L.I8, n, k, gen)
    rope = torch.randn((m, 128), device="cuda", generator=gen) if rotate else None
    lib = L.load()
    raw = torch.zeros((m, n), device="cuda")
    lib.gemm_nt(a, b, raw, L.I8, L.F32, alpha=0.3, m_live=live)
    got, want = [torch.zeros((m, n), dtype=torch.int16, device="cuda") for _ in range(2)]
    gs, ws = [torch.zeros((n // 128, m), device="cuda") for _ in range(2)]
    lib.gemm_nt(a, b, got, L.I8, L.BF16, alpha=0.3, epilogue=L.EPI_ROW_TILE_NORM, normalize=normalize, vec_scale=1 / 24, tile_scale=gs, rope=rope, tile_config=TALL,
                m_live=live)
    L.call("ts2_row_tile_normalize_rope", live, m, raw, L.F32, 1.0, int(normalize), 1 / 24, rope, want, ws if normalize else None)
    torch.cuda.synchronize()
    assert torch.equal(gs, ws)
    if not rotate:
        assert torch.equal(got, want)
        return
    x, y = got.view(torch.bfloat16).double(), want.view(torch.bfloat16).double()
    pair = y.view(m, -1, 2).norm(dim=-1, keepdim=True).expand(-1, -1, 2).reshape(m, n)
    assert bool(((x - y).abs() <= 2.0 ** -7 * y.abs() + 2.0 ** -22 * pair).all()) and float((got != want).double().mean()) < 1e-3
