"""The kernel for products with few output tiles (ts2_gemm_args.tileConfig bit 16) against fp64 products of the same 8-bit / bf16 values:
every operand type and layout (int8 with k-tile scales and int8 sums: test_grouped_products_gpu.py), contractions of one, an odd and an
even number of its half steps and more than its pipeline holds, every result type.  Bounds: i8 sums are exact (one rounding to fp32 is left); fp32 sums of bf16 products in any order stay within K * 2^-24 of
sum |a b|; the e4m3 instruction adds its 64 products with fewer bits than an fp32 sum has (1.5e-5 rms of the result on every kernel
here), and its products are held to 2e-4 of the largest result like in the tests of the other kernels; a bf16 result adds half a unit in
the last place (2^-9), a packed one half of its row's step (max / 254)."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402

SLICE = 65536
UNIT = {L.I8: 128, L.E4M3: 128, L.BF16: 64}  # contraction elements of half a step


def operand(t, rows, cols, gen):
    x = torch.randn((rows, cols), device="cuda", generator=gen)
    if t == L.BF16:
        return x.bfloat16().view(torch.int16)
    if t == L.I8:
        return torch.clamp(torch.round(x * 40), -127, 127).to(torch.int8)
    return (x * 16).to(torch.float8_e4m3fn).view(torch.uint8)


def real(t, x):
    return x.double() if t == L.I8 else x.view(torch.bfloat16 if t == L.BF16 else torch.float8_e4m3fn).double()


def product(t, m, n, k, k_major, gen):
    a, b = (operand(t, k, m, gen), operand(t, k, n, gen)) if k_major else (operand(t, m, k, gen), operand(t, n, k, gen))
    ra, rb = real(t, a), real(t, b)
    ra, rb = (ra.t(), rb.t()) if k_major else (ra, rb)
    return a, b, ra @ rb.t(), ra.abs() @ rb.abs().t()


def bound(t, k, mag, want):
    if t == L.E4M3:
        return torch.full_like(mag, 2e-4) * want.abs().max()
    return 2.0 ** -23 * mag if t == L.I8 else (k + 8) * 2.0 ** -24 * mag


@pytest.mark.parametrize("half_steps", [1, 2, 3, 7, 12])
@pytest.mark.parametrize("t", [L.I8, L.E4M3, L.BF16])
@pytest.mark.parametrize("m,n", [(128, 128), (384, 640)])
def test_stored_results(t, half_steps, m, n):
    print("case slice stored", t, half_steps, m, n, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(half_steps)
    k = half_steps * UNIT[t]
    a, b, want, mag = product(t, m, n, k, False, gen)
    lib = L.load()
    live = m - 37  # rows beyond it are written as zeros
    rs = torch.rand(m, device="cuda", generator=gen) + 0.5
    scale = 0.25 * rs.double()[:, None]
    want, tol = want * scale, bound(t, k, mag, want) * scale + 2.0 ** -22 * (want * scale).abs()
    for ct, dt in ((L.F32, torch.float32), (L.BF16, torch.int16), (L.F16, torch.float16)):
        c = torch.full((m, n), 7, dtype=dt, device="cuda")
        lib.gemm_nt(a, b, c, t, ct, row_scale=rs, alpha=0.25, m_live=live, tile_config=SLICE)
        got = (c.view(torch.bfloat16) if ct == L.BF16 else c).double()
        if ct == L.F16:
            w, extra = want.clamp(-65504, 65504), 2.0 ** -11 * want.abs() + 2.0 ** -24
            ok = (got[:live] - w[:live]).abs() <= (tol + extra)[:live]
            ok |= want[:live].abs() > 65000
        else:
            ok = (got[:live] - want[:live]).abs() <= (tol + (2.0 ** -8 * want.abs() if ct == L.BF16 else 0))[:live]
        assert bool(ok.all()) and not bool(got[live:].any())
    for ct in (L.F32, L.BF16):  # accumulating: rows beyond the live ones keep what they held
        c0 = torch.randn((m, n), device="cuda", generator=gen)
        c0 = c0 if ct == L.F32 else c0.bfloat16()
        c = c0.clone() if ct == L.F32 else c0.clone().view(torch.int16)
        lib.gemm_nt(a, b, c, t, ct, row_scale=rs, alpha=0.25, m_live=live, epilogue=L.EPI_ADD, tile_config=SLICE)
        got = (c.view(torch.bfloat16) if ct == L.BF16 else c).double()
        w = want + c0.double()
        extra = (2.0 ** -8 if ct == L.BF16 else 2.0 ** -23) * w.abs()
        assert bool(((got - w).abs() <= tol + extra)[:live].all()) and torch.equal(got[live:], c0.double()[live:])


@pytest.mark.parametrize("t", [L.E4M3, L.BF16])
@pytest.mark.parametrize("k", [128, 256, 384, 640, 1920])
def test_contraction_major_operands(t, k):
    print("case slice k-major", t, k, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(k)
    m, n = 512, 256
    a, b, want, mag = product(t, m, n, k, True, gen)
    lib = L.load()
    c = torch.zeros((m, n), device="cuda")
    lib.gemm_nt(a, b, c, t, L.F32, m=m, n=n, k=k, k_major=True, tile_config=SLICE)
    assert bool(((c.double() - want).abs() <= bound(t, k, mag, want)).all())
    splits = 3 if k >= 384 else 1
    if splits > 1:
        c = torch.zeros((m * splits, n), device="cuda")
        lib.gemm_nt(a, b, c, t, L.F32, m=m, n=n, k=k, k_major=True, split_k=splits, split_slab_bytes=m * n * 4, tile_config=SLICE)
        assert bool(((c.double().view(splits, m, n).sum(0) - want).abs() <= bound(t, k, mag, want)).all())


@pytest.mark.parametrize("t,k_major", [(L.I8, False), (L.E4M3, False), (L.E4M3, True), (L.BF16, True)])
def test_packed_delta(t, k_major):
    print("case slice packed", t, k_major, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    m, n, k = 256, 512, 5 * UNIT[t] * 2
    a, b, want, mag = product(t, m, n, k, k_major, gen)
    lib = L.load()
    c = torch.zeros((m, n), dtype=torch.int8, device="cuda"); ts = torch.zeros((n // 128, m), device="cuda")
    kw = dict(m=m, n=n, k=k, k_major=True) if k_major else {}
    lib.gemm_nt(a, b, c, t, L.I8, alpha=0.5, epilogue=L.EPI_ROW_TILE_MAXNORM, tile_scale=ts, tile_config=SLICE, **kw)
    step = ts.t().repeat_interleave(128, 1).double()
    assert bool(((c.double() * step - want * 0.5).abs() <= 0.5 * bound(t, k, mag, want) + step * 0.5001).all())
    top = (want * 0.5).abs().view(m, n // 128, 128).amax(-1)
    assert bool(((ts.t().double() * 127 - top).abs() <= 0.5 * bound(t, k, mag, want).amax() + 1e-6 * top).all())


@pytest.mark.parametrize("t", [L.E4M3, L.BF16])
def test_normalised_rows_and_several_products(t):
    print("case slice norm / segments", t, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(4)
    m, n, k = 256, 256, 3 * UNIT[t]
    lib = L.load()
    a, b, want, mag = product(t, m, n, k, False, gen)
    rope = torch.randn((m, 128), device="cuda", generator=gen)
    c = torch.zeros((m, n), dtype=torch.int16, device="cuda"); ts = torch.zeros((n // 128, m), device="cuda")
    lib.gemm_nt(a, b, c, t, L.BF16, alpha=0.5, epilogue=L.EPI_ROW_TILE_NORM, normalize=True, vec_scale=1 / 24, tile_scale=ts, rope=rope, tile_config=SLICE)
    v = (want * 0.5).view(m, n // 128, 128)
    sc = v.pow(2).mean(-1).sqrt() / 24
    e = 0.5 * bound(t, k, mag, want).amax()  # of a value; a row's rms moves by no more
    assert bool(((ts.t().double() - sc).abs() <= e / 24 + 1e-6 * sc).all())
    p, x = rope.double().view(m, 1, 64, 2), (v / sc[..., None]).view(m, n // 128, 64, 2)
    w = torch.stack([x[..., 0] * p[..., 0] - x[..., 1] * p[..., 1], x[..., 1] * p[..., 0] + x[..., 0] * p[..., 1]], -1).reshape(m, n)
    # value and scale are off by e and e / 24 at most, and a rotation mixes two of them
    far = (2 * (e / sc)[..., None, None] * (1 + x.abs().amax(-1, keepdim=True) / 24) * p.abs().amax(-1, keepdim=True)).expand(-1, -1, 64, 2).reshape(m, n)
    rad = (x.abs() * p.abs().amax(-1, keepdim=True)).sum(-1, keepdim=True).expand(-1, -1, -1, 2).reshape(m, n)
    assert bool(((c.view(torch.bfloat16).double() - w).abs() <= 2.0 ** -8 * w.abs() + 1e-6 * rad + far).all())
    # two further products, one of them with factor zero (left out), the others in units of their own
    zero, two = torch.zeros(1, device="cuda"), torch.full((1,), 2.0, device="cuda")
    a2, b2, want2, mag2 = product(t, m, n, k, False, gen)
    a3, b3, _, _ = product(t, m, n, k, False, gen)
    c = torch.zeros((m, n), device="cuda")
    lib.gemm_nt(a, b, c, t, L.F32, alpha=0.5, segments=[(a3, b3, 1.0, zero), (a2, b2, 0.125, two)], tile_config=SLICE)
    w = want * 0.5 + want2 * 0.25
    tol = bound(t, 2 * k, mag * 0.5 + mag2 * 0.25, w)
    assert bool(((c.double() - w).abs() <= tol + 2.0 ** -22 * w.abs()).all())


@pytest.mark.parametrize("k", [128, 512, 640, 1536, 1664, 2048])
@pytest.mark.parametrize("ct,dt", [(L.F32, torch.float32), (L.BF16, torch.bfloat16), (L.F16, torch.float16), (L.I32, torch.int32)])
def test_int8_stored_results_have_the_same_bits_from_every_kernel(k, ct, dt):
    """both sides of the contractions where the dispatcher changes kernels: int32 sums are exact, what is left is their conversion to fp32, one
    product with alpha * rowScale and one rounding; also rows that start on the 4-byte grid only, which the kernel for few tiles declines"""
    print("case int8 stored, every kernel", k, ct, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(k)
    m, n, live = 384, 256, 333
    a, b, want, _ = product(L.I8, m, n, k, False, gen)
    rs = torch.rand(m, device="cuda", generator=gen) + 0.5
    raw = ct == L.I32
    if raw:
        want = want.to(torch.int32)
    else:
        want = (want.float() * (rs * 2.0 ** -10)[:, None]).to(dt)  # (inside the range of a half)
        want[live:] = 0
    for config in (0, SLICE, 2 * SLICE):
        for pad in (0, 4 // torch.empty(0, dtype=dt).element_size()):
            if pad and config == SLICE:
                continue
            wide = torch.full((m, n + pad), 7, dtype=dt, device="cuda")
            c = wide[:, :n]
            out = c.view(torch.int16) if ct == L.BF16 else c
            if raw:
                L.load().gemm_nt(a, b, out, L.I8, ct, tile_config=config)
            else:
                L.load().gemm_nt(a, b, out, L.I8, ct, row_scale=rs, alpha=2.0 ** -10, m_live=live, tile_config=config)
            assert torch.equal(c, want) and bool((wide[:, n:] == 7).all()), (config, pad)
