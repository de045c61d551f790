"""The 64x64 kernel for products of at most a tile per CU (ts2_gemm_args.tileConfig bit 19) against fp64 products of the same 8-bit values, with the bounds
of the kernel for few tiles, and bit by bit against that kernel: contractions of half a step to more than its pipeline holds, row tiles without a
live row, sums of several e4m3 products with a factor of zero among them."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_gemm_slice_gpu import SLICE, bound, operand, product, real  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402

SQUARE = 524288


@pytest.mark.parametrize("half_steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 17])
@pytest.mark.parametrize("t", [L.I8, L.E4M3])
@pytest.mark.parametrize("m,n,dead", [(128, 128, 37), (384, 640, 37), (384, 256, 200)])
def test_stored_and_accumulated(t, half_steps, m, n, dead):
    print("case square", t, half_steps, m, n, dead, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(half_steps)
    k = 128 * half_steps
    a, b, want, mag = product(t, m, n, k, False, gen)
    lib = L.load()
    live = m - dead  # rows beyond it are written as zeros, or keep what they held
    rs = torch.rand(m, device="cuda", generator=gen) + 0.5
    factor = torch.full((1,), 0.5, device="cuda")
    scale = 0.125 * rs.double()[:, None]
    want, tol = want * scale, bound(t, k, mag, want) * scale + 2.0 ** -22 * (want * scale).abs()
    for ct, dt in ((L.F32, torch.float32), (L.BF16, torch.bfloat16)):
        for epi in (L.EPI_STORE, L.EPI_ADD):
            c0 = torch.randn((m, n), device="cuda", generator=gen).to(dt)
            got, few = c0.clone(), c0.clone()
            for c, config in ((got, SQUARE), (few, SLICE)):
                lib.gemm_nt(a, b, c.view(torch.int16) if ct == L.BF16 else c, t, ct, row_scale=rs, alpha=0.25, alpha_ptr=factor, m_live=live, epilogue=epi,
                            tile_config=config)
            assert torch.equal(got, few)
            w = want + (c0.double() if epi == L.EPI_ADD else 0)
            extra = (2.0 ** -8 if ct == L.BF16 else 2.0 ** -23) * w.abs()
            assert bool(((got.double() - w).abs() <= tol + extra)[:live].all())
            assert torch.equal(got[live:], c0[live:] if epi == L.EPI_ADD else torch.zeros_like(c0[live:]))


@pytest.mark.parametrize("half_steps", [1, 3, 4])
@pytest.mark.parametrize("factors", [(1.0, 0.25), (0.0, 2.0, 0.5), (1.0, 1.0, 0.0, 3.0), (0.0, 0.0)])
def test_sums(half_steps, factors):
    print("case square sums", half_steps, factors, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(len(factors))
    m, n, k = 256, 256, 128 * half_steps
    ops = [(operand(L.E4M3, m, k, gen), operand(L.E4M3, n, k, gen)) for _ in factors]
    ptr = [torch.full((1,), f, device="cuda") for f in factors]
    want = sum(0.5 * f * (real(L.E4M3, a) @ real(L.E4M3, b).t()) for f, (a, b) in zip(factors, ops))
    got, few = torch.full((m, n), 7.0, device="cuda"), torch.full((m, n), 7.0, device="cuda")
    for c, config in ((got, SQUARE), (few, SLICE)):
        L.load().gemm_nt(ops[0][0], ops[0][1], c, L.E4M3, L.F32, alpha=0.5, alpha_ptr=ptr[0], segments=[(a, b, 0.5, p) for (a, b), p in zip(ops[1:], ptr[1:])],
                         tile_config=config)
    assert torch.equal(got, few)
    assert bool(((got.double() - want).abs() <= len(factors) * 2e-4 * want.abs().max()).all())


# sizes that the 256x128 kernel takes by itself: asked for, it is this kernel (e4m3 sums in the order of the kernel for few tiles, which the other's is not)
@pytest.mark.parametrize("ct,epi", [(L.F32, L.EPI_STORE), (L.F32, L.EPI_ADD)])
def test_asked_for_beyond_its_range(ct, epi):
    print("case square asked for", ct, epi, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    m, n, k = 2048, 1152, 512
    # (magnitudes of 2^-9 to 2^8: sums that fp32 does not hold exactly)
    a, b = [(torch.randn((r, k), device="cuda", generator=gen) * torch.exp2(torch.randint(-7, 7, (r, k), device="cuda", generator=gen).float())).to(
        torch.float8_e4m3fn).view(torch.uint8) for r in (m, n)]
    c0 = torch.randn((m, n), device="cuda", generator=gen)
    got, few, tall, free = [c0.clone() for _ in range(4)]
    for c, config in ((got, SQUARE), (few, SLICE), (tall, 262144), (free, 0)):
        L.load().gemm_nt(a, b, c, L.E4M3, ct, alpha=0.25, epilogue=epi, tile_config=config)
    assert torch.equal(got, few) and torch.equal(free, tall) and not torch.equal(got, tall)
