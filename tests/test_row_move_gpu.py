"""int8: the codes that the layer-norm backward leaves with a row, moved to the next power of two of the gradients (Ts2ScaleGradRows): for rows of any
magnitude - denormal in fp32 or in bf16, a scale whose reciprocal overflows, zero, so large that a power of two more is infinite - codes, scale and
maximum are the row quantiser's bits for the gradients at the new power, with and without dither."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_row_quant_forms_gpu import LAYER_NORM, Slot, call, empty, p  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402

MOVE = "_Z16Ts2ScaleGradRowsPKfS0_PK7ts2_matS3_iPfS4_RK11RowQuantOutPv"


# the largest gradient of the pass, in powers of two: the multiplier becomes 2^(7 - that), or stays (7)
@pytest.mark.parametrize("power", [-90, -20, 7, 40])
@pytest.mark.parametrize("final,seed,n,rows,dim", [(True, 0, 331, 384, 512), (False, 77, 1100, 1152, 1024), (True, 5, 250, 256, 1536), (False, 0, 5, 128, 128)])
def test_codes_follow_the_multiplier(final, seed, n, rows, dim, power):
    print("case moved rows", final, seed, n, rows, dim, power, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    norm = torch.randint(-127, 128, (rows, dim), device="cuda", generator=gen).to(torch.int8)
    scale = torch.full((dim // 128, rows), 1 / 128, device="cuda")
    # row magnitudes 2^-152 .. 2^power, and rows of zeros
    e = torch.randint(-152, power - 3, (rows, 1), device="cuda", generator=gen)
    x = torch.randn((rows, dim), device="cuda", generator=gen).clamp(-6, 6).double()
    grad = (x * torch.exp2(e.double())).float()
    grad[1::7] = 0
    dn = grad if final else torch.zeros_like(grad)  # (what is added to a state gradient is zero, which leaves that one's rows)
    st, fast = (empty(rows, dim, torch.float32) if final else grad.clone()), empty(rows, dim)
    fast[:] = 0
    top, slot = torch.zeros(1, device="cuda"), Slot(rows, dim, seed)
    one = torch.ones(1, device="cuda")
    a = [L.mat(t) for t in (norm, scale, dn, st, fast)]
    call(LAYER_NORM, C.c_bool(final), n, rows, C.byref(a[0]), C.byref(a[1]), C.byref(a[2]), None if final else p(one), None if final else p(one),
         C.byref(a[3]), C.byref(a[4]), p(top), C.byref(slot.c))
    mult, inv = torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda")
    peak = torch.full((1,), 2.0 ** power, device="cuda")
    call(MOVE, p(peak), p(one), C.byref(a[3]), C.byref(a[4]), n, p(inv), p(mult), C.byref(slot.c))
    torch.cuda.synchronize()
    assert float(mult) == 2.0 ** (7 - power) and float(top) < 2.0 ** power
    assert torch.equal(fast[:n].view(torch.bfloat16), (st[:n] * mult).bfloat16()) and not bool(fast[n:].any())
    if power == 7:  # (nothing moved; a row that bf16 rounds to zero keeps the scale 1 that says so)
        slot.scale[(slot.top == 0) & (slot.scale == 1)] = 0
    assert slot.equals_quantiser_of(fast, n)


# every width of registers, a workgroup per four rows and walked rows
@pytest.mark.parametrize("final", [False, True])
@pytest.mark.parametrize("n,rows,dim", [(999, 1024, 384), (1000, 1024, 896), (333, 384, 1536), (8211, 8320, 512), (1999, 2048, 1024), (1500, 1536, 1408)])
def test_layer_norm_backward_has_the_bits_of_the_pass(final, n, rows, dim):
    print("case layer norm backward bits", final, n, rows, dim, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(dim)
    norm = torch.randint(-127, 128, (rows, dim), device="cuda", generator=gen).to(torch.int8)
    scale = torch.rand((dim // 128, rows), device="cuda", generator=gen) * 0.01
    dn, state = [torch.randn((rows, dim), device="cuda", generator=gen) for _ in range(2)]
    gs, gm = torch.full((1,), 0.25, device="cuda"), torch.full((1,), 4.0, device="cuda")
    out = []
    for rows_form in (True, False):
        st, fast, top = state.clone(), empty(rows, dim), torch.zeros(1, device="cuda")
        if rows_form:
            slot, a = Slot(rows, dim, 0), [L.mat(t) for t in (norm, scale, dn, st, fast)]
            call(LAYER_NORM, C.c_bool(final), n, rows, C.byref(a[0]), C.byref(a[1]), C.byref(a[2]), None if final else p(gs), None if final else p(gm),
                 C.byref(a[3]), C.byref(a[4]), p(top), C.byref(slot.c))
        elif final:
            L.call("ts2_backprop_final_normalize", n, rows, norm, L.I8, scale, dn, st, fast, L.BF16, top)
        else:
            L.call("ts2_backprop_layer_normalize", norm, L.I8, scale, dn, None, gs, gm, st, fast, L.BF16, top, n)
        torch.cuda.synchronize()
        out.append((st, fast, top))
    for a, b in zip(*out):
        assert torch.equal(a, b)
