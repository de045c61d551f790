"""int8: the gradient passes that leave the rows they write quantised (the driver's entry points, called by their own symbols) against the separate
passes and the row quantiser: codes, scales and maxima are the quantiser's bits for the gradients written, rows beyond the live ones are cleared.
The gradients' tile sums are the same tree, in which the compiler may fuse other products: a unit of fp32, which bf16 gradients do not show at
these seeds.  In fp32, sums of 128 products differ by 8 * 2^-24 of the sum of their magnitudes, x = (g - src * dp / sum2) * scale by a few
times that of the row's largest value: 2^-19 of it."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402

LOLU = "_Z19Ts2BackpropLoluRowsiiiPK7ts2_matS1_fS1_S1_S1_S1_S1_RK11RowQuantOutS4_Pv"
NORM_ROPE = "_Z23Ts2BackpropNormRopeRowsiiiPKPK7ts2_matfS3_S3_S3_S3_PK11RowQuantOutPv"
LAYER_NORM = "_Z29Ts2BackpropLayerNormalizeRowsbiiPK7ts2_matS1_S1_PKfS3_S1_S1_PfRK11RowQuantOutPv"
SCALE_GRAD = "_Z16Ts2ScaleGradRowsPKfS0_PK7ts2_matS3_iPfS4_S4_S4_Pv"


class RowQuantOut(C.Structure):
    _fields_ = [("dst", C.c_void_p), ("dstStride", C.c_int64), ("rowScale", C.c_void_p), ("rowAbsMax", C.c_void_p), ("seed", C.c_uint32)]


class Slot:
    def __init__(self, rows, dim, seed):
        self.codes = torch.full((rows, dim), 7, dtype=torch.int8, device="cuda")
        self.scale, self.top = torch.full((rows,), -1.0, device="cuda"), torch.full((rows,), -1.0, device="cuda")
        self.c = RowQuantOut(self.codes.data_ptr(), dim, self.scale.data_ptr(), self.top.data_ptr(), seed)

    def equals_quantiser_of(self, grad, n):
        rows, dim = self.codes.shape
        want = Slot(rows, dim, 0)
        L.call("ts2_normalize_vecs_row_max_dither", n, rows, grad, L.BF16, None, want.codes, want.scale, want.top, C.c_uint32(self.c.seed))
        torch.cuda.synchronize()
        return all(torch.equal(a, b) for a, b in ((self.codes, want.codes), (self.scale, want.scale), (self.top, want.top)))


def bf16(gen, rows, dim, spread=1.0):
    x = torch.randn((rows, dim), device="cuda", generator=gen) * torch.exp(torch.randn((rows, 1), device="cuda", generator=gen) * spread)
    return x.bfloat16().view(torch.int16)


def empty(rows, dim, dt=torch.int16):
    return torch.full((rows, dim), 3, dtype=dt, device="cuda")


def p(t):
    return C.c_void_p(t.data_ptr())


def call(symbol, *args):
    lib = L.load()
    assert getattr(lib.dll, symbol)(*args, lib.stream()) == 0


# chunks of 512 columns: one not full, one, the edges of two and three, the widest; one live row, rows off the four of a workgroup
WIDTHS = [(1, 128, 128), (130, 256, 512), (77, 128, 640), (500, 512, 1536), (9, 128, 2176), (131, 256, 4096)]


@pytest.mark.parametrize("seed", [0, 12345])
@pytest.mark.parametrize("n,rows,dim", WIDTHS)
def test_gate_backward(n, rows, dim, seed):
    print("case gate backward rows", n, rows, dim, seed, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(dim)
    gate, vals, grad = bf16(gen, rows, dim, 0.1), bf16(gen, rows, dim, 0.1), bf16(gen, rows, dim)
    scale = torch.rand((dim // 128, rows), device="cuda", generator=gen) + 0.1
    if n > 5:
        vals[3] = 0  # tiles of zeros
        grad[4] = 0
    m = L.mat
    for mode in (0, 1):
        g, v, g0, v0 = [empty(rows, dim) for _ in range(4)]
        ds, ds0 = torch.full_like(scale, 5), torch.full_like(scale, 6)
        qg, qv = Slot(rows, dim, seed), Slot(rows, dim, seed and seed + 2)
        args = [m(gate), m(vals), m(scale), m(grad), m(g), m(v), m(ds)]
        call(LOLU, mode, n, rows, C.byref(args[0]), C.byref(args[1]), C.c_float(1 / 24 if mode == 0 else 1.0), C.byref(args[2]), C.byref(args[3]),
             C.byref(args[4]), C.byref(args[5]), C.byref(args[6]), C.byref(qg.c), C.byref(qv.c))
        if mode == 0:
            L.call("ts2_backprop_row_tile_normalize_lolu", n, rows, gate, vals, 1 / 24, scale, grad, L.BF16, g0, v0, L.BF16)
        else:
            L.call("ts2_backprop_lolu_dscale", n, rows, gate, vals, 1.0, grad, L.BF16, g0, L.BF16, v0, L.BF16, ds0)
            assert torch.equal(ds, ds0)
        assert torch.equal(g, g0) and torch.equal(v, v0) and qg.equals_quantiser_of(g0, n) and (mode == 1 or qv.equals_quantiser_of(v0, n))


@pytest.mark.parametrize("n,rows,dim", WIDTHS)
def test_norm_and_rotation_backward(n, rows, dim):
    print("case norm rope rows", n, rows, dim, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(dim)
    grad, norm, scale, dst, dst0, slots = [], [], [], [], [], []
    rope = torch.randn((rows, 128), device="cuda", generator=gen)
    for i in range(3):
        grad.append(bf16(gen, rows, dim)); norm.append(bf16(gen, rows, dim, 0.1)); scale.append(torch.rand((dim // 128, rows), device="cuda", generator=gen))
        dst.append(empty(rows, dim)); dst0.append(empty(rows, dim)); slots.append(Slot(rows, dim, 0))
    has_norm, has_rope = (True, False, True), (True, True, False)

    def mats(ts, use=(True,) * 3):
        keep = [L.mat(t) for t in ts]
        return (C.c_void_p * 3)(*[C.addressof(k) if u else None for k, u in zip(keep, use)]), keep
    a = [mats(grad), mats(norm, has_norm), mats(scale, has_norm), mats([rope] * 3, has_rope), mats(dst)]
    q = (RowQuantOut * 3)(*[s.c for s in slots])
    call(NORM_ROPE, 3, n, rows, a[0][0], C.c_float(1.0), a[1][0], a[2][0], a[3][0], a[4][0], q)
    for i in range(3):
        L.call("ts2_backprop_row_tile_normalize_rope", n, rows, grad[i], L.BF16, 1.0, norm[i] if has_norm[i] else None, scale[i] if has_norm[i] else None,
               rope if has_rope[i] else None, dst0[i], L.BF16)
        assert torch.equal(dst[i], dst0[i]) and slots[i].equals_quantiser_of(dst0[i], n)


# up to 1536 columns; workgroups of 256 threads up to 1024 rows, of 1024 beyond, which walk several rows each from 8192 on
@pytest.mark.parametrize("n,rows,dim", [(1, 128, 128), (200, 256, 512), (1000, 1024, 640), (1025, 1152, 1024), (1700, 1792, 1536), (9000, 9088, 128)])
def test_layer_norm_backward_and_the_scale_that_follows(n, rows, dim):
    print("case layer norm backward rows", n, rows, dim, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(dim)
    norm = torch.randint(-127, 128, (rows, dim), device="cuda", generator=gen).to(torch.int8)
    scale = torch.rand((dim // 128, rows), device="cuda", generator=gen) * 0.01
    dn = torch.randn((rows, dim), device="cuda", generator=gen)
    state = torch.randn((rows, dim), device="cuda", generator=gen)
    if n > 5:
        norm[2], dn[5] = 0, 0
    gs, gm = torch.full((1,), 0.25, device="cuda"), torch.full((1,), 4.0, device="cuda")
    for final in (False, True):
        out = []
        for rows_form in (True, False):
            st, fast, top = state.clone(), empty(rows, dim), torch.zeros(1, device="cuda")
            if rows_form:
                slot = Slot(rows, dim, 0)
                a = [L.mat(t) for t in (norm, scale, dn, st, fast)]
                call(LAYER_NORM, C.c_bool(final), n, rows, C.byref(a[0]), C.byref(a[1]), C.byref(a[2]), None if final else p(gs), None if final else p(gm),
                     C.byref(a[3]), C.byref(a[4]), p(top), C.byref(slot.c))
            elif final:
                L.call("ts2_backprop_final_normalize", n, rows, norm, L.I8, scale, dn, st, fast, L.BF16, top)
            else:
                L.call("ts2_backprop_layer_normalize", norm, L.I8, scale, dn, None, gs, gm, st, fast, L.BF16, top, n)
            out.append((st, fast, top))
        (st, fast, top), (st0, fast0, top0) = out
        assert ((st - st0).abs() <= 2.0 ** -19 * st0.abs().amax(1, keepdim=True)).all() and abs(float(top) - float(top0)) <= 2.0 ** -19 * float(top0)
        live = rows if final else n
        assert torch.equal(fast[:live].view(torch.bfloat16), (st[:live] * (1.0 if final else 4.0)).bfloat16()) and torch.equal(fast[live:], fast0[live:])
        assert torch.equal(st[n:], st0[n:]) and slot.equals_quantiser_of(fast, n)
        # the power of two changes (or not): values, scales and maxima move together, the codes stay
        for before in (1.0, 2.0 ** 20):
            prev = torch.full((1,), before, device="cuda")
            mult, inv = torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda")
            st, fast, top = out[0]
            f2, s2 = (st * before).bfloat16().view(torch.int16).clone(), Slot(rows, dim, 0)
            L.call("ts2_normalize_vecs_row_max_dither", n, rows, f2, L.BF16, None, s2.codes, s2.scale, s2.top, C.c_uint32(0))
            a = [L.mat(st), L.mat(f2)]
            call(SCALE_GRAD, p(top), p(prev), C.byref(a[0]), C.byref(a[1]), n, p(inv), p(mult), p(s2.scale), p(s2.top))
            torch.cuda.synchronize()
            assert s2.equals_quantiser_of(f2, n) and float(mult) * float(inv) == 1.0
            assert torch.equal(f2[:n].view(torch.bfloat16), (st[:n] * float(mult)).bfloat16())
