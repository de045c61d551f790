"""Calls that the operators refuse before anything is launched.  The arrays are host memory: nothing here may reach a kernel, so the file
does not run where a GPU is present."""
import builtins
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402

pytestmark = pytest.mark.skipif(torch.cuda.device_count() > 0, reason="refusals only: no launch may see these host arrays")
SHAPE, UNSUPPORTED, NULL = -1, -3, -4


def u8(rows, cols):
    return torch.zeros((rows, cols), dtype=torch.uint8)


def buffers(rows, src, grad, t_cols=None):
    b = L.BwdBuffers()
    keep = {"gradT": u8(grad, t_cols or rows), "srcT": u8(src, t_cols or rows), "transformT": u8(src, grad)}
    for k, v in keep.items():
        setattr(b, k, L.mat(v))
    return b, keep


def delta(n, rows, src, grad, buf):
    x, dy, d, s = u8(512, src), u8(512, grad), torch.zeros((grad, src), dtype=torch.int8), torch.zeros((src // 128, grad))
    m = [L.mat(t) for t in (x, dy, d, s)]
    return L.load().dll.ts2_matmul_backprop_delta(L.E4M3, n, rows, src, grad, C.byref(m[0]), None, C.byref(m[1]), L.E4M3, C.c_float(1), None, 512,
                                                  C.byref(buf), C.byref(m[2]), C.byref(m[3]), None)


@pytest.mark.parametrize("n,rows,grad", [(180, 192, 384), (300, 256, 384), (64, 64, 384), (256, 256, 192)])
def test_packed_delta_refuses_sizes_off_the_tile_grid_and_more_rows_than_there_are(n, rows, grad):
    b, _keep = buffers(rows, 256, grad, 512)
    assert delta(n, rows, 256, grad, b) == SHAPE


def test_the_kernel_for_few_tiles_refuses_a_contraction_that_ends_inside_its_unit():
    """bit 11 admits contractions of 64 bytes, bit 16 asks for the kernel whose unit is 128"""
    g = L.GemmArgs(a=L.mat(u8(128, 192)), b=L.mat(u8(128, 192)), c=L.mat(torch.zeros((128, 128))), abType=L.E4M3, cType=L.F32, m=128, n=128, k=192, alpha=1,
                   splitK=1, tileConfig=65536 | 2048)
    assert L.load().dll.ts2_gemm_nt(C.byref(g), None) == UNSUPPORTED


@pytest.mark.parametrize("m,n,config", [(384, 256, 0), (256, 384, 0), (384, 384, 0), (384, 384, 2)])
def test_several_products_off_the_256_grid_only_where_the_call_asks_for_the_kernel(m, n, config):
    """two further products: the 256x256 kernel's call; other sizes run with bit 16 of tileConfig and are refused without it"""
    a, b, c = u8(m, 128), u8(n, 128), torch.zeros((m, n))
    g = L.GemmArgs(a=L.mat(a), b=L.mat(b), c=L.mat(c), abType=L.E4M3, cType=L.F32, m=m, n=n, k=128, alpha=1, splitK=1, tileConfig=config,
                   extraSegments=2)
    for i in range(2):
        g.segment[i].a, g.segment[i].b, g.segment[i].alpha = a.data_ptr(), b.data_ptr(), 1
    assert L.load().dll.ts2_gemm_nt(C.byref(g), None) == UNSUPPORTED


@pytest.mark.parametrize("rows,src", [(384, 384), (512, 512)])
@pytest.mark.parametrize("wrong", ["rows of a gradient", "columns of a gradient", "rows of a transposed matrix", "columns of a transposed matrix"])
def test_grouped_input_gradient_checks_every_product(rows, src, wrong):
    """the second product's operands count as much as the first's, at sizes that run as one launch"""
    grad = 256
    bufs, keep = zip(*[buffers(rows, src, grad) for _ in range(2)])
    grads = [L.mat(u8(rows, grad)) for _ in range(2)]
    if wrong == "rows of a gradient":
        grads[1].y = rows - 128
    elif wrong == "columns of a gradient":
        grads[1].x = grad - 128
    elif wrong == "rows of a transposed matrix":
        bufs[1].transformT.y = src - 128
    else:
        bufs[1].transformT.x = grad - 128
    out = torch.zeros((rows, src))
    c = L.mat(out)
    gp, bp = (C.POINTER(L.Mat) * 2)(*[C.pointer(g) for g in grads]), (C.POINTER(L.BwdBuffers) * 2)(*[C.pointer(b) for b in bufs])
    alpha = (C.c_float * 2)(1, 1)
    assert L.load().dll.ts2_matmul_backprop_group(L.E4M3, rows, rows, src, grad, 2, gp, bp, alpha, None, C.byref(c), L.F32, 0, None) == SHAPE


@pytest.mark.parametrize("columns", [0, 128])
def test_packed_delta_wants_its_transposing_scratch_whichever_kernel_runs(columns):
    """e4m3 pad rows that nobody vouches for: the caller provides gradT (and srcT), also where the product reads the operands as they lie"""
    b, keep = buffers(256, 256, 384)
    b.gradT = L.mat(keep["gradT"][:, :columns]) if columns else L.Mat(None, 0, 0, 0)
    assert delta(200, 256, 256, 384, b) == SHAPE


@pytest.mark.parametrize("mode", [L.E4M3, L.I8])
@pytest.mark.parametrize("rows,columns,code", [(0, 0, NULL), (128, 384, SHAPE), (256, 256, SHAPE)])
def test_normalised_forward_wants_its_scratch_below_the_large_tile(mode, rows, columns, code):
    """the fp32 scratch of product + pass belongs to the call, also where a fused store makes no use of it"""
    x, w, res, scale = u8(256, 128), u8(384, 128), torch.zeros((256, 384), dtype=torch.int16), torch.zeros((3, 256))
    raw = torch.zeros((rows, columns)) if rows else None
    m = [L.mat(t) for t in (x, w, res, scale, raw)]
    assert L.load().dll.ts2_matmul_forward_norm_rope(mode, 200, 256, 128, 384, C.byref(m[0]), C.byref(m[1]), C.c_float(1), None, 1, C.c_float(1), None,
                                                     C.byref(m[2]), C.byref(m[3]), C.byref(m[4]) if rows else None, None) == code


def test_a_thread_that_finds_the_library_loaded_can_convert_its_arguments(monkeypatch):
    """load() publishes the library last: a thread that meets another's load half done either loads for itself or has all that a call needs"""
    seen = []

    lib = L.load()
    importer = builtins.__import__

    def spy(name, *args, **kw):
        if name == "torch":
            seen.append(L._lib is not None)
            if seen[-1]:
                L._conv(u8(2, 2))
        return importer(name, *args, **kw)
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(L, "_tensor", None)
    monkeypatch.setattr(L, "Lib", lambda: lib)
    monkeypatch.setattr(builtins, "__import__", spy)
    assert L.load() is lib and seen == [False]
    L._conv(u8(2, 2))
