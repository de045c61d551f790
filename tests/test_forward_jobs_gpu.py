"""Several separately stored products that share their input, at the sizes where one launch of the 128x128 (e4m3) or 256x128 (int8) kernel takes them:
the values of single calls.  Those may run on another kernel, whose fp32 sums have another order (e4m3: 2e-4 of the largest result, see
test_gemm_slice_gpu.py; int8 sums are exact): a scale is off by that part of it plus 2^-20, a stored value by that part of its row's scale times the
rotation's norm (sqrt 2 of the table's largest entry) and one unit in the last place of bf16."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_grouped_products_gpu import FORWARD_GROUP, generator, mat_pointers, mats, pointers, run  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402


# the first size past the kernel for few tiles, rows off 256 (int8 stays with that kernel), the last row tile dead; K below and above eight steps
@pytest.mark.parametrize("mode", [L.E4M3, L.I8])
@pytest.mark.parametrize("count,rows,n,dst", [(4, 2048, 1790, 512), (4, 1152, 1152, 768), (2, 4096, 4000, 512), (3, 2304, 2049, 512)])
@pytest.mark.parametrize("src", [128, 384, 1152])
def test_products_that_share_their_input(mode, count, rows, n, dst, src):
    print("case forward jobs", mode, count, rows, n, dst, src, flush=True)
    gen = generator(rows + src)
    vec = 1 / 24
    x, *w = [(torch.randn((r, src), device="cuda", generator=gen) * 16) for r in (rows, *[dst] * count)]
    x, *w = [t.to(torch.float8_e4m3fn).view(torch.uint8) if mode == L.E4M3 else t.to(torch.int8) for t in (x, *w)]
    rope = torch.randn((rows, 128), device="cuda", generator=gen)
    factor = [torch.full((1,), 0.5 + i, device="cuda") if i < 3 else None for i in range(count)]
    new = lambda: ([torch.full((rows, dst), 7, dtype=torch.int16, device="cuda") for _ in range(count)],  # noqa: E731
                   [torch.full((dst // 128, rows), 7.0, device="cuda") for _ in range(count)])
    (got, gs), (want, ws) = new(), new()
    normalize, rotate = 1 | 4, 1 | 2
    pad = lambda a: a + [a[0]] * (4 - count)  # noqa: E731
    wm, sm = [L.mat(t) for t in w], [L.mat(t) for t in gs]
    run(FORWARD_GROUP, mode, count, n, rows, src, dst, x, mat_pointers(pad(wm)), 0.01, pointers(pad(factor)), normalize & ((1 << count) - 1), vec,
        rotate, rope, mats(pad(got)), mat_pointers(pad([m if (normalize >> i) & 1 else None for i, m in enumerate(sm)])))
    raw = torch.empty((rows, dst), device="cuda")
    off = 4e-4 if mode == L.E4M3 else 0.0
    for i in range(count):
        norm, turn = (normalize >> i) & 1, (rotate >> i) & 1
        L.call("ts2_matmul_forward_norm_rope", mode, n, rows, src, dst, x, w[i], 0.01, factor[i], norm, vec, rope if turn else None, want[i],
               ws[i] if norm else None, raw)
        a, b = got[i].view(torch.bfloat16).double(), want[i].view(torch.bfloat16).double()
        largest = b.abs().amax()
        assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + (off + 2.0 ** -18) * 1.5 * largest).all()) and not bool(a[n:].any())
        if norm:
            assert bool(((gs[i] - ws[i]).abs() <= (off + 2.0 ** -20) * ws[i].abs().amax()).all())


# whole numbers, so that no order of a product's sum rounds: what single calls store (the kernel for few tiles), scales and rows bit by bit.  65 to 256
# workgroups of that kernel, K below and above eight steps
@pytest.mark.parametrize("count,rows,n,dst", [(4, 2048, 1790, 512), (4, 1152, 1152, 768), (2, 4096, 4000, 512), (3, 2304, 2049, 512)])
@pytest.mark.parametrize("src", [128, 1152])
def test_e4m3_squares_are_added_as_in_single_calls(count, rows, n, dst, src):
    print("case forward jobs' squares", count, rows, n, dst, src, flush=True)
    gen = generator(rows + src + 1)
    x, *w = [torch.randint(-4, 5, (r, src), device="cuda", generator=gen).float().to(torch.float8_e4m3fn).view(torch.uint8) for r in (rows, *[dst] * count)]
    new = lambda: ([torch.zeros((rows, dst), dtype=torch.int16, device="cuda") for _ in range(count)],  # noqa: E731
                   [torch.zeros((dst // 128, rows), device="cuda") for _ in range(count)])
    (got, gs), (want, ws) = new(), new()
    pad = lambda a: a + [a[0]] * (4 - count)  # noqa: E731
    wm, sm = [L.mat(t) for t in w], [L.mat(t) for t in gs]
    run(FORWARD_GROUP, L.E4M3, count, n, rows, src, dst, x, mat_pointers(pad(wm)), 0.01, pointers([None] * 4), (1 << count) - 1, 1 / 24, 0,
        torch.zeros((rows, 128), device="cuda"), mats(pad(got)), mat_pointers(pad(sm)))
    raw = torch.empty((rows, dst), device="cuda")
    for i in range(count):
        L.call("ts2_matmul_forward_norm_rope", L.E4M3, n, rows, src, dst, x, w[i], 0.01, None, 1, 1 / 24, None, want[i], ws[i], raw)
        assert want[i][:n].any() and torch.equal(got[i], want[i]) and torch.equal(gs[i], ws[i])
