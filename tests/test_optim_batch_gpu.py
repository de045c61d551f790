"""Updates of matrices of unequal height in one batch (Ts2OptApplyBatch): whether the conversion forms the matrix scales or a launch of its own does
(by the sum of the squared heights), a matrix gets the bits that it gets alone - the widest matrix decides how a row's sums are added, so the widths
of a batch here are of one such form - and these are the update's formulas: scale = rms of the weights, fast
weights = the weights in units of a 32nd of it, rows beyond the matrix cleared."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_optim_gpu import OptMatrix, mat  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402

BATCH = "_Z16Ts2OptApplyBatchiPKPK14ts2_opt_matrixPKPK7ts2_matS8_PK23ts2_add_gradient_paramsPv"
DECAY = 0.95


class Job:
    def __init__(self, rows, cols, fast_type, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        z = lambda *s: torch.zeros(s, device="cuda")  # noqa: E731
        padded = (rows + 127) // 128 * 128
        self.t = t = {"weights": torch.randn((rows, cols), device="cuda", generator=g) * 0.05, "avgGrad": z(rows, cols), "gradRowSum2": z(rows),
                      "weightsRowSum2": z(rows), "rowScale": z(rows), "rowDisp": z(rows), "sumWeight": torch.full((1,), 2.0, device="cuda"),
                      "sparsity": torch.full((1,), 0.5, device="cuda"), "fast": torch.full((padded, cols), 55, dtype=torch.int8, device="cuda"),
                      "matrixScale": z(1), "convertMult": z(1)}
        self.delta = torch.randint(-127, 128, (rows, cols), device="cuda", generator=g).to(torch.int8)
        self.scale = torch.rand((cols // 128, rows), device="cuda", generator=g) * 1e-3
        self.c = OptMatrix(xSize=cols, ySize=rows, yBufSize=padded, rowDispSize=rows, fastType=fast_type)
        for k in ("weights", "avgGrad", "fast"):
            setattr(self.c, k, mat(t[k]))
        for k in ("gradRowSum2", "weightsRowSum2", "rowScale", "rowDisp", "sumWeight", "sparsity", "matrixScale", "convertMult"):
            setattr(self.c, k, t[k].data_ptr())
        self.mats = (mat(self.delta), mat(self.scale))


def apply(jobs):
    lib = L.load()
    params = torch.tensor([DECAY, 0.9, 0.3, 0.7, 0.1, 0.01], device="cuda")
    ptrs = lambda xs: (C.c_void_p * len(jobs))(*[C.addressof(x) for x in xs])  # noqa: E731
    rc = getattr(lib.dll, BATCH)(len(jobs), ptrs([j.c for j in jobs]), ptrs([j.mats[0] for j in jobs]), ptrs([j.mats[1] for j in jobs]),
                                 C.c_void_p(params.data_ptr()), lib.stream())
    assert rc == 0
    torch.cuda.synchronize()


# scales formed by the conversion; by a launch of their own (a tall matrix first, last); alone on either side of both lines; more than one launch takes
@pytest.mark.parametrize("shapes", [
    [(1, 128), (130, 512), (64, 256), (1000, 384)], [(4097, 256), (1, 512), (257, 384)], [(300, 384), (4096, 256)], [(8192, 2048), (8193, 2048), (127, 1536)],
    [(64, 4096), (200, 2176)], [(128 + 3 * i, 128) for i in range(17)], [(5793, 256), (1, 512), (257, 384)], [(8193, 256), (64, 128)]])
def test_matrices_of_unequal_height(shapes):
    print("case optimiser batch", shapes, flush=True)
    make = lambda: [Job(r, c, (L.I8, L.E4M3)[i & 1], i) for i, (r, c) in enumerate(shapes)]  # noqa: E731
    together, alone = make(), make()
    for _ in range(2):  # (the second step starts from the weights and estimates of the first)
        apply(together)
        for j in alone:
            apply([j])
    for a, b in zip(together, alone):
        for k in a.t:
            assert torch.equal(a.t[k].view(torch.uint8), b.t[k].view(torch.uint8)), k
        w = a.t["weights"].double()
        want = float(w.pow(2).mean().sqrt())
        assert abs(float(a.t["matrixScale"]) - want) <= 2e-6 * want
        assert abs(float(a.t["sumWeight"]) - ((2.0 * DECAY + 1) * DECAY + 1)) <= 1e-6
        rows = w.shape[0]
        x = a.t["weights"] * a.t["convertMult"]
        assert abs(float(a.t["convertMult"]) * want / 32 - 1) <= 3e-6 and not bool(a.t["fast"][rows:].any())
        if a.c.fastType == L.I8:
            assert torch.equal(a.t["fast"][:rows], x.round().clamp(-128, 127).to(torch.int8))
        else:
            assert torch.equal(a.t["fast"][:rows].view(torch.uint8), x.clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))
