"""The embedding's gradient where the delta has many labels (each row is stored, cleared or added to by a mark per label) and where it has few, against
64-bit sums: rows with no label, one, several, the same one twice, labels that are subtracted, labels that many rows share.  A label that one term
names holds that term exactly; n terms in fp32 in any order are off by at most n * 2^-24 of the sum of their magnitudes."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402

EMBED_BACKWARD = "_Z16Ts2EmbedBackwardiiPKiPKjPK7ts2_matS5_iPiPv"


@pytest.mark.parametrize("labels,dim", [(65536, 1024), (174763, 384), (300, 256)])  # (the labels of the first are marked from 30720 rows on)
@pytest.mark.parametrize("n", [257, 43690, 50001])
def test_embed_gradient(labels, dim, n):
    print("case embed gradient", labels, dim, n, flush=True)
    r = np.random.default_rng(n + labels)
    count = r.integers(0, 4, n)
    ptr = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    ids = r.integers(0, labels, int(ptr[-1]))
    ids[r.random(ids.size) < 0.1] = 7
    ids[1:][r.random(max(ids.size - 1, 0)) < 0.05] = ids[:1] if ids.size else 0
    minus = r.random(ids.size) < 0.3
    raw = np.where(minus, ids | 0x80000000, ids).astype(np.uint32)
    grad = r.standard_normal((n, dim)).astype(np.float32)
    term = grad[np.repeat(np.arange(n), count)].astype(np.float64) * np.where(minus, -1.0, 1.0)[:, None]
    want, mag = np.zeros((labels, dim)), np.zeros((labels, dim))
    np.add.at(want, ids, term)
    np.add.at(mag, ids, np.abs(term))
    named = np.bincount(ids, minlength=labels)
    tp, tl, tg = torch.from_numpy(ptr).cuda(), torch.from_numpy(np.append(raw, np.uint32(0)).view(np.int32)).cuda(), torch.from_numpy(grad).cuda()
    mark = torch.full((labels,), 5, dtype=torch.int32, device="cuda")
    lib = L.load()
    for _ in range(2):  # (marks of an earlier batch do not stay)
        out = torch.full((labels, dim), float("nan"), device="cuda")
        rc = getattr(lib.dll, EMBED_BACKWARD)(n, dim, C.c_void_p(tp.data_ptr()), C.c_void_p(tl.data_ptr()), C.byref(L.mat(tg)), C.byref(L.mat(out)), labels,
                                              C.c_void_p(mark.data_ptr()), lib.stream())
        assert rc == 0
        got = out.double().cpu().numpy()
        assert (got[named <= 1] == want[named <= 1]).all()
        assert (np.abs(got - want) <= named[:, None] * 2.0 ** -24 * mag).all()
        tp = torch.from_numpy(np.minimum(ptr, ptr[n // 2])).cuda()  # the second batch: half of the rows have no label
        k = int(ptr[n // 2])
        want, mag, named = np.zeros((labels, dim)), np.zeros((labels, dim)), np.bincount(ids[:k], minlength=labels)
        np.add.at(want, ids[:k], term[:k])
        np.add.at(mag, ids[:k], np.abs(term[:k]))


# both sides of every line of the choice: elements, rows, labels, rows to labels (few, many).  The marked form stores where one term names a label, the
# other adds to a cleared row, and both are sums in fp32 of any order; the marks tell which ran
@pytest.mark.parametrize("labels,dim,n,marked", [
    (57344, 1024, 57345, True), (57343, 1024, 57345, False), (65536, 896, 30720, True), (65536, 896, 30719, False), (45056, 1408, 40000, True), (45055, 1408, 40000, False),
    (81920, 768, 35840, True), (81920, 768, 35839, False), (58720, 1024, 88080, True), (58720, 1024, 88081, False)])
def test_choice_of_the_embed_gradient(labels, dim, n, marked):
    print("case embed gradient choice", labels, dim, n, marked, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    ids = (torch.rand(n, device="cuda", generator=gen) ** 2 * labels).long().clamp(0, labels - 1)
    minus = torch.rand(n, device="cuda", generator=gen) < 0.3
    raw = torch.where(minus, ids - 2 ** 31, ids).to(torch.int32)  # (the sign bit subtracts)
    ptr = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    grad = torch.randn((n, dim), device="cuda", generator=gen)
    mark = torch.full((labels,), 5, dtype=torch.int32, device="cuda")
    out = torch.full((labels, dim), float("nan"), device="cuda")
    lib = L.load()
    assert raw.numel() == n and int(ids.min()) >= 0 and int(ids.max()) < labels
    rc = getattr(lib.dll, EMBED_BACKWARD)(n, dim, C.c_void_p(ptr.data_ptr()), C.c_void_p(raw.data_ptr()), C.byref(L.mat(grad)), C.byref(L.mat(out)), labels,
                                          C.c_void_p(mark.data_ptr()), lib.stream())
    assert rc == 0
    assert bool((mark == 5).all()) != marked
    named = torch.bincount(ids, minlength=labels)
    for c in range(0, dim, 128):
        term = grad[:, c:c + 128].double() * torch.where(minus, -1.0, 1.0).double()[:, None]
        want = torch.zeros((labels, 128), device="cuda", dtype=torch.float64).index_add_(0, ids, term)
        size = torch.zeros((labels, 128), device="cuda", dtype=torch.float64).index_add_(0, ids, term.abs())
        got = out[:, c:c + 128].double()
        assert bool((got[named <= 1] == want[named <= 1]).all()) and bool(((got - want).abs() <= named[:, None] * 2.0 ** -24 * size).all())
