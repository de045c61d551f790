"""The step driver over batches of several lengths: what a batch leaves in the model's arrays must not reach the next one, and the products
chosen for a long batch must give what those chosen for a short one give."""
from types import SimpleNamespace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from model_harness import E4M3, I8, Harness, rel_err, scale_fit  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402


def spans(n, doc, width):
    t = np.arange(n, dtype=np.int32)
    start = t // doc * doc
    return np.maximum(start, t - width).astype(np.int32), np.where(t == start, -1, t - 1).astype(np.int32)


def load(h, max_len):
    m = L.Model(h.mode, h.dim, h.heads, h.ffn, h.lt, h.la, h.ls, len(h.att_width), h.vocab, h.label_count, max_len,
                h.xp if h.experts else 0, h.experts, h.selected if h.experts else 0)
    for d in range(h.depth):
        for i, q in enumerate(h.layers[d]):
            m.set_matrix(d, i, q.fast, q.scale)
    m.set_matrix(L.LAYER_EMBED, 0, h.embed.fast, h.embed.scale)
    m.set_matrix(L.LAYER_FINAL, 0, h.final.fast, h.final.scale)
    m.set_bias(h.bias)
    return m


def batch(m, h, tokens, doc):
    n = tokens.size
    target = np.full(tokens.shape, -1, np.int32)
    target[:-1] = tokens[1:]
    target[doc - 1::doc] = -1
    s = [spans(n, doc, int(w)) for w in h.att_width]
    m.set_batch(np.arange(n + 1, dtype=np.int32), (1 + tokens).astype(np.uint32), target, [a for a, _ in s], [b for _, b in s], L.fill_rope_buf(128, n))
    return n


def results(m, h, n):
    torch.cuda.synchronize()
    return [m.get_delta(d, i, *q.fast.shape) for d in range(h.depth) for i, q in enumerate(h.layers[d])] + \
        [m.get_delta(L.LAYER_FINAL, 0, h.vocab, h.dim), m.array("stateGrad").float().cpu().numpy()[:n]]


@pytest.mark.parametrize("mode,dim,experts", [(I8, 256, 0), (E4M3, 256, 0), (E4M3, 384, 0), (E4M3, 256, 8)])
@pytest.mark.parametrize("n", [1, 129, 777])
def test_a_short_batch_after_a_long_one_equals_the_same_batch_alone(mode, dim, experts, n):
    """rows beyond the batch, of what a longer batch left in the model's arrays: int8 delta products read them up to the end of the last row
    group, at these sizes e4m3 ones stop at the last live row (the large tile does not: next test)"""
    print("case short batch after a long one", mode, dim, experts, n, flush=True)
    h = Harness(mode, dim=dim, heads=2, ffn_tiles=4, depth=2, vocab=256, frag_count=2, frag_len=64, wide_window=64, seed=3, experts=experts)
    r = np.random.default_rng(5)
    long, short = r.integers(0, h.vocab, 1500), r.integers(0, h.vocab, n)
    out = []
    for first in (long, None):
        m = load(h, long.size)
        try:
            if first is not None:
                batch(m, h, first, 500)
                m.backprop()
            k = batch(m, h, short, n)
            m.backprop()
            out.append(results(m, h, k))
        finally:
            m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)


class Weights:
    """e4m3 weights drawn on the device: models whose oracle copy would take minutes"""

    def __init__(self, dim, heads, ffn, vocab, seed):
        self.mode, self.dim, self.heads, self.ffn, self.vocab, self.label_count = E4M3, dim, heads, ffn, vocab, vocab + 1
        self.experts = 0
        self.lt, self.la, self.ls, self.att_width = L.model_schedule(1, 0, 64)
        self.depth = len(self.lt)
        gen = torch.Generator(device="cuda").manual_seed(seed)

        def matrix(rows, cols):
            return SimpleNamespace(fast=(torch.randn((rows, cols), device="cuda", generator=gen) * 32).to(torch.float8_e4m3fn).view(torch.uint8).cpu().numpy(),
                                   scale=0.02)
        self.layers = [[matrix(r, c) for r, c in L.layer_shapes(int(t), dim, heads, ffn)] for t in self.lt]
        self.embed, self.final = matrix(self.label_count, dim), matrix(vocab, dim)
        self.bias = np.zeros(vocab, np.float32)


def reads_rows_beyond(m, layer, n, shape):
    """whether the delta of a layer's first matrix changes when its source holds NaN beyond the batch: the 256x256 tile contracts over the
    whole row group (its gradients are zero there, NaN times zero is not), the kernel for few tiles stops at the last live row"""
    grad = torch.randn(tuple(m.array("stateGrad").shape), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    m.layer_forward(layer)
    out = []
    for poison in (False, True):
        m.array("stateGrad").copy_(grad)
        m.array("gradMaxNorm")[0, 0] = grad.abs().max()
        if poison:
            m.array("normState", layer)[n:].fill_(0x7f)
        m.layer_backward(layer)
        out.append(m.get_delta(layer, 0, *shape))
    return not np.array_equal(*out)


@pytest.mark.parametrize("dim,heads,ffn,rows,n", [(1024, 8, 2048, 16384, 12001), (2048, 16, 4096, 4096, 2777)])
def test_a_short_batch_after_a_long_one_where_the_large_tile_reads_whole_row_groups(dim, heads, ffn, rows, n):
    """e4m3 widths on the 256 grid and results large enough for the 256x256 tile, in stored slices that are packed (dim 1024) and whole (dim
    2048): its delta products read the rows beyond the batch, so what a longer batch left there must be gone"""
    print("case large tile after a long batch", dim, rows, n, flush=True)
    h = Weights(dim, heads, ffn, 512, 21)
    r = np.random.default_rng(22)
    long, short = r.integers(0, h.vocab, rows), r.integers(0, h.vocab, n)
    out, beyond = [], []
    for first in (long, None):
        m = load(h, rows)
        try:
            if first is not None:
                batch(m, h, first, 512)
                m.backprop()
            k = batch(m, h, short, 512)
            m.backprop()
            out.append(results(m, h, k))
            if first is None:
                beyond = [reads_rows_beyond(m, d, n, h.layers[d][0].fast.shape) for d in range(h.depth)]
        finally:
            m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and a.any() and np.array_equal(a, b)
    assert all(beyond), beyond  # (else these sizes no longer test what they are here for)


@pytest.mark.parametrize("mode,dim", [(I8, 384), (E4M3, 384)])
def test_repeated_documents_have_equal_gradients_and_summed_deltas(mode, dim):
    """40 copies of a 512-token document (20480 rows: the products for large results, int8 dX as one sum) against two copies (1024 rows:
    the kernel for few tiles).  Every copy's gradient is that of the short batch and the deltas are 20 times its deltas, up to what 8-bit
    storage makes of results that are rounded to bf16 from sums in another order (a value at a tie moves by one step of 1/254 of its row's
    largest or of 2^-4 of itself, a few in a hundred do)."""
    print("case repeated documents", mode, dim, flush=True)
    h = Harness(mode, dim=dim, heads=2, ffn_tiles=3, depth=2, vocab=256, frag_count=2, frag_len=64, wide_window=64, seed=4)
    doc = np.random.default_rng(6).integers(0, h.vocab, 512)
    out = []
    for copies in (2, 40):
        m = load(h, 512 * copies)
        try:
            n = batch(m, h, np.tile(doc, copies), 512)
            m.backprop()
            out.append(results(m, h, n))
        finally:
            m.close()
    small, large = out
    for c in range(40):
        rms, _ = rel_err(large[-1][512 * c:512 * (c + 1)], small[-1][:512])
        assert rms <= 2e-2, (c, rms)
    for i, (a, b) in enumerate(zip(large[:-1], small[:-1])):
        fit, corr = scale_fit(a, 20 * b)
        print("matrix", i, "fit", fit, "correlation", corr)
        assert abs(fit - 1) <= 5e-3 and corr >= 0.999


@pytest.mark.parametrize("top", [0.5, 200.0])
@pytest.mark.parametrize("vocab", [128, 512, 640, 1152, 1664, 2048, 2176])
def test_final_gradient_of_small_vocabularies(vocab, top):
    """(one-hot - soft-max) of every row against fp64, around the vocabularies where a wave's share of a row grows by a chunk and where the
    workgroup kernel takes over; also with one bias no exponential holds by itself.  Logits travel in half (2^-11 of a logit, here below 4:
    4 * 2^-11 * ln 2 = 1.4e-3 of a probability), the gradient in bf16 (2^-9)."""
    print("case final gradient", vocab, top, flush=True)
    h = Harness(E4M3, dim=256, heads=1, ffn_tiles=1, depth=2, vocab=vocab, frag_count=2, frag_len=64, wide_window=64, seed=7)
    bias = (np.random.default_rng(8).standard_normal(vocab) * 0.5).astype(np.float32)
    bias[vocab // 3] = top
    m = load(h, 200)
    try:
        n = batch(m, h, np.random.default_rng(9).integers(0, vocab, 200), 50)
        m.set_bias(np.zeros(vocab, np.float32))
        m.forward()
        torch.cuda.synchronize()
        x = np.log2(m.array("prediction")[:n, :vocab].double().cpu().numpy())
        m.set_bias(bias)
        m.backprop()
        torch.cuda.synchronize()
        got = m.array("finalGrad")[:n, :vocab].double().cpu().numpy()
        loss = m.loss_sum()
        tokens = np.random.default_rng(9).integers(0, vocab, 200)
    finally:
        m.close()
    x = x + bias
    p = np.exp2(x - x.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    rows = np.array([t for t in range(n) if t % 50 != 49])
    want = np.zeros_like(p)
    want[rows] = -p[rows]
    want[rows, tokens[rows + 1]] += 1
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 6e-3 * p + 1e-7).all()
    if top < 1:
        ref = np.log(p[rows, tokens[rows + 1]]).sum()
        assert abs(loss - ref) <= 2e-3 * abs(ref)
