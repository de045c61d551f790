"""The packed deltas that wait for the end of a backward pass (one launch for all of them) against the same model in recompute mode, where every
layer's deltas run at once on the kernels for single products.  The operands are the same bits.  int8 sums are exact per k-tile, and the k-tiles
are added in the same groups: same bits (held to here up to four k-tiles, for more in a test of its own).  e4m3: fp32 sums are added in another order, which moves a value by far less than
the step of its tile (largest / 127) and can turn one rounding: one step, and the scale's own 1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tscale2_amd import lib as L  # noqa: E402


def deltas(mode, dim, heads, ffn, depth, k_tile, n, doc, recompute):
    lt, la, ls, widths = L.model_schedule(depth, 0, 64)
    vocab = 256
    m = L.Model(mode, dim, heads, ffn, lt, la, ls, len(widths), vocab, vocab + 1, n, k_tile=k_tile, recompute=recompute)
    try:
        r = np.random.default_rng(7)
        shapes = [(d, i, s) for d in range(len(lt)) for i, s in enumerate(L.layer_shapes(int(lt[d]), dim, heads, ffn, 0, 0))]
        for d, i, s in shapes + [(L.LAYER_EMBED, 0, (vocab + 1, dim)), (L.LAYER_FINAL, 0, (vocab, dim))]:
            w = r.standard_normal(s).astype(np.float32) * 32
            fast = np.clip(np.rint(w), -127, 127).astype(np.int8) if mode == L.I8 else torch.from_numpy(w).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
            m.set_matrix(d, i, fast, 0.2 if d == L.LAYER_EMBED else 0.02)
        m.set_bias(np.zeros(vocab, np.float32))
        t = np.arange(n, dtype=np.int32)
        start = t // doc * doc
        tokens = r.integers(0, vocab, n)
        target = np.append(tokens[1:], -1).astype(np.int32)
        spans = [(np.maximum(start, t - int(w)).astype(np.int32), np.where(t == start, -1, t - 1).astype(np.int32)) for w in widths]
        m.set_batch(np.arange(n + 1, dtype=np.int32), (1 + tokens).astype(np.uint32), target, [a for a, _ in spans], [b for _, b in spans],
                    L.fill_rope_buf(128, n))
        m.backprop()
        torch.cuda.synchronize()
        return [m.get_delta(d, i, *s) for d, i, s in shapes]
    finally:
        m.close()


# one tile of half its height, one row; widths off the 256-row tile; k-tiles of 128 to 1024, more than one register of scales holds; more matrices
# than one launch takes
@pytest.mark.parametrize("mode,dim,heads,ffn,depth,k_tile,n", [
    (L.I8, 128, 1, 128, 1, 128, 1), (L.I8, 384, 1, 640, 1, 256, 1000), (L.I8, 256, 3, 384, 1, 128, 8300), (L.I8, 512, 2, 1024, 1, 1024, 2500),
    (L.I8, 128, 1, 256, 18, 128, 257), (L.E4M3, 128, 1, 128, 1, 0, 1), (L.E4M3, 384, 1, 640, 1, 0, 1000), (L.E4M3, 256, 2, 512, 1, 0, 8300),
    (L.E4M3, 128, 3, 384, 18, 0, 129)])
def test_deltas_at_the_end_of_a_pass_equal_deltas_layer_by_layer(mode, dim, heads, ffn, depth, k_tile, n):
    print("case waiting deltas", mode, dim, heads, ffn, depth, k_tile, n, flush=True)
    args = (mode, dim, heads, ffn, depth, k_tile, n, 500)
    got, want = deltas(*args, False), deltas(*args, True)
    same = mode == L.I8 and -(-n // k_tile) <= 4
    for a, b in zip(got, want):
        assert np.isfinite(a).all() and (b.any() or n == 1)
        if same:
            assert np.array_equal(a, b)
            continue
        top = np.abs(b).reshape(b.shape[0], -1, 128).max(2).repeat(128, 1)
        assert (np.abs(a - b) <= top * (1.0 / 127 + 2e-5)).all()
        assert (a != b).mean() < 0.02 or (np.abs(a - b) <= 2e-5 * np.abs(b)).mean() > 0.98


# the groups of k-tiles: three and two, four each and three, one each beyond a register of scales
@pytest.mark.parametrize("dim,heads,ffn,depth,k_tile,n", [(256, 2, 384, 1, 128, 600), (384, 1, 640, 1, 128, 1400), (128, 1, 256, 2, 256, 5000), (256, 3, 384, 1, 128, 8300)])
def test_k_tiles_are_summed_as_layer_by_layer(dim, heads, ffn, depth, k_tile, n):
    print("case k-tile groups", dim, heads, ffn, depth, k_tile, n, flush=True)
    args = (L.I8, dim, heads, ffn, depth, k_tile, n, 500)
    for a, b in zip(deltas(*args, False), deltas(*args, True)):
        assert b.any() and np.array_equal(a, b)


WAITING = "_Z21Ts2ModelWaitingDeltasPK9ts2_model"
MODELS = [(L.I8, 256, 2, 384, 1, 128), (L.I8, 384, 1, 640, 2, 512), (L.E4M3, 256, 2, 512, 1, 0), (L.E4M3, 128, 3, 384, 3, 0)]


def model(mode, dim, heads, ffn, depth, k_tile, max_len, recompute=False):
    """a model with weights, and step(n): a batch of n tokens in documents of 100, one backward pass, every delta of its layers"""
    lt, la, ls, widths = L.model_schedule(depth, 0, 64)
    vocab = 256
    m = L.Model(mode, dim, heads, ffn, lt, la, ls, len(widths), vocab, vocab + 1, max_len, k_tile=k_tile, recompute=recompute)
    r = np.random.default_rng(7)
    shapes = [(d, i, s) for d in range(len(lt)) for i, s in enumerate(L.layer_shapes(int(lt[d]), dim, heads, ffn, 0, 0))]
    for d, i, s in shapes + [(L.LAYER_EMBED, 0, (vocab + 1, dim)), (L.LAYER_FINAL, 0, (vocab, dim))]:
        w = r.standard_normal(s).astype(np.float32) * 32
        fast = np.clip(np.rint(w), -127, 127).astype(np.int8) if mode == L.I8 else torch.from_numpy(w).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
        m.set_matrix(d, i, fast, 0.2 if d == L.LAYER_EMBED else 0.02)
    m.set_bias(np.zeros(vocab, np.float32))

    def step(n):
        tokens = np.random.default_rng(n).integers(0, vocab, n)
        t = np.arange(n, dtype=np.int32)
        start = t // 100 * 100
        spans = [(np.maximum(start, t - int(w)).astype(np.int32), np.where(t == start, -1, t - 1).astype(np.int32)) for w in widths]
        m.set_batch(np.arange(n + 1, dtype=np.int32), (1 + tokens).astype(np.uint32), np.append(tokens[1:], -1).astype(np.int32), [a for a, _ in spans],
                    [b for _, b in spans], L.fill_rope_buf(128, n))
        m.backprop()
        torch.cuda.synchronize()
        return [m.get_delta(d, i, *s) for d, i, s in shapes]
    return m, step, len(lt)


# every attention and feed-forward layer of such models leaves two (its stack and its last matrix), none where activations are recomputed
@pytest.mark.parametrize("args", MODELS)
def test_deltas_do_wait(args):
    print("case deltas that wait", args, flush=True)
    for recompute in (False, True):
        m, step, layers = model(*args, 500, recompute)
        try:
            step(500)
            assert getattr(m.lib.dll, WAITING)(m.h) == (0 if recompute else 2 * layers)
        finally:
            m.close()


# what a longer batch left in the kept gradients, row maxima, scales and state gradients does not reach a shorter one: the bits of a model that saw
# the short batch alone.  Ends inside a row tile, on one, one row; longer again
@pytest.mark.parametrize("args", MODELS)
@pytest.mark.parametrize("lengths", [(1000, 333), (900, 256, 1), (700, 1, 650)])
def test_a_shorter_batch_after_a_longer_one(args, lengths):
    print("case shorter batch", args, lengths, flush=True)
    m, step, _ = model(*args, 1000)
    try:
        for n in lengths:
            got = step(n)
            assert getattr(m.lib.dll, WAITING)(m.h) > 0
    finally:
        m.close()
    m, step, _ = model(*args, 1000)
    try:
        want = step(lengths[-1])
    finally:
        m.close()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
