"""The state a batch starts from, at the lengths where a workgroup of the embedding pass takes one row, two and four: rows without a label, with
one, with several, labels that are subtracted.  Sums of a few 8-bit values times one scale in fp32, in the order of the labels: each of up to
four terms rounds once in the product and once in the sum, 8 * 2^-24 of the largest partial sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from model_harness import E4M3, I8, Harness  # noqa: E402
from test_model_batches_gpu import load, spans  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402


@pytest.mark.parametrize("mode", [I8, E4M3])
@pytest.mark.parametrize("n", [1, 130, 8191, 8193, 12161, 12291, 32641, 32771])
def test_embedded_state(mode, n):
    print("case embedding", mode, n, flush=True)
    h = Harness(mode, dim=256, heads=1, ffn_tiles=1, depth=2, vocab=256, frag_count=2, frag_len=64, wide_window=64, seed=9)
    r = np.random.default_rng(n)
    count = r.integers(0, 5, n)
    ptr = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    ids = r.integers(0, h.label_count, int(ptr[-1])).astype(np.uint32)
    minus = r.random(ids.size) < 0.3
    labels = np.where(minus, ids | np.uint32(0x80000000), ids).astype(np.uint32)
    values = h.embed.fast.astype(np.float64) if mode == I8 else torch.from_numpy(h.embed.fast.view(np.uint8).copy()).view(torch.float8_e4m3fn).double().numpy()
    want = np.zeros((n, h.dim))
    rows = np.repeat(np.arange(n), count)
    np.add.at(want, rows, values[ids] * np.where(minus, -1.0, 1.0)[:, None])
    m = load(h, n)
    try:
        for d in range(h.depth):  # layers that add nothing: the state stays what the embedding made it
            for i, q in enumerate(h.layers[d]):
                m.set_matrix(d, i, np.zeros_like(q.fast), q.scale)
        s = [spans(n, 64, int(w)) for w in h.att_width]
        target = np.full(n, -1, np.int32)
        m.set_batch(ptr, labels if labels.size else np.zeros(1, np.uint32), target, [a for a, _ in s], [b for _, b in s], L.fill_rope_buf(128, n))
        m.forward()
        torch.cuda.synchronize()
        got = m.array("state")[:n].double().cpu().numpy()
    finally:
        m.close()
    ratio = (got * want).sum() / max((want * want).sum(), 1e-30)  # the driver's factor: matrix scale times a constant
    assert np.abs(got - want * ratio).max() <= 2.0 ** -20 * np.abs(want * ratio).max()
