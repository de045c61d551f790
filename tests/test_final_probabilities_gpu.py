"""Probabilities of ts2_model_forward around the vocabularies where a row changes from one wave to four, eight and sixteen, and to the two-pass kernel,
and where a lane's share grows.  The logits are overwritten, so a pass without bias gives them up to a constant (p0), and a pass with a bias b
must give p0 2^b / sum(p0 2^b): everything in fp32, so 2^-20 of a value holds with room for the exponential's own error (arguments up to 30 carry
30 * 2^-24 * ln 2 = 2^-19.6), and below 1e-30 nothing is asked."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from model_harness import E4M3, I8, Harness  # noqa: E402
from test_model_batches_gpu import batch, load  # noqa: E402


@pytest.mark.parametrize("vocab", [128, 512, 640, 1024, 1152, 2048, 2176, 4096, 4224, 8192, 8320, 16384, 16512, 26624, 26752, 53248, 53376])
def test_probabilities_follow_the_bias(vocab):
    print("case probabilities", vocab, flush=True)
    h = Harness(E4M3, dim=256, heads=1, ffn_tiles=1, depth=2, vocab=vocab, frag_count=2, frag_len=64, wide_window=64, seed=7)
    r = np.random.default_rng(vocab)
    bias = (r.standard_normal(vocab) * 2).astype(np.float32)
    bias[vocab - 1] = 9.0
    tokens = r.integers(0, vocab, 67)
    m = load(h, 67)
    try:
        n = batch(m, h, tokens, 50)
        p = []
        for b in (np.zeros(vocab, np.float32), bias):
            m.set_bias(b)
            m.forward()
            torch.cuda.synchronize()
            p.append(m.array("prediction")[:n, :vocab].double().cpu().numpy())
        g = m.array("finalGrad")[:n, :vocab].double().cpu().numpy()
    finally:
        m.close()
    want = p[0] * np.exp2(bias.astype(np.float64))
    want /= want.sum(1, keepdims=True)
    assert (np.abs(p[1] - want) <= 2.0 ** -17 * want + 1e-30).all()
    assert np.abs(p[1].sum(1) - 1).max() < 1e-5
    grad = -p[1]
    has = np.array([t % 50 != 49 and t != n - 1 for t in range(n)])
    rows = np.nonzero(has)[0]
    grad[rows, tokens[rows + 1]] += 1
    grad[~has] = 0
    assert (np.abs(g - grad) <= 2.0 ** -8 * np.abs(grad) + 1e-30).all()


@pytest.mark.parametrize("vocab", [128, 53248, 53376])
@pytest.mark.parametrize("big", [60.0, 70.0, 300.0, 1e5])
def test_large_bias(vocab, big):
    """two entries whose bias stands far above the logits (all below 1 in size) share the probability as 2 to 1.  In fp32 a sum of
    about 1e5 is rounded by up to 2^-8 (of about 300 by 2^-16): two of them, ln 2 / 3 of which reaches the probability, are 1.8e-3 < 2^-9"""
    print("case large bias", vocab, big, flush=True)
    h = Harness(I8, dim=256, heads=1, ffn_tiles=1, depth=2, vocab=vocab, frag_count=2, frag_len=64, wide_window=64, seed=7)
    bias = np.zeros(vocab, np.float32)
    bias[5], bias[vocab - 1] = big, big - 1
    m = load(h, 67)
    try:
        n = batch(m, h, np.random.default_rng(vocab).integers(0, vocab, 67), 50)
        p = []
        for b in (np.zeros(vocab, np.float32), bias):
            m.set_bias(b)
            m.forward()
            torch.cuda.synchronize()
            p.append(m.array("prediction")[:n, :vocab].double().cpu().numpy())
    finally:
        m.close()
    a, b = p[0][:, 5] * 2, p[0][:, vocab - 1]
    np.testing.assert_allclose(p[1][:, 5], a / (a + b), rtol=2 ** -9 if big > 1e4 else 2 ** -15)
    np.testing.assert_allclose(p[1].sum(1), 1, rtol=1e-6)
