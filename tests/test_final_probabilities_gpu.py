"""Probabilities of ts2_model_forward around the vocabularies where a row changes from one wave to four, eight and sixteen, and to the two-pass kernel,
and where a lane's share grows.  The logits are overwritten: a pass without bias gives them up to a constant (p0), and a pass with a bias b must
give p0 2^b / sum(p0 2^b), which holds to 2^-17 (two passes, each within the bound of test_probabilities_against_float64, at logits up to 40: 12 + 44 + ln 2 120
units of 2^-24); below 1e-30 nothing is asked.  The tests against 64 bits compare with logits formed from the final state and the head matrix."""
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


@pytest.mark.parametrize("spread", [0, 3, 30, -3])
@pytest.mark.parametrize("vocab", [128, 512, 640, 1024, 1152, 2048, 2176, 4224, 8192, 8320, 16384, 16512, 26752, 32768, 32896, 53248, 53376])
def test_probabilities_against_float64(vocab, spread):
    """Base-2 soft-max in 64 bits of the final state times the head matrix (exact int8 products, one scale).  A probability rounds in its
    logit's factor (few roundings of a logit below 0.2), in logit + bias (u |x|, u = 2^-24), in its argument relative to a largest logit beyond
    64 (u |x - max|), in the exponential, the reciprocal and the product (4 roundings), and in the sum, whose at most 40 roundings, weighted
    by the part summed so far, come to u sqrt(40 / 9) rms; the sum also carries the rounding of its largest terms' logits (u |max|).  In all less than
    4 u + ln 2 u (|x| + |max| + |x - max|) in the root mean square; no single value is off by more than all of them added, 44 u + ...
    Spread 30 passes 64 and -126; -3: one logit at -200 and one at minus infinity"""
    print("case probabilities float64", vocab, spread, flush=True)
    h = Harness(I8, dim=256, heads=1, ffn_tiles=1, depth=2, vocab=vocab, frag_count=2, frag_len=64, wide_window=64, seed=7)
    r = np.random.default_rng(vocab)
    bias = (r.standard_normal(vocab) * abs(spread)).astype(np.float32)
    if spread < 0:
        bias[1], bias[2] = -200, -np.inf
    m = load(h, 67)
    try:
        n = batch(m, h, r.integers(0, vocab, 67), 50)
        m.set_bias(bias)
        m.forward()
        torch.cuda.synchronize()
        p = m.array("prediction")[:n, :vocab].double().cpu().numpy()
        state = m.array("normState", h.depth)[:n].double().cpu().numpy()
    finally:
        m.close()
    factor = 1 / 24 / 32 / 16 / float(np.float32(0.693147)) * float(np.float32(h.final.scale))  # vector scale, matrix scale, 256^-1/2, log 2
    x = state @ h.final.fast.astype(np.float64).T * factor + bias
    top = x.max(1, keepdims=True)
    want = np.exp2(x - top)
    want /= want.sum(1, keepdims=True)
    assert (p[want < 1e-38] <= 2e-38).all()
    some = want > 1e-30
    u = 2.0 ** -24
    unit = u * np.log(2) * (np.abs(x) + np.abs(top) + np.where(np.abs(top) > 64, np.abs(x - top), 0))
    rel = (np.abs(p - want) / np.where(some, want, 1))[some]
    print("  rms", np.sqrt((rel ** 2).mean()) / u, "u, max", rel.max() / u, "u, of the bound", np.sqrt(((rel / (4 * u + unit[some])) ** 2).mean()), flush=True)
    assert np.sqrt(((rel / (4 * u + unit[some])) ** 2).mean()) <= 1
    assert (rel <= 44 * u + unit[some]).all()


@pytest.mark.parametrize("vocab", [128, 2048, 8192, 53248, 53376])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_rows_without_a_target_have_no_gradient(vocab, bad):
    """one logit that is not finite makes its rows' probabilities NaN; the gradient of a row without a target is zero all the same"""
    print("case rows without a target", vocab, bad, flush=True)
    h = Harness(I8, dim=256, heads=1, ffn_tiles=1, depth=2, vocab=vocab, frag_count=2, frag_len=64, wide_window=64, seed=7)
    bias = np.zeros(vocab, np.float32)
    bias[5] = bad
    m = load(h, 67)
    try:
        n = batch(m, h, np.random.default_rng(vocab).integers(0, vocab, 67), 50)
        m.set_bias(bias)
        m.forward()
        torch.cuda.synchronize()
        p = m.array("prediction")[:n, :vocab].float().cpu().numpy()
        g = m.array("finalGrad")[:n, :vocab].float().cpu().numpy()
    finally:
        m.close()
    none = np.array([t % 50 == 49 or t == n - 1 for t in range(n)])
    assert (g[none] == 0).all() and np.isnan(p).all() and np.isnan(g[~none]).all()
