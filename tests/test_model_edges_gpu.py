"""What the step driver's accessors show at the edges: rows beyond the batch, gradient scratch by layer type, wide k-tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from model_harness import E4M3, I8, Harness  # noqa: E402
from tscale2_amd import lib as L  # noqa: E402


def test_gradient_scratch_of_a_mixture_of_experts_layer_is_its_own():
    """"scratch.f0" / "scratch.f1" after the backward of a mixture-of-experts layer are its gradients of the expand and gate products, not
    those of the attention layer before it: expert 0's rows come first (one tile of 128), and its packed deltas are sums of products with
    exactly those rows, so they lie in the rows' span up to the packing (1/254 of a row-tile's largest value per element)."""
    print("case gradient scratch of an expert layer", flush=True)
    h = Harness(E4M3, dim=256, heads=2, ffn_tiles=2, depth=3, vocab=256, frag_count=2, frag_len=30, wide_window=64, experts=8, selected=2, xp=128,
                seed=11, std=0.05)
    att, moe = list(h.lt).index(0), list(h.lt).index(3)
    m = h.device_model()
    try:
        m.backprop()
        torch.cuda.synchronize()
        G = m.array("stateGrad").clone()
        for layer in (att, moe):
            m.array("stateGrad").copy_(G)
            m.array("gradMaxNorm")[0, 0] = G.abs().max()
            m.layer_forward(layer)
            m.layer_backward(layer)
        torch.cuda.synchronize()
        for i in (0, 1):
            rows = m.array(f"scratch.f{i}", 128)[:128].contiguous().view(torch.float8_e4m3fn).double().cpu()
            d = torch.from_numpy(m.get_delta(moe, i, 8 * 128, h.dim)[:128]).double()
            assert 2 <= int(rows.any(1).sum()) <= 64 and bool(d.any())
            _, s, basis = torch.linalg.svd(rows, full_matrices=False)
            basis = basis[s > 1e-6 * s.max()]
            left = d - basis.t() @ (basis @ d)
            print("matrix", i, "rows", len(basis), "outside the span", float(left.norm() / d.norm()))
            assert float(left.norm()) <= 0.03 * float(d.norm())
    finally:
        m.close()


@pytest.mark.parametrize("mode", [I8, E4M3])
def test_predictions_beyond_the_batch_are_probabilities_too(mode):
    """the view has every row of the last row group: rows beyond the batch have logits zero, so they hold the soft-max of the bias"""
    print("case predictions beyond the batch", mode, flush=True)
    h = Harness(mode, dim=256, heads=2, ffn_tiles=2, depth=1, vocab=384, frag_count=1, frag_len=100, wide_window=64, seed=12, bias_std=1.0)
    m = h.device_model()
    try:
        m.forward()
        torch.cuda.synchronize()
        p = m.array("prediction")[:, :h.vocab].double().cpu().numpy()
    finally:
        m.close()
    assert p.shape[0] > h.n
    assert np.abs(p.sum(1) - 1).max() <= 1e-5
    want = np.exp2(h.bias.astype(np.float64))
    assert np.abs(p[h.n:] - want / want.sum()).max() <= 1e-6


def test_k_tiles_too_wide_for_the_row_major_delta_product():
    """int8, one k-tile of 32768 rows over two gradients of 4096 columns side by side: the product that reads them as they lie cannot
    address a k-tile's rows, so the step takes the transposing sequence.  The batch fills a part of one k-tile either way: the same
    scales, the same exact integer sums, so the same deltas as with k-tiles of 16384."""
    print("case wide k-tiles", flush=True)
    h = Harness(I8, dim=128, heads=1, ffn_tiles=32, depth=1, vocab=128, frag_count=2, frag_len=150, wide_window=64, seed=13)
    out = []
    for k_tile in (16384, 32768):
        m = h.device_model(k_tile=k_tile)
        try:
            m.backprop()
            torch.cuda.synchronize()
            out.append([m.get_delta(d, i, *q.fast.shape) for d in range(h.depth) for i, q in enumerate(h.layers[d])])
        finally:
            m.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and a.any() and np.array_equal(a, b)
