"""The forms of the attention kernels, which a rule on the number of workgroups (and on the key range of a workgroup) chooses between:
a pipelined forward for long key ranges and a plain one for narrow windows; the backward as one launch with two waves (or pairs of waves)
per row block where few workgroups are asked for both its halves, as one launch for dQ and one for dK and dV otherwise, with the score gradients
handed from one to the other or formed twice.  The repetition of two heads of data fills a launch of any size, and the oracle computes those two only.
Inputs are bf16-representable; the device rounds probabilities and score gradients to bf16 before a product, hence the same tolerance as in
test_attention_gpu.py: max |err| <= 1e-2 * max |ref| per tensor."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from oracle_lib import Oracle  # noqa: E402
from test_attention_gpu import bf16_round, ragged_spans, spans_to_ranges  # noqa: E402

SCALE = float(np.float32(np.sqrt(np.float32(1.0 / 128))) * np.float32(0.5 / 0.693147))


@pytest.fixture(scope="module")
def L():
    from tscale2_amd import lib
    lib.load()
    return lib


@pytest.fixture(scope="module")
def orc():
    return Oracle()


def device_pass(L, n, heads, arrays, start, finish, slope, scale=SCALE, dscale=None):
    """val, sumWeightLog and, with dscale, dq, dk, dv (each [n_round, heads * 128], statistics [heads, n_round])"""
    n_round, i16 = start.size, torch.int16

    def padded(a):
        t = torch.zeros((n_round, a.shape[1]), dtype=torch.bfloat16, device="cuda")
        t[:n] = torch.from_numpy(a).cuda().bfloat16()
        return t
    q, k, v, dval = [padded(a) for a in arrays]
    ts, tf = torch.from_numpy(start).cuda(), torch.from_numpy(finish).cuda()
    out = [torch.full((n_round, heads * 128), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    swl = torch.full((heads, n_round), -5.0, device="cuda")
    L.att_forward(n, heads, q.view(i16), k.view(i16), v.view(i16), ts, tf, scale, slope, out[0].view(i16), swl)
    if dscale is not None:
        ds = torch.zeros((heads, n_round), device="cuda")
        ds[:, :n] = torch.from_numpy(dscale).cuda()
        lo = torch.zeros(n_round // 128, dtype=torch.int32, device="cuda")
        hi = torch.zeros_like(lo)
        L.call("ts2_att_build_rev", n, n_round, ts, tf, lo, hi)
        L.att_backward(n, heads, q.view(i16), k.view(i16), v.view(i16), dval.view(i16), ts, tf, lo, hi, scale, slope, swl, ds,
                       *[t.view(i16) for t in out[1:]], L.BF16)
    torch.cuda.synchronize()
    return out, swl


def inputs(n, heads, seed, q_mul=1.0):
    r = np.random.default_rng(seed)
    a = [bf16_round(r.standard_normal((n, heads * 128)).astype(np.float32)) for _ in range(4)]
    a[0] = bf16_round(a[0] * np.float32(q_mul))
    return a


# documents, window, heads of the launch, slope.  1100 tokens are nine 128-row blocks: with 2 heads the backward is one launch of 54 workgroups,
# with 10 and 16 it is two.  Windows of 40 keep a workgroup's keys within seven tiles, whole documents go beyond; 64 and 65 tokens end a document
# on a tile and one past it
CASES = [
    ([300, 1, 299, 500], 40, 2, 0.0), ([300, 1, 299, 500], 40, 16, 0.0), ([300, 1, 299, 500], 40, 16, 0.25),
    ([1100], 4096, 10, 0.0), ([1100], 4096, 16, 0.0), ([1100], 4096, 16, 0.01), ([1100], 4096, 2, 0.01),
    ([64, 65, 63, 128, 129, 651], 300, 16, 0.0), ([64, 65, 63, 128, 129, 651], 300, 2, 0.125), ([64, 65, 63, 128, 129, 651], 4096, 10, 0.125),
    ([31, 33, 1, 5], 4096, 1, 0.0), ([1], 4096, 1, 0.0),
]


@pytest.mark.parametrize("docs,window,heads,slope", CASES)
def test_forms_against_the_oracle(L, orc, docs, window, heads, slope):
    print("case att forms", docs, window, heads, slope, flush=True)
    sp, spans = ragged_spans(docs, window)
    n, base = sp.size - 1, min(heads, 2)
    n_round = (n + 127) // 128 * 128
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    a = inputs(n, base, seed=n + heads)
    ref = orc.attention(base, 128, 128, slope, sp, spans, *a)
    rep = heads // base
    out, swl = device_pass(L, n, heads, [np.tile(x, (1, rep)) for x in a], start, finish, slope, dscale=np.tile(ref["dscale"], (rep, 1)))
    want_l = ref["max_dp"] + np.log2(ref["sum_weight"])
    np.testing.assert_allclose(swl.cpu().numpy()[:, :n], np.tile(want_l, (rep, 1)), rtol=1e-4, atol=1e-4)
    for name, t in zip(("val", "dq", "dk", "dv"), out):
        g = t.float().cpu().numpy()
        assert np.all(g[n:] == 0), name
        for h in range(rep):
            got = g[:n, h * base * 128:(h + 1) * base * 128]
            assert np.abs(got - ref[name]).max() <= 1e-2 * max(np.abs(ref[name]).max(), 1e-30), (name, h)


@pytest.mark.parametrize("docs,window,heads,slope", [([300, 1, 299, 500], 40, 10, 0.25), ([1100], 4096, 10, 0.0), ([64, 65, 63, 128, 129, 651], 300, 16, 0.125),
                                                      ([64, 65, 63, 128, 129, 651], 300, 16, 0.0), ([300, 1, 299, 500], 40, 2, 0.0), ([1100], 4096, 2, 0.01)])
@pytest.mark.parametrize("f32", [False, True])
def test_backward_in_every_way_it_can_be_asked_for(L, orc, docs, window, heads, slope, f32):
    """gradients in fp32 and bf16; both bits, one bit at a time, both with the score gradients handed over (over NaN patterns).  With 10 and 16 heads
    the two kernels run one after the other whatever is asked for: the bits of dK and dV are the same in every way, those of dQ but for the
    hand-over.  With 2 heads both bits are one launch, which adds a gradient in two halves.  Row blocks that straddle document starts are seen
    partly by one key block of a workgroup and completely by the other, so the dK/dV waves take their two-block and one-block paths in turn"""
    print("case att ways", docs, window, heads, slope, f32, flush=True)
    sp, spans = ragged_spans(docs, window)
    n, i16, rep = sp.size - 1, torch.int16, heads // 2
    n_round = (n + 127) // 128 * 128
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    a = inputs(n, 2, seed=n + heads)
    ref = orc.attention(2, 128, 128, slope, sp, spans, *a)

    def padded(x):
        t = torch.zeros((n_round, heads * 128), dtype=torch.bfloat16, device="cuda")
        t[:n] = torch.from_numpy(np.tile(x, (1, rep))).cuda().bfloat16()
        return t.view(i16)
    q, k, v, dval = [padded(x) for x in a]
    ts, tf = torch.from_numpy(start).cuda(), torch.from_numpy(finish).cuda()
    val, swl = torch.zeros_like(q), torch.zeros((heads, n_round), device="cuda")
    L.att_forward(n, heads, q, k, v, ts, tf, SCALE, slope, val, swl)
    lo = torch.zeros(n_round // 128, dtype=torch.int32, device="cuda")
    hi = torch.zeros_like(lo)
    L.call("ts2_att_build_rev", n, n_round, ts, tf, lo, hi)
    ds = torch.zeros((heads, n_round), device="cuda")
    ds[:, :n] = torch.from_numpy(np.tile(ref["dscale"], (rep, 1))).cuda()
    handed = L.att_ds_scratch(n_round, heads, ts, tf)
    handed[1].fill_(0x7f)

    def back(which, pair=None):
        o = [torch.full((n_round, heads * 128), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda") for _ in range(3)]
        L.att_backward(n, heads, q, k, v, dval, ts, tf, lo, hi, SCALE, slope, swl, ds, *[t if f32 else t.view(i16) for t in o], L.F32 if f32 else L.BF16,
                       which=which, ds=pair)
        torch.cuda.synchronize()
        return o
    both, dq_only, dkv_only, via = back(3), back(1), back(2), back(3, handed)
    assert (dq_only[1] == 7).all() and (dq_only[2] == 7).all() and (dkv_only[0] == 7).all()
    apart = [dq_only[0], dkv_only[1], dkv_only[2]]
    for ways in (both, apart, via):
        for name, t in zip(("dq", "dk", "dv"), ways):
            g = t.float().cpu().numpy()
            assert np.all(g[n:] == 0), name
            for h in range(rep):
                assert np.abs(g[:n, h * 256:(h + 1) * 256] - ref[name]).max() <= 1e-2 * np.abs(ref[name]).max(), (name, h)
    if heads > 2:
        assert all(torch.equal(x, y) for x, y in zip(both, apart))
        assert torch.equal(via[1], both[1]) and torch.equal(via[2], both[2]) and not (handed[1] == 0x7f).all()
    else:
        assert all(torch.equal(x, y) for x, y in zip(both, via)) and (handed[1] == 0x7f).all()


@pytest.mark.parametrize("heads", [2, 16])
def test_logits_far_beyond_the_reference(L, orc, heads):
    """logits of +-40: the reference of the running weights has to move, in the middle of a sequence too; peaked weights"""
    print("case att large logits", heads, flush=True)
    sp, spans = ragged_spans([1100], 4096)
    n, n_round = 1100, 1152
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    a = inputs(n, 2, seed=5, q_mul=14.0)
    ref = orc.attention(2, 128, 128, 0.0, sp, spans, *a)
    assert ref["max_dp"].max() > 24
    rep = heads // 2
    out, swl = device_pass(L, n, heads, [np.tile(x, (1, rep)) for x in a], start, finish, 0.0, dscale=np.tile(ref["dscale"], (rep, 1)))
    np.testing.assert_allclose(swl.cpu().numpy()[:, :n], np.tile(ref["max_dp"] + np.log2(ref["sum_weight"]), (rep, 1)), rtol=1e-4, atol=1e-4)
    for name, t in zip(("val", "dq", "dk", "dv"), out):
        got = t.float().cpu().numpy()[:n, :256]
        assert np.abs(got - ref[name]).max() <= 1e-2 * np.abs(ref[name]).max(), name


@pytest.mark.parametrize("heads,window", [(2, 4096), (16, 4096), (16, 40)])
def test_negative_scale(L, heads, window):
    """a negative scale with negated queries is the same computation, dQ with the other sign.  The matrix instruction need not round a
    negated sum to the negated value, so fp32 sums may differ by their own error, 1100 * 2^-24 of the largest term (far below 2^-14 of the
    largest result), and what is stored by one bf16 step (at most 2^-7 of the value)"""
    print("case att negative scale", heads, window, flush=True)
    sp, spans = ragged_spans([700, 400], window)
    n, n_round = 1100, 1152
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    a = inputs(n, heads, seed=6)
    ds = np.random.default_rng(7).standard_normal((heads, n)).astype(np.float32) * 0.1
    x, lx = device_pass(L, n, heads, a, start, finish, 0.0, dscale=ds)
    y, ly = device_pass(L, n, heads, [-a[0]] + a[1:], start, finish, 0.0, scale=-SCALE, dscale=ds)
    assert ((lx - ly).abs() <= 2.0 ** -14 * lx.abs().max()).all()
    for name, s, t in zip(("val", "dq", "dk", "dv"), x, y):
        s, t = s.float(), -t.float() if name == "dq" else t.float()
        assert ((s - t).abs() <= 2.0 ** -7 * s.abs() + 2.0 ** -14 * s.abs().max()).all(), name


@pytest.mark.parametrize("heads", [2, 16])
def test_zero_scale_and_masked_rows(L, heads):
    """scale 0: every key that is seen weighs the same as the sink, whatever lies under the mask"""
    print("case att zero scale", heads, flush=True)
    sp, spans = ragged_spans([37, 400, 663], 333)
    n, n_round = 1100, 1152
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    a = inputs(n, heads, seed=8)
    out, swl = device_pass(L, n, heads, a, start, finish, 0.0, scale=0.0)
    count = np.where(finish[:n] >= start[:n], finish[:n] - start[:n] + 1, 0)
    np.testing.assert_allclose(swl.cpu().numpy()[0, :n], np.log2(1 + count), rtol=1e-5, atol=1e-5)
    v = np.concatenate([np.zeros((1, heads * 128)), np.cumsum(a[2].astype(np.float64), 0)])
    want = (v[np.maximum(finish[:n], -1) + 1] - v[np.where(count > 0, start[:n], finish[:n] + 1)]) / (1 + count)[:, None]
    got = out[0].float().cpu().numpy()[:n]
    assert np.abs(got - want).max() <= 2.0 ** -8 * np.abs(want).max() + 1e-3


@pytest.mark.parametrize("docs,window,heads", [([608, 1000], 4096, 2), ([608, 1000], 500, 1), ([1600], 333, 1), ([1600], 40, 1)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_values_that_no_row_of_a_wave_sees_need_not_be_finite(L, docs, window, heads, bad):
    """a value row that is not finite reaches the 32-row blocks some row of which has a key range over its block of 32 keys, and no others:
    those have the very bits they have without it.  Key ranges over and under seven tiles of 64 keys, documents that start inside a tile"""
    print("case att values not finite", docs, window, bad, flush=True)
    sp, spans = ragged_spans(docs, window)
    n = sp.size - 1
    n_round = (n + 127) // 128 * 128
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    a = inputs(n, heads, seed=11)
    clean, _ = device_pass(L, n, heads, a, start, finish, 0.0)
    lo = np.where(finish >= start, start, 1 << 30).reshape(-1, 32).min(1)
    hi = np.where(finish >= start, finish, -1).reshape(-1, 32).max(1)
    for row in (100, 544, 575, 576, 607, 608, 640, 1200, 1300, n - 1):
        b = [x.copy() for x in a]
        b[2][row] = bad
        got, _ = device_pass(L, n, heads, b, start, finish, 0.0)
        k = row // 32 * 32
        good = torch.from_numpy(np.repeat((lo > k + 31) | (hi < k), 32)).cuda()
        assert good.any() and not good.all()
        assert torch.equal(got[0][good], clean[0][good]), row


def spans_with_gaps(n):
    """one key range per row, with 32-key blocks between the ranges of neighbouring rows that none of them sees: the rest of a 64-key tile, and
    whole 128-key blocks that no query reaches at all (256..383); rows without a span"""
    start, finish, t = np.zeros(n, np.int32), np.full(n, -1, np.int32), np.arange(n) % 64
    for lo, hi, a, b in ((0, 16, 0, 10), (16, 28, 64, 95), (32, 50, 3, 40), (50, 60, 400, 450), (60, 64, 130, 131)):
        start[(t >= lo) & (t < hi)], finish[(t >= lo) & (t < hi)] = a, b
    return start, finish


@pytest.mark.parametrize("heads", [1, 32])
@pytest.mark.parametrize("f32", [False, True])
def test_handed_over_score_gradients_of_spans_with_gaps(L, heads, f32):
    """32 heads: a block of score gradients that no row sees need not be written, and must not be read.  dK and dV are the very same values with
    and without the hand-over; dQ is formed from dS rounded to bf16 in either case (2^-9 of every term, of which few dozen are added: far
    below 4e-3 of the largest).  1 head: one launch for dQ, dK and dV, which leaves the array alone"""
    print("case att gaps", heads, f32, flush=True)
    n = 512
    start, finish = spans_with_gaps(n)
    i16 = torch.int16
    q, k, v, dval = [torch.from_numpy(x).cuda().bfloat16().view(i16) for x in inputs(n, heads, seed=3)]
    ts, tf = torch.from_numpy(start).cuda(), torch.from_numpy(finish).cuda()
    val, swl = torch.zeros((n, heads * 128), dtype=i16, device="cuda"), torch.zeros((heads, n), device="cuda")
    L.att_forward(n, heads, q, k, v, ts, tf, SCALE, 0.0, val, swl)
    lo = torch.zeros(n // 128, dtype=torch.int32, device="cuda")
    hi = torch.zeros_like(lo)
    L.call("ts2_att_build_rev", n, n, ts, tf, lo, hi)
    ds = torch.from_numpy(np.random.default_rng(4).standard_normal((heads, n)).astype(np.float32) * 0.1).cuda()
    handed = L.att_ds_scratch(n, heads, ts, tf)
    handed[1].fill_(0x7f)  # NaN patterns where nothing is written
    out = []
    for pair in (None, handed):
        o = [torch.full((n, heads * 128), 3.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda") for _ in range(3)]
        L.att_backward(n, heads, q, k, v, dval, ts, tf, lo, hi, SCALE, 0.0, swl, ds, *[t if f32 else t.view(i16) for t in o], L.F32 if f32 else L.BF16,
                       ds=pair)
        out.append(o)
    torch.cuda.synchronize()
    assert torch.equal(out[0][1], out[1][1]) and torch.equal(out[0][2], out[1][2])
    if heads == 1:
        assert torch.equal(out[0][0], out[1][0]) and (handed[1] == 0x7f).all()
    a, b = out[0][0].float(), out[1][0].float()
    assert (a - b).abs().max() <= 4e-3 * a.abs().max()


@pytest.mark.parametrize("docs,window", [([300, 1, 299, 500], 40), ([1100], 4096)])
def test_gradients_in_place_of_keys_and_values(L, docs, window):
    """dK over K and dV over V: a workgroup reads the rows it writes, and dQ, which reads them all, is done before.  The very bits of the calls
    for one gradient each, which run the same kernels.  Column ranges of one wide matrix are no such case: the same bits as separate
    matrices, and as the call with both bits in one launch"""
    print("case att in place", docs, window, flush=True)
    sp, spans = ragged_spans(docs, window)
    n, n_round, heads, w, i16 = sp.size - 1, (sp.size + 126) // 128 * 128, 2, 256, torch.int16
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    ts, tf = torch.from_numpy(start).cuda(), torch.from_numpy(finish).cuda()

    def padded(a):
        t = torch.zeros((n_round, w), dtype=torch.bfloat16, device="cuda")
        t[:n] = torch.from_numpy(a).cuda().bfloat16()
        return t.view(i16)
    q, k, v, dval = [padded(a) for a in inputs(n, heads, seed=13)]
    val, swl = torch.zeros_like(q), torch.zeros((heads, n_round), device="cuda")
    L.att_forward(n, heads, q, k, v, ts, tf, SCALE, 0.0, val, swl)
    lo = torch.zeros(n_round // 128, dtype=torch.int32, device="cuda")
    hi = torch.zeros_like(lo)
    L.call("ts2_att_build_rev", n, n_round, ts, tf, lo, hi)
    ds = torch.from_numpy(np.random.default_rng(4).standard_normal((heads, n_round)).astype(np.float32) * 0.1).cuda()

    def back(k, v, out, which):
        L.att_backward(n, heads, q, k, v, dval, ts, tf, lo, hi, SCALE, 0.0, swl, ds, *out, L.BF16, which=which)
    apart, both = [[torch.full_like(q, 7) for _ in range(3)] for _ in range(2)]
    back(k, v, apart, 1)
    back(k, v, apart, 2)
    back(k, v, both, 3)
    wide = torch.full((n_round, 5 * w), 7, dtype=i16, device="cuda")
    parts = [wide[:, i * w:(i + 1) * w] for i in range(5)]  # dQ, K, dK, V, dV side by side
    parts[1].copy_(k)
    parts[3].copy_(v)
    back(parts[1], parts[3], [parts[0], parts[2], parts[4]], 3)
    k2, v2, dq = k.clone(), v.clone(), torch.full_like(q, 7)
    back(k2, v2, [dq, k2, v2], 3)
    torch.cuda.synchronize()
    for name, a, b in zip(("dq", "dk", "dv"), apart, (dq, k2, v2)):
        assert torch.equal(a, b), name
    for name, a, b, c in zip(("dq", "dk", "dv"), both, (parts[0], parts[2], parts[4]), apart):
        assert torch.equal(a, b), name
        # one launch adds a gradient in two halves: fp32 sums of at most 1100 terms in another order, then one bf16 step
        x, y = a.view(torch.bfloat16).float(), c.view(torch.bfloat16).float()
        assert ((x - y).abs() <= 2.0 ** -7 * y.abs() + 2.0 ** -14 * y.abs().max()).all(), name


@pytest.mark.parametrize("docs,window", [([300, 1, 299, 500], 40), ([1100], 4096)])
@pytest.mark.parametrize("place", ["q", "v", "dval"])
def test_dq_in_place_with_handed_over_score_gradients(L, docs, window, place):
    """dQ formed from the handed-over score gradients reads K and them alone, so it may take the place of Q, V or the incoming gradient, which
    the launch before it has read.  dK and dV are the very bits of a call for them alone; dQ is formed from dS rounded to bf16 either way (2^-9 of
    every term, with signs either way: far below 4e-3 of the largest)"""
    print("case att dq in place", docs, window, place, flush=True)
    sp, spans = ragged_spans(docs, window)
    n, n_round, heads, w, i16 = sp.size - 1, (sp.size + 126) // 128 * 128, 2, 256, torch.int16
    start, finish = spans_to_ranges(sp, spans, n, n_round)
    ts, tf = torch.from_numpy(start).cuda(), torch.from_numpy(finish).cuda()

    def padded(a):
        t = torch.zeros((n_round, w), dtype=torch.bfloat16, device="cuda")
        t[:n] = torch.from_numpy(a).cuda().bfloat16()
        return t.view(i16)
    t = dict(zip(("q", "k", "v", "dval"), [padded(a) for a in inputs(n, heads, seed=17)]))
    val, swl = torch.zeros_like(t["q"]), torch.zeros((heads, n_round), device="cuda")
    L.att_forward(n, heads, t["q"], t["k"], t["v"], ts, tf, SCALE, 0.0, val, swl)
    lo = torch.zeros(n_round // 128, dtype=torch.int32, device="cuda")
    hi = torch.zeros_like(lo)
    L.call("ts2_att_build_rev", n, n_round, ts, tf, lo, hi)
    ds = torch.from_numpy(np.random.default_rng(4).standard_normal((heads, n_round)).astype(np.float32) * 0.1).cuda()

    def back(t, out, which, pair=None):
        L.att_backward(n, heads, t["q"], t["k"], t["v"], t["dval"], ts, tf, lo, hi, SCALE, 0.0, swl, ds, *out, L.BF16, which=which, ds=pair)
    apart = [torch.full_like(val, 7) for _ in range(3)]
    back(t, apart, 1)
    back(t, apart, 2)
    copy = {k: x.clone() for k, x in t.items()}
    out = [copy[place], torch.full_like(val, 7), torch.full_like(val, 7)]
    back(copy, out, 3, L.att_ds_scratch(n_round, heads, ts, tf))
    torch.cuda.synchronize()
    assert torch.equal(out[1], apart[1]) and torch.equal(out[2], apart[2])
    x, y = out[0].view(torch.bfloat16).float(), apart[0].view(torch.bfloat16).float()
    assert (x - y).abs().max() <= 4e-3 * y.abs().max()
