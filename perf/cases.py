"""What the performance of this framework is measured on: the calls a training program makes, through the public entry points of
tscale2_amd.lib, over the sizes the repository's own configurations, tests and benchmark use.

Five kinds of case:
  step       ts2_model_backprop of a whole model on one batch: forward, loss gradient, backward through every layer, every packed delta.
             "then" = "apply" adds what a training loop does next: the optimiser update of every matrix, and the forward pass with the
             new weights that gives the loss after it (the probabilities depend on every delta of the step).
  forward    ts2_model_forward: probabilities of every token of a batch (evaluation, the prompt pass of a server).
  linear     one linear layer through its operators (TMatMulBuffers): forward, dX and the packed delta.
  attention  the inside of an attention layer through its operators: attention forward, gate, gate backward, dQ / dK / dV.
  optimizer  the update of one layer's matrices from their packed deltas.

Every model keeps its weights on the device; a batch is uploaded once (ts2_model_set_batch) before the pass, as a data loader does."""
import ctypes as C
import math

import numpy as np
import torch

from tscale2_amd import lib as L

ATT_DOT_SCALE = math.sqrt(1 / 128) * 0.5 / 0.693147  # what the model driver passes to its attention layers


def listed():
    def step(name, mode, dim, heads, ffn, depth, vocab, docs, doc_len, wide, experts=0, expert_dim=0, then="", kind="step"):
        return {"name": name, "kind": kind, "mode": mode, "dim": dim, "heads": heads, "ffn": ffn, "depth": depth, "vocab": vocab, "docs": docs,
                "doc_len": doc_len, "wide": wide, "experts": experts, "expert_dim": expert_dim, "then": then}

    def linear(name, mode, rows, src, grad, splits):
        return {"name": name, "kind": "linear", "mode": mode, "rows": rows, "src": src, "grad": grad, "splits": splits}

    def attention(name, heads, docs, doc_len, width, ragged):
        return {"name": name, "kind": "attention", "heads": heads, "docs": docs, "doc_len": doc_len, "width": width, "ragged": ragged}

    return [
        # the smallest model of the test-suite's configurations: 8 sequences of 64 bytes, where launches and latency are what is left
        step("step_tiny_i8", "i8", 256, 2, 1024, 4, 256, 8, 64, 64),
        # a small fp8 model trained for real: step, optimiser update, loss after the update (the benchmark's reduced model)
        step("train_small_fp8", "e4m3", 512, 4, 2048, 4, 1024, 8, 512, 512, then="apply"),
        # e512 d8 h3 ffn4 on 8 x 2048 tokens in int8: the reference's published single-GPU training run
        step("step_e512_i8", "i8", 512, 3, 512, 8, 1024, 8, 2048, 2048),
        # the headline model: e2048 h16 d12 ffn64 w1024, vocabulary 50304, 32 x 1024 tokens
        step("step_e2048_fp8", "e4m3", 2048, 16, 8192, 12, 50304, 32, 1024, 1024),
        # mixture of experts, 8 experts of width 256, on a batch that fills no tile: 5 documents of 777 tokens
        step("step_moe8_ragged_fp8", "e4m3", 512, 4, 1024, 4, 1024, 5, 777, 512, experts=8, expert_dim=256),
        # one mixture-of-experts layer at full width: 64 experts of width 512, 65536 tokens (depth 0: the layer alone, between embedding and head)
        step("layer_moe64_fp8", "e4m3", 1024, 8, 1024, 0, 128, 32, 2048, 128, experts=64, expert_dim=512),
        # probabilities for one prompt of 777 tokens, vocabulary 50304
        step("forward_prompt_fp8", "e4m3", 1024, 8, 4096, 6, 50304, 1, 777, 1024, kind="forward"),
        # the int8 linear layer of the benchmark: X [16384 x 1024], dY [16384 x 4096]
        linear("linear_i8", "i8", 16384, 1024, 4096, 2),
        # a linear layer on a batch that ends inside a row tile
        linear("linear_ragged_fp8", "e4m3", 3000, 512, 1536, 1),
        # full causal attention, 16 x 2048 tokens, 16 heads
        attention("attention_causal", 16, 16, 2048, 2048, False),
        # the 64-token window most attention layers of a model have, over documents of unequal length
        attention("attention_window_ragged", 4, 24, 700, 64, True),
        # the update of a feed-forward layer's three 8192 x 2048 matrices
        {"name": "optimizer_ffn_fp8", "kind": "optimizer", "mode": "e4m3", "rows": 8192, "cols": 2048, "count": 3},
    ]


def _log(rng, lo, hi, multiple=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple)) * multiple))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "forward", "linear", "linear", "attention", "attention", "optimizer"])
    mode = rng.choice(["i8", "e4m3"])
    if kind in ("step", "forward"):
        experts = rng.choice([0, 0, 8, 16, 64]) if kind == "step" else 0
        if experts:
            mode = "e4m3"
        dim = _log(rng, 256, 1024, 128)
        tokens = _log(rng, 256, 16384)
        doc_len = min(tokens, _log(rng, 32, 2048))
        vocab = _log(rng, 256, 16384, 128)
        return {"kind": kind, "mode": mode, "dim": dim, "heads": _log(rng, 1, 8), "ffn": _log(rng, 256, 4096, 128), "depth": rng.choice([2, 3, 4, 6]) if not experts else 4,
                "vocab": vocab, "docs": max(1, tokens // doc_len), "doc_len": doc_len, "wide": _log(rng, 64, 2048), "experts": experts,
                "expert_dim": _log(rng, 128, 512, 128) if experts else 0, "then": rng.choice(["", "", "apply"]) if kind == "step" else ""}
    if kind == "linear":
        rows = _log(rng, 128, 32768)
        return {"kind": kind, "mode": mode, "rows": rows, "src": _log(rng, 256, 4096, 128), "grad": _log(rng, 256, 8192, 128), "splits": 1}
    if kind == "attention":
        tokens, heads = _log(rng, 256, 32768), _log(rng, 1, 16)
        doc_len = min(tokens, _log(rng, 64, 2048))
        return {"kind": kind, "heads": heads, "docs": max(1, tokens // doc_len), "doc_len": doc_len,
                "width": rng.choice([1, 64, doc_len, _log(rng, 64, 2048)]), "ragged": rng.choice([True, False])}
    return {"kind": kind, "mode": mode, "rows": _log(rng, 128, 8192, 1), "cols": _log(rng, 256, 4096, 128), "count": rng.randint(1, 4)}


# ---------------------------------------------------------------------------------------------------------------------------------------
# models

def _schedule(case):
    if case["depth"] == 0:  # the mixture-of-experts layer alone
        return np.array([3], np.int32), np.zeros(1, np.int32), np.zeros(1, np.float32), np.array([1], np.int32)
    return L.model_schedule(case["depth"], case["experts"], case["wide"])


def _labels(case):
    # the layer alone gets a state of its own for every token; a model one embedding row per vocabulary entry
    return case["docs"] * case["doc_len"] + 1 if case["depth"] == 0 else case["vocab"] + 1


def _matrices(case):
    """(layer, index, rows, cols) of every matrix of the model"""
    lt = _schedule(case)[0]
    out = [(d, i, r, c) for d in range(len(lt))
           for i, (r, c) in enumerate(L.layer_shapes(int(lt[d]), case["dim"], case["heads"], case["ffn"], case["expert_dim"], case["experts"]))]
    return out + [(L.LAYER_EMBED, 0, _labels(case), case["dim"]), (L.LAYER_FINAL, 0, case["vocab"], case["dim"])]


def _spans(n, doc_start, width):
    t = np.arange(n, dtype=np.int32)
    start = np.maximum(doc_start, t - width).astype(np.int32)
    return start, np.where(t == doc_start, -1, t - 1).astype(np.int32)


class _View:
    """array interface of a tensor in a model's own memory that keeps the model: results stay readable when the handle is dropped"""

    def __init__(self, owner, tensor):
        self.owner, self.__cuda_array_interface__ = owner, tensor.__cuda_array_interface__


class _ModelState:
    """a program's model handle: the device memory goes back when the program drops it and every result that lies in it"""

    def __init__(self, case, seed):
        L.load()
        lt, la, ls, widths = _schedule(case)
        n, vocab = case["docs"] * case["doc_len"], case["vocab"]
        gen = torch.Generator(device="cuda").manual_seed(seed)
        moe = case["experts"] > 0
        self.case = case
        self.model = m = L.Model(L.I8 if case["mode"] == "i8" else L.E4M3, case["dim"], case["heads"], case["ffn"], lt, la, ls, len(widths), vocab,
                                 _labels(case), n, case["expert_dim"] if moe else 0, case["experts"], 2 if moe else 0)
        for layer, i, rows, cols in _matrices(case):
            w = torch.randn((rows, cols), device="cuda", generator=gen)
            # as in a model that has learnt something, the residual stream is large beside what one layer adds to it
            std = 0.2 if layer == L.LAYER_EMBED else 0.02
            if case["then"] == "apply":
                m.set_master(layer, i, (w * std).cpu().numpy(), rows)  # fp32 master weights; the driver derives the 8-bit ones
            elif case["mode"] == "i8":
                m.set_matrix(layer, i, torch.clamp(torch.round(w * 32), -128, 127).to(torch.int8).cpu().numpy(), std)
            else:
                m.set_matrix(layer, i, (w * 32).to(torch.float8_e4m3fn).view(torch.uint8).cpu().numpy(), std)
        r = np.random.default_rng(seed)
        m.set_bias((r.standard_normal(vocab) * 0.1).astype(np.float32))
        tokens = r.integers(0, vocab, (case["docs"], case["doc_len"]))
        target = np.full(tokens.shape, -1, np.int32)
        target[:, :-1] = tokens[:, 1:]
        labels = np.arange(n) if case["depth"] == 0 else tokens.ravel()
        t = np.arange(n, dtype=np.int32)
        spans = [_spans(n, t // case["doc_len"] * case["doc_len"], int(w)) for w in widths]
        m.set_batch(np.arange(n + 1, dtype=np.int32), (1 + labels).astype(np.uint32), target.ravel(), [s[0] for s in spans], [s[1] for s in spans],
                    L.fill_rope_buf(128, n))
        self.n = n

    def __del__(self):
        if getattr(self, "model", None) is not None:
            self.model.close()

    def array(self, name, cols):
        t = self.model.array(name)[:self.n, :cols]
        if t.dtype != torch.bfloat16:
            return torch.as_tensor(_View(self, t), device="cuda")
        return torch.as_tensor(_View(self, t.view(torch.int16)), device="cuda").view(torch.bfloat16)

    def run(self):
        m, case, dim, vocab = self.model, self.case, self.case["dim"], self.case["vocab"]
        if case["kind"] == "forward":
            m.forward()
            return {"state": self.array("state", dim), "prediction": self.array("prediction", vocab)}
        m.backprop()
        out = {"stateGrad": self.array("stateGrad", dim), "finalGrad": self.array("finalGrad", vocab)}
        if case["then"] == "apply":
            m.apply_deltas(0.002, l2_reg=1.0, beta1=0.9, weight0=1.0, weight1=0.5, disp_decay=0.9)
            m.forward()
            out["prediction"] = self.array("prediction", vocab)
        out["state"] = self.array("state", dim)
        return out


# ---------------------------------------------------------------------------------------------------------------------------------------
# operators

class _LinearState:
    def __init__(self, case, seed):
        L.load()
        g = torch.Generator(device="cuda").manual_seed(seed)
        n, src, grad = case["rows"], case["src"], case["grad"]
        self.case, self.mode = case, L.I8 if case["mode"] == "i8" else L.E4M3
        rounded = -(-n // 512) * 512
        x = torch.randn((n, src), device="cuda", generator=g)
        w = torch.randn((grad, src), device="cuda", generator=g)
        # gradients have rows and channels of very different size
        dy = torch.randn((n, grad), device="cuda", generator=g) * torch.exp(torch.randn((n, 1), device="cuda", generator=g) * 0.5)
        dt = torch.int8 if self.mode == L.I8 else torch.uint8

        def rows(t):  # rows of a batch end on a tile boundary; the pad rows hold zeros
            full = torch.zeros((rounded, t.shape[1]), dtype=t.dtype, device="cuda")
            full[:n] = t
            return full
        self.bufs = L.MatMulBuffers(self.mode, rounded, src, grad, k_tile=512, splits=case["splits"], share_row_max=self.mode == L.I8)
        self.scale = torch.full((1,), 0.02, device="cuda")
        if self.mode == L.I8:
            # X with per-row, W with per-channel abs-max scales; the gradient arrives in bf16
            self.x_scale = torch.zeros(rounded, device="cuda")
            self.x_scale[:n] = x.abs().amax(1) / 127
            self.x8 = rows(torch.round(x / self.x_scale[:n, None]).to(dt))
            self.w_scale = w.abs().amax(1) / 127 * 0.02
            self.w8 = torch.round(w / w.abs().amax(1, keepdim=True) * 127).to(dt)
            self.dy, self.dy_type = rows(dy.bfloat16().view(torch.int16)), L.BF16
        else:
            self.x_scale = self.w_scale = None
            self.x8 = rows((x * 24).to(torch.float8_e4m3fn).view(dt))
            self.w8 = (w * 32).to(torch.float8_e4m3fn).view(dt)
            self.dy, self.dy_type = rows((dy * 16).clamp(-448, 448).to(torch.float8_e4m3fn).view(dt)), L.E4M3
        self.y = torch.zeros((rounded, grad), dtype=torch.int16, device="cuda")
        self.dx = torch.zeros((rounded, src), device="cuda")

    def run(self):
        c, b = self.case, self.bufs
        n = c["rows"]
        L.call("ts2_matmul_forward", self.mode, n, b.len_round, c["src"], c["grad"], self.x8, self.w8, 1 / 768, self.scale, self.y, L.BF16, 0)
        b.backprop_multi(n, self.w8, self.dy, self.dy_type, self.w_scale)
        b.backprop(n, None if self.mode == L.I8 else self.dy, 1.0, None if self.mode == L.I8 else self.scale, self.dx, L.F32)
        b.backprop_delta(n, self.x8, self.x_scale, self.dy, self.dy_type)
        return {"y": self.y.view(torch.bfloat16)[:n], "dx": self.dx[:n], "delta": b.delta, "deltaTileScale": b.delta_tile_scale}


class _AttentionState:
    def __init__(self, case, seed):
        L.load()
        g = torch.Generator(device="cuda").manual_seed(seed)
        r = np.random.default_rng(seed)
        docs, doc_len, heads = case["docs"], case["doc_len"], case["heads"]
        if case["ragged"]:
            cuts = np.sort(r.choice(np.arange(1, docs * doc_len), docs - 1, replace=False)) if docs > 1 else np.zeros(0, int)
            first = np.concatenate([[0], cuts]).astype(np.int32)
        else:
            first = (np.arange(docs) * doc_len).astype(np.int32)
        n = docs * doc_len
        rounded, width = -(-n // 128) * 128, heads * 128
        doc_start = np.zeros(n, np.int32)
        doc_start[first] = first
        s, f = _spans(n, np.maximum.accumulate(doc_start), case["width"])
        pad = rounded - n
        self.start = torch.from_numpy(np.concatenate([s, np.zeros(pad, np.int32)])).cuda()
        self.finish = torch.from_numpy(np.concatenate([f, np.full(pad, -1, np.int32)])).cuda()
        self.case, self.n, self.rounded = case, n, rounded

        def rows():
            t = torch.randn((rounded, width), device="cuda", generator=g)
            t[n:] = 0
            return t.bfloat16().view(torch.int16)
        self.q, self.k, self.v, self.gate, self.dvlg = rows(), rows(), rows(), rows(), rows()
        new = lambda dt: torch.zeros((rounded, width), dtype=dt, device="cuda")  # noqa: E731
        self.val, self.dval, self.dq, self.dk, self.dv = [new(torch.int16) for _ in range(5)]
        self.vlg, self.dgate = new(torch.uint8), new(torch.uint8)
        self.swl, self.dscale = torch.zeros((heads, rounded), device="cuda"), torch.zeros((heads, rounded), device="cuda")
        self.rev_lo = torch.zeros(rounded // 128, dtype=torch.int32, device="cuda")
        self.rev_hi = torch.zeros_like(self.rev_lo)
        # (once per batch, for all layers)
        L.call("ts2_att_build_rev", n, rounded, self.start, self.finish, self.rev_lo, self.rev_hi)

    def run(self):
        n, r, h = self.n, self.rounded, self.case["heads"]
        L.att_forward(n, h, self.q, self.k, self.v, self.start, self.finish, ATT_DOT_SCALE, 0.0, self.val, self.swl)
        L.call("ts2_matrix_lolu", n, r, self.gate, self.val, 24.0, self.vlg, L.E4M3)
        L.call("ts2_backprop_lolu_dscale", n, r, self.gate, self.val, 1.0, self.dvlg, L.BF16, self.dgate, L.E4M3, self.dval, L.BF16, self.dscale)
        L.att_backward(n, h, self.q, self.k, self.v, self.dval, self.start, self.finish, self.rev_lo, self.rev_hi, ATT_DOT_SCALE, 0.0, self.swl,
                       self.dscale, self.dq, self.dk, self.dv, L.BF16)
        out = {k: getattr(self, k).view(torch.bfloat16)[:n] for k in ("val", "dq", "dk", "dv")}
        out["vlg"], out["dgate"] = [t.view(torch.float8_e4m3fn)[:n] for t in (self.vlg, self.dgate)]
        out["swl"], out["dscale"] = self.swl[:, :n], self.dscale[:, :n]
        return out


class _OptMatrix(C.Structure):
    _fields_ = [("xSize", C.c_int32), ("ySize", C.c_int32), ("yBufSize", C.c_int32), ("rowDispSize", C.c_int32), ("weights", L.Mat), ("avgGrad", L.Mat),
                ("grad", L.Mat), ("gradRowSum2", C.c_void_p), ("weightsRowSum2", C.c_void_p), ("rowScale", C.c_void_p), ("rowDisp", C.c_void_p),
                ("sumWeight", C.c_void_p), ("sparsity", C.c_void_p), ("fast", L.Mat), ("fastType", C.c_int32), ("matrixScale", C.c_void_p),
                ("convertMult", C.c_void_p)]


class _OptimizerState:
    def __init__(self, case, seed):
        L.load()
        g = torch.Generator(device="cuda").manual_seed(seed)
        rows, cols = case["rows"], case["cols"]
        padded = -(-rows // 128) * 128
        self.params = torch.tensor([0.9, 0.9, 1.0, 0.5, 1.0, 0.002], device="cuda")  # dispDecay, beta1, weight0, weight1, l2Reg, stepMult
        self.layers = []
        for _ in range(case["count"]):
            z = lambda *s: torch.zeros(s, device="cuda")  # noqa: E731
            t = {"weights": torch.randn((rows, cols), device="cuda", generator=g) * 0.02, "avgGrad": z(rows, cols), "gradRowSum2": z(rows),
                 "weightsRowSum2": z(rows), "rowScale": z(rows), "rowDisp": z(rows), "sumWeight": z(1), "sparsity": torch.ones(1, device="cuda"),
                 "fast": torch.zeros((padded, cols), dtype=torch.int8 if case["mode"] == "i8" else torch.uint8, device="cuda"), "matrixScale": z(1),
                 "convertMult": z(1)}
            delta = torch.clamp(torch.randn((rows, cols), device="cuda", generator=g) * 40, -127, 127).to(torch.int8)
            tile_scale = torch.exp(torch.randn((cols // 128, rows), device="cuda", generator=g)) * 1e-4
            o = _OptMatrix(xSize=cols, ySize=rows, yBufSize=padded, rowDispSize=rows, fastType=L.I8 if case["mode"] == "i8" else L.E4M3)
            for k in ("weights", "avgGrad", "fast"):
                setattr(o, k, L.mat(t[k]))
            for k in ("gradRowSum2", "weightsRowSum2", "rowScale", "rowDisp", "sumWeight", "sparsity", "matrixScale", "convertMult"):
                setattr(o, k, t[k].data_ptr())
            self.layers.append((o, t, delta, tile_scale))

    def run(self):
        out = []
        for o, t, delta, tile_scale in self.layers:
            L.call("ts2_opt_add_delta", C.byref(o), delta, tile_scale, 2, self.params)  # 2: apply at once
            out.append({k: t[k] for k in ("weights", "avgGrad", "rowDisp", "matrixScale", "fast")})
        return out


KINDS = {"step": _ModelState, "forward": _ModelState, "linear": _LinearState, "attention": _AttentionState, "optimizer": _OptimizerState}


def prepare(case, seed):
    return KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------------------------------------------------------------------------------
# work and tolerances

def work(case):
    """Weights, labels and spans read once, results written once; matrix products and the causal part of the attention, nothing else."""
    if case["kind"] in ("step", "forward"):
        n, dim, vocab = case["docs"] * case["doc_len"], case["dim"], case["vocab"]
        lt, la, _, widths = _schedule(case)
        stored = sum(r * c for layer, _, r, c in _matrices(case) if layer != L.LAYER_EMBED)
        active = stored
        if case["experts"]:  # two of the experts' slabs per token
            slabs = sum(r * c for layer, i, r, c in _matrices(case) if layer >= 0 and lt[layer] == 3 and i < 3)
            active += slabs * 2 // case["experts"] - slabs
        pairs = [case["docs"] * sum(min(i, int(w)) for i in range(case["doc_len"])) for w in widths]
        att = sum(pairs[la[d]] for d in range(len(lt)) if lt[d] == 0) * 128 * case["heads"]
        forward = {"bytes": stored + n * (2 * dim + 4 * dim + 4 * vocab), "flops": 2 * active * n + 4 * att}
        if case["kind"] == "forward":
            return forward
        # weights read, packed deltas written, embedding rows read and their fp32 gradient written, state, state gradient, logit gradient
        w = {"bytes": 2 * stored + _labels(case) * dim * 4 + n * (dim + 8 * dim + 2 * vocab), "flops": 6 * active * n + 14 * att}
        if case["then"] == "apply":
            total = stored + _labels(case) * dim
            w["bytes"] += 18 * total + forward["bytes"]  # delta, weights and average read, weights, average and fast weights written
            w["flops"] += forward["flops"]
        return w
    if case["kind"] == "linear":
        n, src, grad = case["rows"], case["src"], case["grad"]
        dy = 2 if case["mode"] == "i8" else 1
        return {"bytes": n * src * 5 + n * grad * (dy + 2) + src * grad * 2, "flops": 6 * n * src * grad}
    if case["kind"] == "attention":
        n, width = case["docs"] * case["doc_len"], case["heads"] * 128
        pairs = case["docs"] * sum(min(i, case["width"]) for i in range(case["doc_len"]))
        return {"bytes": n * width * (5 * 2 + 4 * 2 + 2) + n * case["heads"] * 8, "flops": 14 * pairs * width}
    return {"bytes": case["count"] * case["rows"] * case["cols"] * 18, "flops": 0}


def tolerance(case):
    """About four times what was measured.  Models: their own results when half the entries of the rotation table move by one unit in the
    last place - an 8-bit rounding that falls the other way is passed on by every later layer, so state and state gradient differ by 0.001
    to 0.004 (8 layers) and 0.0085 (24 layers, fp8), single elements by up to 0.13.  Linear layers against fp64: bf16 results 0.0017, fp32
    ones 1.5e-5, which moves one packed 8-bit value in a thousand by one.  Attention against fp64: 0.0025 in bf16, single elements 0.045;
    the e4m3 results round that to steps of 0.06 to 0.12.  Optimiser: fp32 sums over a row."""
    if case["kind"] == "optimizer":
        return {"rel": 1e-5, "differ": 1e-3}
    if case["kind"] == "linear":
        return {"rel": 7e-3, "max": 0.02, "differ": 4e-3}
    if case["kind"] == "attention":
        return {"rel": 2e-2, "max": 0.25}
    return {"rel": 0.03 if case["depth"] >= 12 else 0.016, "max": 0.5}
