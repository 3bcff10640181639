"""The workloads whose speed is measured: calls through nlgpu, the Python
binding of libnlgpu, at the sizes of this repository's configurations, tests
and benchmark and over the ranges around them.

Two ways of use are covered.  A program that serves a quantised model calls
the typed entry points (linears on 2-bit weights, fp16-cache attention, the
decoder stack).  The Lisp driver composes its models from kernels by name on
the reference's f32 layouts (f32 products, attention, ternary linears and
their input gradients).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nelisp-gpu_amd"))
import nlgpu  # noqa: E402

DEV = "cuda:0"


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # One projection of one decoded token: the 4096 x 4096 GEMV with its
        # activation quantisation in the same launch.
        {"name": "linear_token", "kind": "linear", "tokens": 1, "out": 4096, "cols": 4096},
        # The SwiGLU block of the 2B-class model over a 512-token prompt.
        {"name": "ffn_prompt", "kind": "ffn", "tokens": 512, "d_model": 2560, "d_ff": 6912},
        # Attention of one decode step, eight sequences well into their contexts.
        {"name": "attn_decode", "kind": "attn_decode", "batch": 8, "heads": 32, "kvheads": 8, "head_dim": 128,
         "pos": 4095, "max_seq": 8192},
        # Attention of one long prompt with the 2B-class model's heads.
        {"name": "attn_prompt", "kind": "attn_prompt", "prompts": 1, "qper": 2048, "pos0": 0, "heads": 20,
         "kvheads": 5, "head_dim": 128},
        # A serving step over paged caches: sequences of very different lengths.
        {"name": "attn_paged", "kind": "attn_paged", "batch": 32, "heads": 20, "kvheads": 5, "head_dim": 128,
         "bs": 16, "longest": 4096},
        # Row softmax of 32 heads' causal 4096 x 4096 scores.
        {"name": "softmax_scores", "kind": "softmax", "rows": 131072, "cols": 4096},
        # A whole decoder (two layers of the 2B-class model and its head), one
        # sequence, token by token (graph replay).
        {"name": "stack_tokens", "kind": "stack", "mode": "steps", "batch": 1, "tokens": 32},
        # By name: an f32 matrix product (the matmul bench host's).
        {"name": "matmul_f32", "kind": "matmul", "kernel": "matmul", "m": 1024, "k": 1024, "n": 1024},
        # By name: causal attention of a prompt on f32 tensors.
        {"name": "attn_prompt_f32", "kind": "gqa", "seq": 1024, "heads": 20, "kvheads": 5, "head_dim": 128},
        # By name: one decode step's attention on f32 caches.
        {"name": "attn_decode_f32", "kind": "decode_f32", "batch": 4, "heads": 20, "kvheads": 5, "head_dim": 128,
         "pos": 2047, "max_seq": 4096},
        # By name: a ternary linear on f32 activations (forward).
        {"name": "ternary_f32", "kind": "ternary", "seq": 64, "out": 6912, "cols": 2560},
        # By name: its input gradient (backward).
        {"name": "ternary_grad_f32", "kind": "ternary_grad", "seq": 64, "out": 2560, "cols": 6912},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "ffn", "attn_decode", "attn_prompt", "attn_paged", "softmax", "stack", "matmul",
                       "gqa", "decode_f32", "ternary", "ternary_grad"])
    heads = rng.choice([(20, 5), (32, 8), (16, 16), (16, 8), (32, 4), (8, 2)])
    hd = rng.choice([64, 128, 128])
    if kind == "linear":
        return {"kind": kind, "tokens": _log(rng, 1, 1024), "out": _log(rng, 512, 14336),
                "cols": 64 * _log(rng, 8, 172)}
    if kind == "ffn":
        return {"kind": kind, "tokens": _log(rng, 1, 2048), "d_model": 256 * rng.randint(4, 16),
                "d_ff": 256 * rng.randint(10, 43)}
    if kind == "attn_decode":
        batch = _log(rng, 1, 64)
        pos = min(_log(rng, 64, 16384), (1 << 18) // (batch * heads[1]) + 64) - rng.randint(0, 16)
        return {"kind": kind, "batch": batch, "heads": heads[0], "kvheads": heads[1], "head_dim": hd, "pos": pos,
                "max_seq": pos + 1 + rng.randint(0, pos)}
    if kind == "attn_prompt":
        qper = _log(rng, 32, 2048)
        prompts = max(1, min(_log(rng, 1, 32), 4096 // qper))
        return {"kind": kind, "prompts": prompts, "qper": qper, "pos0": rng.choice([0, 0, 0, 256, 1000]),
                "heads": heads[0], "kvheads": heads[1], "head_dim": hd}
    if kind == "attn_paged":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "batch": batch, "heads": heads[0], "kvheads": heads[1], "head_dim": hd,
                "bs": rng.choice([16, 16, 32, 64]),
                "longest": min(_log(rng, 64, 8192), (1 << 19) // (batch * heads[1]) + 64)}
    if kind == "softmax":
        cols = _log(rng, 32, 32768)
        return {"kind": kind, "rows": max(64, min(_log(rng, 64, 131072), (1 << 28) // cols)), "cols": cols}
    if kind == "stack":
        mode = rng.choice(["steps", "prompt"])
        return {"kind": kind, "mode": mode, "batch": rng.choice([1, 2, 4, 8]),
                "tokens": rng.randint(8, 32) if mode == "steps" else _log(rng, 16, 640)}
    if kind == "matmul":
        kernel = rng.choice(["matmul", "matmul", "matmul-tiled", "matmul-reg", "linear"])
        m, k, n = (_log(rng, 24, 2048) for _ in range(3))
        if kernel == "matmul-reg":
            m, n = m // 4 * 4, n // 4 * 4
        return {"kind": kind, "kernel": kernel, "m": m, "k": k, "n": n}
    if kind == "gqa":
        return {"kind": kind, "seq": _log(rng, 16, 1024), "heads": heads[0], "kvheads": heads[1],
                "head_dim": rng.choice([64, 80, 96, 128])}
    if kind == "decode_f32":
        batch = _log(rng, 1, 16)
        pos = min(_log(rng, 32, 8192), (1 << 17) // (batch * heads[1]) + 32) - rng.randint(0, 16)
        return {"kind": kind, "batch": batch, "heads": heads[0], "kvheads": heads[1], "head_dim": hd, "pos": pos,
                "max_seq": pos + 1 + rng.randint(0, pos)}
    return {"kind": kind, "seq": _log(rng, 1, 256), "out": _log(rng, 512, 6912), "cols": 4 * _log(rng, 128, 1728)}


# ------------------------------------------------------------------ the inputs

class View:
    """A torch tensor as the binding takes buffers (its pointer and length)."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr = self.t.data_ptr()
        self.nbytes = self.t.numel() * self.t.element_size()

    def as_buffer(self, nfloats=None):
        return nlgpu.Buffer(self.ptr, self.nbytes // 4 if nfloats is None else int(nfloats))


class Inputs:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        nlgpu.init()
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 1)

    def normal(self, *shape, sigma=1.0):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32) * sigma

    def half(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32).half()

    def uniform(self, n, lo, hi):
        return torch.rand(n, generator=self.g, device=DEV, dtype=torch.float32) * (hi - lo) + lo

    def ints(self, n, lo, hi):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV, dtype=torch.int32)

    def trits(self, out, cols):
        """{-1, 0, +1} with probabilities 1/4, 1/2, 1/4, int8 [out, cols]."""
        r = torch.randint(0, 4, (out, cols), generator=self.g, device=DEV, dtype=torch.int8)
        return (r == 2).to(torch.int8) - (r == 3).to(torch.int8)


def pack_words(t):
    """The 2-bit words [out, ceil(cols/16)] (int32 bits) of trits [out, cols]."""
    out, cols = t.shape
    wng = (cols + 15) // 16
    if cols % 16:
        t = torch.nn.functional.pad(t, (0, wng * 16 - cols))
    codes = (t.to(torch.int32) & 3).view(out, wng, 16)
    words = torch.zeros(out, wng, dtype=torch.int32, device=t.device)
    for f in range(16):
        words |= codes[:, :, f] << (2 * f)
    return words


def weights(t, tiled):
    """2-bit weights as a model loader leaves them: in library memory, with
    the matrix-core copy where the batched linears will read them."""
    w = pack_words(t)
    d = nlgpu.DeviceArray(w.numel() * 4)
    nlgpu._check(nlgpu.lib().nlg_copy_d2d(d.ptr, w.data_ptr(), d.nbytes, None), "copy")
    nlgpu.sync()
    if tiled:
        nlgpu.ternary_tiled_register(d, t.shape[0], t.shape[1])
    return d


def _empty(*shape):
    return torch.zeros(shape, device=DEV, dtype=torch.float32)


def _linear_inputs(c, i):
    return {"t": i.trits(c["out"], c["cols"]), "x": i.normal(c["tokens"], c["cols"]),
            "beta": torch.full((1,), 0.02, device=DEV)}


def _ffn_inputs(c, i):
    dm, ff = c["d_model"], c["d_ff"]
    return {"gu": i.trits(2 * ff, dm), "d": i.trits(dm, ff), "x": i.normal(c["tokens"], dm),
            "gain": i.uniform(dm, 0.75, 1.25), "bgu": torch.full((2 * ff,), math.sqrt(2.0 / dm), device=DEV),
            "bd": torch.full((1,), math.sqrt(2.0 / ff), device=DEV)}


def _cache_inputs(c, i, seqs, slots):
    """q and fp16 caches [seqs][kvheads][max_seq][hd] holding `slots` positions."""
    rows = c.get("qper", 1) * seqs
    k = torch.zeros(seqs, c["kvheads"], c["max_seq"], c["head_dim"], device=DEV, dtype=torch.float16)
    v = torch.zeros_like(k)
    k[:, :, :slots] = i.half(seqs, c["kvheads"], slots, c["head_dim"])
    v[:, :, :slots] = i.half(seqs, c["kvheads"], slots, c["head_dim"])
    return {"q": i.normal(rows, c["heads"] * c["head_dim"]), "k": k, "v": v}


def _paged_inputs(c, i):
    batch, bs = c["batch"], c["bs"]
    mbps = (c["longest"] + bs - 1) // bs
    lens = i.ints(batch, 0, c["longest"])
    lens[0] = c["longest"] - 1
    npool = batch * mbps + 1
    table = torch.randperm(npool, generator=i.g, device=DEV, dtype=torch.int64)[:batch * mbps].to(torch.int32)
    shape = (npool, bs, c["kvheads"], c["head_dim"])
    return {"q": i.normal(batch, c["heads"] * c["head_dim"]), "k": i.half(*shape), "v": i.half(*shape),
            "lens": lens, "table": table.view(batch, mbps)}


def _softmax_inputs(c, i):
    a = i.normal(c["rows"], c["cols"], sigma=3.0)
    # scores of causal tiles: row r keeps the first r % cols + 1 columns
    keep = torch.arange(c["rows"], device=DEV) % c["cols"]
    for r0 in range(0, c["rows"], 16384):
        s = slice(r0, r0 + 16384)
        a[s].masked_fill_(torch.arange(c["cols"], device=DEV)[None, :] > keep[s, None], -math.inf)
    return {"a": a}


def _matmul_inputs(c, i):
    m, k, n = c["m"], c["k"], c["n"]
    if c["kernel"] == "linear":
        return {"a": i.normal(m, k), "b": i.normal(n, k, sigma=1.0 / math.sqrt(k)), "bias": i.normal(n)}
    return {"a": i.uniform(m * k, -1, 1).view(m, k), "b": i.uniform(k * n, -1, 1).view(k, n)}


def _gqa_inputs(c, i):
    kv = c["kvheads"] * c["head_dim"]
    return {"q": i.normal(c["seq"], c["heads"] * c["head_dim"]), "k": i.normal(c["seq"], kv),
            "v": i.normal(c["seq"], kv)}


def _decode_f32_inputs(c, i):
    kv = c["kvheads"] * c["head_dim"]
    k = torch.zeros(c["batch"], c["max_seq"], kv, device=DEV)
    v = torch.zeros_like(k)
    k[:, :c["pos"] + 1] = i.normal(c["batch"], c["pos"] + 1, kv)
    v[:, :c["pos"] + 1] = i.normal(c["batch"], c["pos"] + 1, kv)
    return {"q": i.normal(c["batch"], c["heads"] * c["head_dim"]), "k": k, "v": v}


def _ternary_inputs(c, i):
    nblk = (c["cols"] + 127) // 128
    d = {"t": i.trits(c["out"], c["cols"]), "beta": i.uniform(c["out"] * nblk, 0.01, 0.06).view(c["out"], nblk)}
    if c["kind"] == "ternary":
        d["x"], d["bias"] = i.normal(c["seq"], c["cols"]), i.uniform(c["out"], -0.2, 0.2)
    else:
        d["g"] = i.normal(c["seq"], c["out"])
    return d


def _inputs(case, seed):
    i = Inputs(seed)
    k = case["kind"]
    if k == "linear":
        return _linear_inputs(case, i)
    if k == "ffn":
        return _ffn_inputs(case, i)
    if k == "attn_decode":
        return _cache_inputs(case, i, case["batch"], case["pos"] + 1)
    if k == "attn_prompt":
        slots = case["pos0"] + case["qper"]
        return _cache_inputs(dict(case, max_seq=slots), i, case["prompts"], slots)
    if k == "attn_paged":
        return _paged_inputs(case, i)
    if k == "softmax":
        return _softmax_inputs(case, i)
    if k == "matmul":
        return _matmul_inputs(case, i)
    if k == "gqa":
        return _gqa_inputs(case, i)
    if k == "decode_f32":
        return _decode_f32_inputs(case, i)
    return _ternary_inputs(case, i)


# Two layers: through more of them, one int8 lane that crosses a rounding
# boundary grows into 3-5% of the logits, and nothing could be compared.
STACK = dict(layers=2, d_model=2560, heads=20, kv_heads=5, head_dim=128, d_ff=6912, vocab=128256)


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "stack":
        nlgpu.init()
        s = nlgpu.Stack(max_seq=768, batch=c["batch"], seed=20260921 + int(seed), **STACK)
        prompts = np.random.default_rng(int(seed)).integers(0, STACK["vocab"], (c["batch"], c["tokens"]))
        return {"c": c, "stack": s, "prompts": prompts.astype(np.int32)}
    d = _inputs(c, seed)
    b = {"c": c}
    k = c["kind"]
    if k == "linear":
        b["w"] = weights(d["t"], c["cols"] % 256 == 0 and c["tokens"] >= 4)
        b["ws"] = nlgpu.DeviceArray(max(4, nlgpu.ternary_linear_workspace(c["tokens"], c["cols"])))
        b.update(x=View(d["x"]), beta=View(d["beta"]), y=View(_empty(c["tokens"], c["out"])))
    elif k == "ffn":
        b["gu"], b["d"] = (weights(d[n], c["tokens"] >= 4) for n in ("gu", "d"))
        b.update({n: View(d[n]) for n in ("x", "gain", "bgu", "bd")})
        b.update(h=View(_empty(c["tokens"], c["d_ff"])), y=View(_empty(c["tokens"], c["d_model"])))
    elif k == "attn_decode":
        b.update({n: View(d[n]) for n in "qkv"})
        b["pos"] = View(torch.tensor([c["pos"]], device=DEV, dtype=torch.int32))
        b["ws"] = nlgpu.DeviceArray(nlgpu.decode_attn_f16_workspace(c["batch"], c["heads"], c["kvheads"],
                                                                    c["head_dim"], c["max_seq"]))
        b["y"] = View(_empty(c["batch"], c["heads"] * c["head_dim"]))
    elif k == "attn_prompt":
        b.update({n: View(d[n]) for n in "qkv"})
        b["pos"] = View(torch.tensor([c["pos0"]], device=DEV, dtype=torch.int32))
        b["y"] = View(_empty(c["prompts"] * c["qper"], c["heads"] * c["head_dim"]))
    elif k == "attn_paged":
        b.update({n: View(d[n]) for n in ("q", "k", "v", "lens", "table")})
        b["npool"], b["mbps"] = d["k"].shape[0], d["table"].shape[1]
        b["ws"] = nlgpu.DeviceArray(nlgpu.decode_attn_paged_f16_workspace(
            c["batch"], c["heads"], c["kvheads"], c["head_dim"], c["bs"], b["mbps"]))
        b["y"] = View(_empty(c["batch"], c["heads"] * c["head_dim"]))
    elif k == "softmax":
        b.update(a=View(d["a"]), y=View(_empty(c["rows"], c["cols"])))
    elif k == "matmul":
        y = b["y"] = View(_empty(c["m"], c["n"]))
        b["bufs"] = [View(d[n]) for n in ("a", "b", "bias") if n in d] + [y]
        b["push"] = [c["m"], c["k"], c["n"]]
        b["groups"] = {"matmul-tiled": ((c["m"] + 15) // 16) * ((c["n"] + 15) // 16),
                       "matmul-reg": (c["m"] * c["n"] // 16 + 63) // 64}.get(c["kernel"],
                                                                             (c["m"] * c["n"] + 63) // 64)
        b["name"] = c["kernel"]
    elif k == "gqa":
        y = b["y"] = View(_empty(c["seq"], c["heads"] * c["head_dim"]))
        b["bufs"] = [View(d[n]) for n in "qkv"] + [y]
        b["push"] = [c["seq"], c["heads"], c["kvheads"], c["head_dim"]]
        b["groups"] = (c["heads"] * c["seq"] + 63) // 64
        b["name"] = "attn-causal-gqa"
    elif k == "decode_f32":
        dim = c["heads"] * c["head_dim"]
        y = b["y"] = View(_empty(c["batch"], dim))
        b["bufs"] = [View(d[n]) for n in "qkv"] + [View(torch.tensor([float(c["pos"])], device=DEV)), y]
        b["push"] = [c["batch"], dim, c["heads"], c["kvheads"], c["max_seq"]]
        b["groups"] = (c["batch"] * dim + 63) // 64
        b["name"] = "decode-attn-b"
    else:
        seq, out, cols = c["seq"], c["out"], c["cols"]
        nblk, wng = (cols + 127) // 128, (cols + 15) // 16
        w, beta = View(pack_words(d["t"])), View(d["beta"])
        if k == "ternary":
            y = View(_empty(seq, out))
            b["bufs"], b["push"] = [View(d["x"]), w, View(d["bias"]), beta, y], [seq, out, cols, nblk, wng]
            b["name"], b["groups"] = "ternary-rows", (seq * out + 63) // 64
        else:
            y = View(_empty(seq, cols))
            b["bufs"], b["push"] = [w, beta, View(d["g"]), y], [out, cols, nblk, wng, seq]
            b["name"], b["groups"] = "ternary-rows-t", (seq * cols + 63) // 64
        b["y"] = y
    return b


def run(b):
    c = b["c"]
    k = c["kind"]
    if k == "linear":
        nlgpu.ternary_linear(b["x"], b["w"], None, b["beta"], b["y"], c["tokens"], c["out"], c["cols"],
                             workspace=b["ws"])
    elif k == "ffn":
        nlgpu.rms_ternary_swiglu(b["x"], b["gain"], 1e-5, b["gu"], b["bgu"], b["h"], c["tokens"], c["d_ff"],
                                 c["d_model"])
        nlgpu.ternary_linear_residual(b["h"], b["d"], None, b["bd"], b["x"], b["y"], c["tokens"], c["d_model"],
                                      c["d_ff"])
    elif k == "attn_decode":
        nlgpu.decode_attn_f16(b["q"], b["k"], b["v"], b["pos"], b["y"], c["batch"], c["heads"], c["kvheads"],
                              c["head_dim"], c["max_seq"], b["ws"])
    elif k == "attn_prompt":
        nlgpu.prefill_attn_f16(b["q"], b["k"], b["v"], b["pos"], c["prompts"] * c["qper"], c["qper"], c["heads"],
                               c["kvheads"], c["head_dim"], c["pos0"] + c["qper"], b["y"])
    elif k == "attn_paged":
        nlgpu.decode_attn_paged_f16(b["q"], b["k"], b["v"], b["lens"], b["table"], b["npool"], b["y"], c["batch"],
                                    c["heads"], c["kvheads"], c["head_dim"], c["bs"], b["mbps"], b["ws"])
    elif k == "softmax":
        nlgpu.softmax_rows(b["a"], b["y"], c["rows"], c["cols"])
    elif k == "stack":
        s = b["stack"]
        if c["mode"] == "prompt":
            s.prefill(b["prompts"])
        else:
            s.start(b["prompts"])
            s.step(c["tokens"])
        return {"logits": s.logits()}
    else:
        nlgpu.dispatch(b["name"], b["bufs"], b["push"], b["groups"])
    return b["y"].t


# ------------------------------------------------------------------ the bounds

def work(case):
    c, k = case, case["kind"]
    if k == "linear":
        s, o, n = c["tokens"], c["out"], c["cols"]
        return {"bytes": o * n / 4 + 4 * s * (n + o) + 4, "flops": 2 * s * o * n}
    if k == "ffn":
        s, dm, ff = c["tokens"], c["d_model"], c["d_ff"]
        return {"bytes": 3 * dm * ff / 4 + 8 * s * dm + 4 * dm + 8 * ff, "flops": 6 * s * dm * ff}
    if k == "attn_decode":
        n = c["batch"] * (c["pos"] + 1) * c["head_dim"]
        return {"bytes": 4 * n * c["kvheads"] + 8 * c["batch"] * c["heads"] * c["head_dim"],
                "flops": 4 * n * c["heads"]}
    if k == "attn_prompt":
        p, n = c["qper"], c["pos0"] + c["qper"]
        pairs = c["prompts"] * (p * c["pos0"] + p * (p + 1) // 2)
        return {"bytes": 4 * c["prompts"] * n * c["kvheads"] * c["head_dim"]
                + 8 * c["prompts"] * p * c["heads"] * c["head_dim"],
                "flops": 4 * pairs * c["heads"] * c["head_dim"]}
    if k == "attn_paged":
        n = c["batch"] * (c["longest"] / 2) * c["head_dim"]  # lengths are uniform
        return {"bytes": 4 * n * c["kvheads"] + 8 * c["batch"] * c["heads"] * c["head_dim"],
                "flops": 4 * n * c["heads"]}
    if k == "softmax":
        n = c["rows"] * c["cols"]
        return {"bytes": 8 * n, "flops": 4 * n}
    if k == "stack":
        d, ff, nq, nkv = STACK["d_model"], STACK["d_ff"], 2560, 640
        layer = d * (nq + 2 * nkv) + nq * d + 3 * d * ff
        head = d * STACK["vocab"]
        n, b = c["tokens"], c["batch"]
        kv = STACK["layers"] * 4 * nkv * n * b
        if c["mode"] == "prompt":
            return {"bytes": (STACK["layers"] * layer + head) / 4 + kv + 4 * b * (n * d + STACK["vocab"]),
                    "flops": 2 * b * (n * STACK["layers"] * layer + head)}
        return {"bytes": n * ((STACK["layers"] * layer + head) / 4 + kv / 2 + 4 * b * STACK["vocab"]),
                "flops": 2 * b * n * (STACK["layers"] * layer + head)}
    if k == "matmul":
        m, kk, n = c["m"], c["k"], c["n"]
        return {"bytes": 4 * (m * kk + kk * n + m * n), "flops": 2 * m * kk * n}
    if k == "gqa":
        n, hd = c["seq"], c["head_dim"]
        return {"bytes": 8 * n * hd * (c["heads"] + c["kvheads"]), "flops": 2 * n * (n + 1) * hd * c["heads"]}
    if k == "decode_f32":
        n = c["batch"] * (c["pos"] + 1) * c["head_dim"]
        return {"bytes": 8 * n * c["kvheads"] + 8 * c["batch"] * c["heads"] * c["head_dim"],
                "flops": 4 * n * c["heads"]}
    s, o, n = c["seq"], c["out"], c["cols"]
    return {"bytes": o * n / 4 + o * n / 32 + 4 * s * (o + n), "flops": 2 * s * o * n}


def tolerance(case):
    k = case["kind"]
    if k == "linear":
        return {"rel": 1e-6}
    if k == "ffn":
        # a lane that crosses a rounding boundary because the norm was summed
        # in another order: up to 2.2e-4, one value 0.013
        return {"rel": 1e-3, "max": 0.05}
    if k == "stack":
        # the same through two layers: prefill against single steps 0.8-1.9%
        return {"rel": 0.03, "max": 0.35}
    if k == "softmax":
        return {"rel": 1e-6, "max": 1e-5}
    # f32 sums in another order: up to 9.4e-7, one value 6.8e-6
    return {"rel": 4e-6, "max": 3e-5}


# ------------------------------------------------------------------ in 64 bits

def _quantise(x):
    """int8 lanes and scale per row: the data format itself, rounded in 32 bits as it is defined."""
    x = x.float()
    gamma = x.abs().amax(dim=1, keepdim=True) / 127.0
    q = torch.clamp(torch.floor((x / torch.where(gamma > 0, gamma, torch.ones_like(gamma))).abs() + 0.5), max=127.0)
    return (torch.sign(x) * q).double(), gamma.double()


def _linear64(x, t, beta):
    q, gamma = _quantise(x)
    y = torch.empty(x.shape[0], t.shape[0], device=DEV, dtype=torch.float64)
    for o in range(0, t.shape[0], 2048):
        y[:, o:o + 2048] = q @ t[o:o + 2048].double().t()
    return y * gamma * beta.double()


def _attend64(q, k, v, first):
    """Causal attention of one sequence: q [n, heads, hd], k and v [kvheads, len, hd];
    query i attends positions 0..first + i."""
    n, heads, hd = q.shape
    grp = heads // k.shape[0]
    out = torch.empty(n, heads, hd, device=DEV, dtype=torch.float64)
    at = torch.arange(k.shape[1], device=DEV)[None, :] > first + torch.arange(n, device=DEV)[:, None]
    for h in range(heads):
        s = (q[:, h].double() @ k[h // grp].double().t()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(at, -math.inf), dim=1) @ v[h // grp].double()
    return out.reshape(n, heads * hd)


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "stack":
        return None
    d = _inputs(c, seed)
    if k == "linear":
        return _linear64(d["x"], d["t"], d["beta"])
    if k == "ffn":
        x = d["x"].double()
        xn = x / torch.sqrt(x.square().mean(dim=1, keepdim=True) + 1e-5) * d["gain"].double()
        gu = _linear64(xn, d["gu"], d["bgu"])
        g, u = gu[:, 0::2], gu[:, 1::2]
        return x + _linear64(g * torch.sigmoid(g) * u, d["d"], d["bd"])
    if k in ("attn_decode", "attn_prompt"):
        n, first = (1, c["pos"]) if k == "attn_decode" else (c["qper"], c["pos0"])
        seqs = d["k"].shape[0]
        q = d["q"].view(seqs, n, c["heads"], c["head_dim"])
        return torch.cat([_attend64(q[s], d["k"][s, :, :first + n], d["v"][s, :, :first + n], first)
                          for s in range(seqs)])
    if k == "attn_paged":
        q = d["q"].view(c["batch"], 1, c["heads"], c["head_dim"])
        rows = []
        for s in range(c["batch"]):
            n = int(d["lens"][s]) + 1
            blocks = d["table"][s, :(n + c["bs"] - 1) // c["bs"]].long()
            kv = [d[x][blocks].reshape(-1, c["kvheads"], c["head_dim"])[:n].transpose(0, 1) for x in "kv"]
            rows.append(_attend64(q[s], kv[0], kv[1], n - 1))
        return torch.cat(rows)
    if k == "softmax":
        y = torch.empty(c["rows"], c["cols"], device=DEV, dtype=torch.float64)
        for r in range(0, c["rows"], 16384):
            y[r:r + 16384] = torch.softmax(d["a"][r:r + 16384].double(), dim=1)
        return y
    if k == "matmul":
        if c["kernel"] == "linear":
            return d["a"].double() @ d["b"].double().t() + d["bias"].double()
        return d["a"].double() @ d["b"].double()
    if k in ("gqa", "decode_f32"):
        hd, seqs = c["head_dim"], 1 if k == "gqa" else c["batch"]
        n, first = (c["seq"], 0) if k == "gqa" else (1, c["pos"])
        q = d["q"].view(seqs, n, c["heads"], hd)
        kv = [d[x].view(seqs, -1, c["kvheads"], hd)[:, :first + n].transpose(1, 2) for x in "kv"]
        return torch.cat([_attend64(q[s], kv[0][s], kv[1][s], first) for s in range(seqs)])
    w = d["t"].double() * d["beta"].double().repeat_interleave(128, dim=1)[:, :c["cols"]]
    if k == "ternary":
        return d["x"].double() @ w.t() + d["bias"].double()
    return d["g"].double() @ w
