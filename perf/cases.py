"""The work that this library is used for, as timed cases.

Three kinds, each through the entry points a host program calls:

  linear   one quantized linear through ``QKernelMatMul::forward`` (its C form ``lkh_qkernel_matmul_*``): the
           call of every projection of a model, from a decode step's single row to a prefill chunk of 2048
  decode   the quantized linears of several layers of a decode step over 1 to 64 sequences, recorded once into
           a HIP graph and replayed per step, as a serving loop does
  moe      router and expert block of a mixture layer: ``gate_topk_softmax``, then ``moe_forward``

Shapes are those of the benchmark's configurations (Llama-3-8B, Qwen3-1.7B, Qwen3-30B-A3B) and generic ones.
Weights are random blocks with the field distributions of ``loken_amd/synth.py``; activations are N(0, 1).
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from loken_amd import lib, moe, ops, synth

DEV = "cuda:0"
TYPES = {"q4_k": lib.TYPE_Q4_K, "q5_k": lib.TYPE_Q5_K, "q6_k": lib.TYPE_Q6_K, "q8_0": lib.TYPE_Q8_0,
         "q4_0": lib.TYPE_Q4_0, "mxfp4": lib.TYPE_MXFP4}
X_TYPES = {"f32": (torch.float32, lib.TYPE_F32), "f16": (torch.float16, lib.TYPE_F16), "bf16": (torch.bfloat16, lib.TYPE_BF16)}
# hidden size, k / v rows, feed-forward width of the two dense models the benchmark is quoted on
MODELS = {"llama3-8b": (4096, 1024, 14336), "qwen3-1.7b": (2048, 1024, 6144)}


# ------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest call: one token through a k or v projection of a small model
        {"name": "linear-kv-1row", "kind": "linear", "wtype": "q4_k", "n": 1024, "k": 2048, "rows": 1, "x": "f32"},
        # the largest mat-vec: one token's logits over a 128256-word vocabulary
        {"name": "linear-lm-head-1row", "kind": "linear", "wtype": "q8_0", "n": 128256, "k": 4096, "rows": 1, "x": "f32"},
        # continuous batching of a few sequences in bf16
        {"name": "linear-7rows-bf16", "kind": "linear", "wtype": "q4_k", "n": 4096, "k": 4096, "rows": 7, "x": "bf16"},
        # a short prefill chunk, ragged in rows and columns, in f16
        {"name": "linear-77rows-ragged-f16", "kind": "linear", "wtype": "q5_k", "n": 11003, "k": 4096, "rows": 77, "x": "f16"},
        # prefill: a Q4_K gate projection over 512 tokens, a Q6_K down projection over 2048
        {"name": "linear-prefill-512", "kind": "linear", "wtype": "q4_k", "n": 14336, "k": 4096, "rows": 512, "x": "f32"},
        {"name": "linear-prefill-2048", "kind": "linear", "wtype": "q6_k", "n": 4096, "k": 14336, "rows": 2048, "x": "f32"},
        # decode steps: one sequence of the larger model, sixteen of the smaller
        {"name": "decode-llama-1row", "kind": "decode", "model": "llama3-8b", "layers": 4, "rows": 1},
        {"name": "decode-qwen-16rows", "kind": "decode", "model": "qwen3-1.7b", "layers": 6, "rows": 16},
        # a mixture layer at one token, at sixteen, at a short and at a long prefill chunk; the last with the
        # Q6_K down projection that a Q4_K_M file stores
        {"name": "moe-1token", "kind": "moe", "gu": "q4_k", "down": "q4_k", "experts": 128, "topk": 8, "hidden": 2048, "ffn": 768, "tokens": 1},
        {"name": "moe-16tokens", "kind": "moe", "gu": "q4_k", "down": "q4_k", "experts": 128, "topk": 8, "hidden": 2048, "ffn": 768, "tokens": 16},
        {"name": "moe-256tokens", "kind": "moe", "gu": "q4_k", "down": "q4_k", "experts": 128, "topk": 8, "hidden": 2048, "ffn": 768, "tokens": 256},
        {"name": "moe-1111tokens-mixed", "kind": "moe", "gu": "q4_k", "down": "q6_k", "experts": 128, "topk": 8, "hidden": 2048, "ffn": 768, "tokens": 1111},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "decode", "moe", "moe"])
    if kind == "linear":
        wtype = rng.choice(["q4_k", "q4_k", "q4_k", "q6_k", "q6_k", "q5_k", "q8_0", "q4_0"])
        x = rng.choice(["f32", "f32", "f16", "bf16"])
        if rng.random() < 0.15:   # a vocabulary: few rows, many columns
            return {"kind": kind, "wtype": wtype, "n": _log_int(rng, 32000, 128256), "k": 256 * rng.randint(8, 16),
                    "rows": _log_int(rng, 1, 16), "x": x}
        n, k, rows = _log_int(rng, 512, 16384), 256 * _log_int(rng, 4, 56), _log_int(rng, 1, 2048)
        return {"kind": kind, "wtype": wtype, "n": n, "k": k, "rows": max(1, min(rows, 2048 * 14336 * 4096 // (n * k))), "x": x}
    if kind == "decode":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "layers": rng.randint(2, 6), "rows": _log_int(rng, 1, 64)}
    gu, down = rng.choice([("q4_k", "q4_k"), ("q4_k", "q4_k"), ("q4_k", "q6_k"), ("q6_k", "q6_k"), ("q5_k", "q5_k"),
                           ("q8_0", "q8_0"), ("mxfp4", "mxfp4")])
    return {"kind": kind, "gu": gu, "down": down, "experts": rng.choice([8, 32, 60, 64, 128]), "topk": rng.choice([2, 4, 8]),
            "hidden": 256 * rng.randint(4, 12), "ffn": 256 * rng.randint(2, 6), "tokens": _log_int(rng, 1, 1400)}


# ------------------------------------------------------------------------------------------ inputs
class _Maker:
    """Weights and activations made on the card from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)

    def randn(self, *shape):
        return torch.randn(shape, device=DEV, generator=self.gen)

    def _half(self, blocks, scale):
        return (self.randn(blocks).abs() * scale).to(torch.float16).view(torch.uint8).reshape(blocks, 2)

    def weight(self, wtype, n, k):
        t = TYPES[wtype]
        blocks, size = n * (k // synth.BLOCK_LEN[t]), synth.BLOCK_BYTES[t]
        blob = torch.zeros(blocks * size + 4096, dtype=torch.uint8, device=DEV)   # the zero tail of an uploaded tensor
        w = blob[:blocks * size].view(blocks, size)
        w.random_(0, 256, generator=self.gen)
        if wtype in ("q4_k", "q5_k"):     # d, dmin; packed six-bit scales, fifth bits and nibbles take any byte
            w[:, 0:2] = self._half(blocks, 1e-3)
            w[:, 2:4] = self._half(blocks, 5e-4)
        elif wtype == "q6_k":             # codes, sixteen int8 scales, d
            w[:, 192:208] = (w[:, 192:208] & 127) - 64
            w[:, 208:210] = self._half(blocks, 1e-3)
        elif wtype == "q8_0":
            w[:, 0:2] = self._half(blocks, 1e-3)
            w.view(torch.int8)[:, 2:].clamp_(min=-127)
        elif wtype == "q4_0":
            w[:, 0:2] = self._half(blocks, 2e-3)
        elif wtype == "mxfp4":            # one power-of-two scale byte, 2^-12 .. 2^-5
            w[:, 0] = 116 + (w[:, 0] & 7)
        return blob


class _Linear:
    """The handle a program keeps for one quantized linear."""

    def __init__(self, wtype, n, k, blob):
        self.blob = blob
        self.lib = lib.load()
        self.handle = self.lib.lkh_qkernel_matmul_new(TYPES[wtype], n, k, blob.data_ptr(), 0)

    def __del__(self):
        self.lib.lkh_qkernel_matmul_free(self.handle)


def prepare(case, seed):
    mk = _Maker(seed)
    if case["kind"] == "linear":
        n, k, rows = case["n"], case["k"], case["rows"]
        dtype, x_type = X_TYPES[case["x"]]
        return {"case": case, "linear": _Linear(case["wtype"], n, k, mk.weight(case["wtype"], n, k)), "x_type": x_type,
                "x": mk.randn(rows, k).to(dtype), "out": torch.empty((rows, n), dtype=dtype, device=DEV)}
    if case["kind"] == "moe":
        experts, hidden, ffn = case["experts"], case["hidden"], case["ffn"]
        return {"case": case, "x": mk.randn(case["tokens"], hidden), "router": mk.randn(experts, hidden) / math.sqrt(hidden),
                "gate": mk.weight(case["gu"], experts * ffn, hidden), "up": mk.weight(case["gu"], experts * ffn, hidden),
                "down": mk.weight(case["down"], experts * hidden, ffn)}
    return _prepare_decode(case, mk)


def _prepare_decode(case, mk):
    """One step's launches over the C ABI: f32 rows into every group of linears that share an activation, the
    gate + up launch handing `down` its Q8_1 rows. Up to two rows the mat-vec launches that quantize as they go,
    above that a quantizer launch and the launches on the matrix unit."""
    L = lib.load()
    hidden, kv, ffn = MODELS[case["model"]]
    b = case["rows"]
    plan, keep, outputs = [], [], []

    def f32_out(n, stride=None):
        o = torch.empty((b, stride or n), device=DEV)
        outputs.append(o[:, :n])
        return o

    def several(weights, sizes, stride=None):
        outs = [f32_out(n, stride) for n in sizes]
        vx = (C.c_void_p * len(weights))(*[w.data_ptr() for w in weights])
        dst = (C.c_void_p * len(weights))(*[o.data_ptr() for o in outs])
        ns = (C.c_int * len(weights))(*sizes)
        keep.extend([vx, dst, ns])
        return vx, dst, ns

    for _ in range(case["layers"]):
        wq, wk, wv, wo = (mk.weight("q4_k", n, hidden) for n in (hidden, kv, kv, hidden))
        wg, wu, wd = mk.weight("q4_k", ffn, hidden), mk.weight("q4_k", ffn, hidden), mk.weight("q6_k", hidden, ffn)
        x, attn, x2 = mk.randn(b, hidden), mk.randn(b, hidden), mk.randn(b, hidden)
        h = torch.empty((b, ffn // 32, 36), dtype=torch.uint8, device=DEV)
        keep.extend([wq, wk, wv, wo, wg, wu, wd, x, attn, x2, h])
        if b <= 2:
            for weights, sizes, row in (((wq, wk, wv), [hidden, kv, kv], x), ((wo,), [hidden], attn)):
                vx, dst, ns = several(weights, sizes, hidden)
                plan.append((L.lk_mmvq_fused, (lib.TYPE_Q4_K, len(sizes), vx, row.data_ptr(), hidden, dst, lib.TYPE_F32, hidden, ns, b,
                                               hidden, None)))
            plan.append((L.lk_mmvq_pair_act_q8_1, (lib.TYPE_Q4_K, wg.data_ptr(), wu.data_ptr(), x2.data_ptr(), 1, hidden, h.data_ptr(),
                                                   ffn // 32, hidden, ffn, b, 0)))
            plan.append((L.lk_mmvq, (lib.TYPE_Q6_K, wd.data_ptr(), h.data_ptr(), f32_out(hidden).data_ptr(), lib.TYPE_F32, ffn, hidden, b,
                                     ffn // 32, hidden, None, 0)))
            continue
        q81 = [torch.empty((b, hidden // 32, 36), dtype=torch.uint8, device=DEV) for _ in range(3)]
        keep.extend(q81)

        def quantize(row, q):
            plan.append((L.lk_quantize_q8_1, (row.data_ptr(), lib.TYPE_F32, q.data_ptr(), hidden, hidden, b)))

        quantize(x, q81[0])
        vx, dst, ns = several((wq, wk, wv), [hidden, kv, kv])
        plan.append((L.lk_dense_q4k_rows_multi, (vx, dst, ns, 3, q81[0].data_ptr(), b, hidden, 0)))
        quantize(attn, q81[1])
        plan.append((L.lk_dense_q4k_rows, (wo.data_ptr(), q81[1].data_ptr(), f32_out(hidden).data_ptr(), b, hidden, hidden)))
        quantize(x2, q81[2])
        plan.append((L.lk_dense_q4k_rows_actmul_q8_1, (wg.data_ptr(), wu.data_ptr(), q81[2].data_ptr(), h.data_ptr(), b, ffn, hidden, 0, 0)))
        plan.append((L.lk_dense_q6k_rows, (wd.data_ptr(), h.data_ptr(), f32_out(hidden).data_ptr(), b, hidden, ffn)))

    def step():
        stream = torch.cuda.current_stream().cuda_stream
        for fn, args in plan:
            lib.check("decode step", fn(*args, stream))

    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        step()
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            step()
    torch.cuda.synchronize()
    return {"case": case, "graph": graph, "outputs": outputs, "keep": keep}


# ------------------------------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        linear, x, out = state["linear"], state["x"], state["out"]
        lib.check("forward", linear.lib.lkh_qkernel_matmul_forward(linear.handle, x.data_ptr(), state["x_type"], case["rows"],
                                                                   out.data_ptr(), torch.cuda.current_stream().cuda_stream, 0))
        return out
    if case["kind"] == "moe":
        weights, choices = moe.gate_topk_softmax(state["x"], state["router"], case["topk"])
        out = moe.moe_forward(TYPES[case["gu"]], TYPES[case["down"]], state["x"], state["gate"], state["up"], state["down"], choices,
                              weights, case["experts"], case["ffn"])
        return out, weights, choices
    state["graph"].replay()
    return state["outputs"]


# ------------------------------------------------------------------------------------------ what a pass needs
def work(case):
    if case["kind"] == "linear":
        n, k, rows = case["n"], case["k"], case["rows"]
        size = 4 if case["x"] == "f32" else 2
        return {"bytes": synth.weight_bytes(TYPES[case["wtype"]], n, k) + rows * (n + k) * size, "flops": 2.0 * rows * n * k}
    if case["kind"] == "decode":
        hidden, kv, ffn = MODELS[case["model"]]
        b, layers = case["rows"], case["layers"]
        q4k, q6k = (2 * hidden + 2 * kv + 2 * ffn) * hidden, hidden * ffn
        values = 3 * hidden + (3 * hidden + 2 * kv)      # rows in, rows out
        return {"bytes": layers * (synth.weight_bytes(TYPES["q4_k"], 1, q4k) + synth.weight_bytes(TYPES["q6_k"], 1, q6k) + 4 * b * values),
                "flops": 2.0 * layers * b * (q4k + q6k)}
    experts, topk, hidden, ffn, tokens = (case[key] for key in ("experts", "topk", "hidden", "ffn", "tokens"))
    topk = min(topk, experts)
    # experts that some token chooses, were every choice equally likely
    hit = experts * (1.0 - (1.0 - topk / experts) ** tokens)
    per_expert = 2 * synth.weight_bytes(TYPES[case["gu"]], ffn, hidden) + synth.weight_bytes(TYPES[case["down"]], hidden, ffn)
    return {"bytes": hit * per_expert + 4.0 * experts * hidden + 8.0 * tokens * (hidden + topk),
            "flops": 2.0 * tokens * (3 * topk * ffn * hidden + experts * hidden)}


def tolerance(case):
    if case["kind"] == "linear":
        # exact integer dots, f32 scales and sums; then the rounding of the output type
        return {"f32": {"rel": 1e-5}, "f16": {"rel": 5e-4, "max": 2e-3}, "bf16": {"rel": 4e-3, "max": 1.6e-2}}[case["x"]]
    # the gated rows are quantized to eight bits again: a last-place difference can move a code by one
    return {"rel": 1e-3, "max": 2e-2, "differ": 1e-3}
