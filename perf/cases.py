"""The work this library is measured on: what a program that serves a model with Q4 / Q8 weights
asks of it, from the smallest decode call to a large prefill, through the public Python faces
(capi.Context for programs that keep their data on the device, Graph / Session for programs that
hand over and read back host arrays).

A case is a dict of plain values; `kind` says which part of such a program it is:

  qkv     the q, k and v projections of one token behind their rms_norm: one batched call
  gemm    one matmul (f32 or fp16 activations, with or without a residual)
  ffn     decode of one or two tokens through a stack of gated MLPs: rms_norm -> gate|up, then
          SwiGLU -> down + residual, each one fused call
  mlp     the same for any number of rows and a plain MLP: up with silu epilogue, down + residual
  layers  decoder layers in a Session (norms, projections, gated MLP), host inputs to host output
  load    a weight from host f32 values to the device and its packed bytes back (import / export)

Weights are N(0, 0.02), activations N(0, 1), as in the benchmark.
"""
import math

import numpy as np
import torch

from meganeura_amd import capi
from meganeura_amd.graph import Graph, build_inference_session

FMTS = {"q4": capi.FMT_Q4, "q8": capi.FMT_Q8}
MAX_WEIGHT = 4096 * 14336            # elements of the largest single weight
MAX_FLOPS = 2 * 2048 * MAX_WEIGHT    # of the largest case


def listed():
    return [
        # one token, one small layer: the launch-bound end of decode (SmolLM2-135M widths, Q8)
        dict(name="qkv_q8_m1_576", kind="qkv", fmt="q8", m=1, k=576, n=576, kv=192),
        # logits of one token over a small model's vocabulary: very wide, short K
        dict(name="lm_head_q4_576x49152", kind="gemm", fmt="q4", m=1, k=576, n=49152, act="f32", residual=False),
        # one token through eight decoder layers and the lm_head, as a host program sees it
        dict(name="decode_session_q4", kind="layers", fmt="q4", m=1, k=576, kv=192, n=1536, layers=8, vocab=49152),
        # one token through an 8B-sized model's gated MLPs: bandwidth-bound decode
        dict(name="ffn_q4_m1_4096x14336", kind="ffn", fmt="q4", m=1, k=4096, n=14336, layers=4),
        dict(name="ffn_q8_m1_4096x14336", kind="ffn", fmt="q8", m=1, k=4096, n=14336, layers=4),
        # small decode batches on the same weights
        dict(name="mlp_q4_m4_4096x14336", kind="mlp", fmt="q4", m=4, k=4096, n=14336, layers=4),
        dict(name="mlp_q8_m16_4096x14336", kind="mlp", fmt="q8", m=16, k=4096, n=14336, layers=4),
        # prefill of a 512-token prompt on a small model's up projection, fp16 activations
        dict(name="prefill_f16_q4_512x1024x3072", kind="gemm", fmt="q4", m=512, k=1024, n=3072, act="f16", residual=False),
        # a short, ragged prompt (or a large decode batch) through large MLPs, f32 activations
        dict(name="mlp_q4_m77_4096x14336", kind="mlp", fmt="q4", m=77, k=4096, n=14336, layers=2),
        # a ragged prompt through a small model's layers in a Session
        dict(name="prefill_session_q8_333x1024", kind="layers", fmt="q8", m=333, k=1024, kv=512, n=3072, layers=2, vocab=0),
        # a long prompt on a large model's up projection: the largest single call
        dict(name="prefill_f16_q4_2048x4096x14336", kind="gemm", fmt="q4", m=2048, k=4096, n=14336, act="f16", residual=False),
        # start-up: one large projection from f32 values to the device, and its packed bytes back
        dict(name="load_q4_4096x4096", kind="load", fmt="q4", k=4096, n=4096),
    ]


def _logint(rng, lo, hi, step=1):
    """An integer of [lo, hi], uniform in its logarithm, rounded to a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    while True:
        kind = rng.choice(["qkv", "gemm", "gemm", "gemm", "gemm", "ffn", "mlp", "mlp", "layers", "layers", "load"])
        case = dict(kind=kind, fmt=rng.choice(["q4", "q8"]))
        if kind == "qkv":
            case.update(m=rng.randint(1, 2), k=_logint(rng, 320, 4096, 32), n=_logint(rng, 320, 4096), kv=_logint(rng, 64, 1024))
        elif kind == "gemm":
            case.update(m=_logint(rng, 1, 2048), k=_logint(rng, 576, 14336, 32), n=_logint(rng, 192, 49152),
                        act=rng.choice(["f32", "f16"]), residual=rng.random() < 0.5)
        elif kind == "ffn":
            case.update(m=rng.randint(1, 2), k=_logint(rng, 576, 4096, 32), n=_logint(rng, 1536, 14336, 32), layers=rng.randint(1, 4))
        elif kind == "mlp":
            case.update(m=_logint(rng, 1, 1024), k=_logint(rng, 512, 4096, 32), n=_logint(rng, 1024, 14336, 32), layers=rng.randint(1, 4))
        elif kind == "layers":
            case.update(m=_logint(rng, 1, 512), k=_logint(rng, 256, 1024, 32), kv=_logint(rng, 64, 512), n=_logint(rng, 768, 3072, 32),
                        layers=rng.randint(1, 8), vocab=0)
            if case["m"] == 1 and rng.random() < 0.5:
                case["vocab"] = _logint(rng, 8192, 49152)
        else:
            case.update(k=_logint(rng, 512, 4096, 32), n=_logint(rng, 512, 14336))
        if case["k"] * case["n"] <= MAX_WEIGHT and work(case)["flops"] <= MAX_FLOPS:
            return case


def _weight_bytes(fmt, k, n):
    return (20 if fmt == "q4" else 34) * (k // 32) * n


def work(case):
    """Every weight and activation read once, every result written once; 2 m k n per matmul."""
    kind, fmt, k, n = case["kind"], case["fmt"], case["k"], case["n"]
    if kind == "load":
        # f32 values in, blocks on the device, the reference layout's bytes out
        return {"bytes": 4 * k * n + _weight_bytes(fmt, k, n) + capi.packed_size(FMTS[fmt], k, n), "flops": 0}
    m = case["m"]
    if kind == "qkv":
        cols = n + 2 * case["kv"]
        return {"bytes": _weight_bytes(fmt, k, cols) + 4 * (m * k + k + m * cols), "flops": 2 * m * k * cols}
    if kind == "gemm":
        a = 2 if case["act"] == "f16" else 4
        return {"bytes": _weight_bytes(fmt, k, n) + a * m * k + 4 * m * n * (2 if case["residual"] else 1), "flops": 2 * m * k * n}
    if kind == "ffn":
        w = _weight_bytes(fmt, k, 2 * n) + _weight_bytes(fmt, n, k)
        return {"bytes": case["layers"] * (w + 4 * k) + 8 * m * k, "flops": case["layers"] * 6 * m * k * n}
    if kind == "mlp":
        w = _weight_bytes(fmt, k, n) + _weight_bytes(fmt, n, k)
        return {"bytes": case["layers"] * w + 8 * m * k, "flops": case["layers"] * 4 * m * k * n}
    per_layer = 2 * k * k + 2 * k * case["kv"] + 3 * k * n
    w = (_weight_bytes(fmt, k, 2 * k + 2 * case["kv"] + 2 * n) + _weight_bytes(fmt, n, k) + 8 * k) * case["layers"]
    w += _weight_bytes(fmt, k, case["vocab"]) + (4 * k if case["vocab"] else 0)
    io = 4 * m * (2 * k + (case["vocab"] or k)) + 4 * m * case["layers"] * (k + 2 * case["kv"])
    return {"bytes": w + io, "flops": 2 * m * (per_layer * case["layers"] + k * case["vocab"])}


# About four times the error against the same computation in 64 bits (on the dequantized weights),
# (2-norm, largest): weights enter exactly, activations with at least 21 bits, sums are f32.  One
# matmul on centred data shows 1e-6; behind a silu the activations have a mean, sums of thousands
# of products cancel two digits of it, and a stack of layers adds that up (5e-5 after two of K = 14336).
_TOLERANCE = {"qkv": (1e-5, 1e-4), "gemm": (1e-5, 1e-4), "layers": (5e-5, 1.5e-4), "ffn": (8e-5, 3e-4), "mlp": (2e-4, 6e-4)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    rel, largest = _TOLERANCE[case["kind"]]
    return {"rel": rel, "max": largest}


_CONTEXTS = []


def _context():
    """The program's one context: it has the device to itself, so all models it holds share it."""
    if not _CONTEXTS:
        _CONTEXTS.append(capi.Context(0))
    return _CONTEXTS[0]


class _Program:
    """What a serving program holds of one model: device buffers and weights."""

    def __init__(self, seed):
        self.ctx = _context()
        self.held = []
        self.rng = torch.Generator(device="cuda").manual_seed(seed)

    def buffer(self, count, dtype=torch.float32):
        b = self.ctx.buffer(count * dtype.itemsize)
        self.held.append(b)
        return b

    def view(self, buf, shape, dtype=torch.float32):
        """The buffer as a torch tensor (no copy); it keeps the program alive."""
        return torch.as_tensor(_Array(self, buf, shape, "<f2" if dtype == torch.float16 else "<f4"), device="cuda")

    def normal(self, shape, sigma=1.0, mean=0.0, dtype=torch.float32):
        b = self.buffer(math.prod(shape), dtype)
        self.view(b, shape, dtype).normal_(mean, sigma, generator=self.rng)
        return b

    def weight(self, fmt, k, n):
        src = self.normal((k, n), 0.02)
        torch.cuda.synchronize()
        w = self.ctx.weight_from_device(FMTS[fmt], src, k, n)
        self.held.pop().free()
        self.held.append(w)
        return w

    def __del__(self):
        for h in reversed(self.held):
            h.free()


class _Array:
    def __init__(self, program, buf, shape, typestr):
        self.program = program
        self.__cuda_array_interface__ = {"data": (program.ctx.lib.mgn_buf_device_ptr(buf.h), False), "shape": tuple(shape),
                                         "typestr": typestr, "strides": None, "version": 2}


def _layers_graph(case):
    """Decoder layers without the attention core (its output is an input, q, k and v are outputs)."""
    m, k, kv, n = case["m"], case["k"], case["kv"], case["n"]
    shapes, norms = {}, []
    g = Graph()

    def quantized(name, rows, cols):
        shapes[name] = (rows, cols)
        return (g.parameter_q4 if case["fmt"] == "q4" else g.parameter_q8)(name, [rows, cols])

    def norm(x, name):
        norms.append(name)
        return g.rms_norm(x, g.parameter(name, [k]), 1e-5)

    x = g.input("x", [m, k])
    attn = g.input("attn", [m, k])
    outs = []
    for i in range(case["layers"]):
        n1 = norm(x, f"norm1.{i}")
        outs += [g.matmul(n1, quantized(f"wq.{i}", k, k)), g.matmul(n1, quantized(f"wk.{i}", k, kv)), g.matmul(n1, quantized(f"wv.{i}", k, kv))]
        h = g.add(g.matmul(attn, quantized(f"wo.{i}", k, k)), x)
        n2 = norm(h, f"norm2.{i}")
        gate, up = g.matmul(n2, quantized(f"wg.{i}", k, n)), g.matmul(n2, quantized(f"wu.{i}", k, n))
        x = g.add(g.matmul(g.swiglu(gate, up), quantized(f"wd.{i}", n, k)), h)
    if case["vocab"]:
        x = g.matmul(norm(x, "norm"), quantized("lm_head", k, case["vocab"]))
    g.set_outputs([x] + outs)
    return g, shapes, norms


def prepare(case, seed):
    kind, fmt, k, n = case["kind"], case["fmt"], case["k"], case["n"]
    if kind == "load":
        w = torch.empty(k, n, device="cuda").normal_(0.0, 0.02, generator=torch.Generator(device="cuda").manual_seed(seed))
        return dict(case=case, program=_Program(seed), w=w.cpu().numpy())
    m = case["m"]
    if kind == "layers":
        g, shapes, norms = _layers_graph(case)
        sess = build_inference_session(g)
        gen = torch.Generator(device="cuda").manual_seed(seed)

        def host(*shape):
            return torch.randn(*shape, generator=gen, device="cuda")

        for name, (rows, cols) in shapes.items():
            sess.set_parameter(name, (host(rows, cols) * 0.02).cpu().numpy())
        for name in norms:
            sess.set_parameter(name, (1 + 0.1 * host(k)).cpu().numpy())
        return dict(case=case, sess=sess, x=host(m, k).cpu().numpy(), attn=host(m, k).cpu().numpy())

    p = _Program(seed)
    s = dict(case=case, program=p)
    if kind == "qkv":
        cols = [n, case["kv"], case["kv"]]
        s.update(x=p.normal((m, k)), norm=p.normal((k,), 0.1, 1.0))
        s["items"] = [(p.weight(fmt, k, c), p.buffer(m * c), None) for c in cols]
        s["out"] = [p.view(c, (m, w.cols)) for w, c, _ in s["items"]]
    elif kind == "gemm":
        f16 = case["act"] == "f16"
        s.update(a=p.normal((m, k), dtype=torch.float16 if f16 else torch.float32), w=p.weight(fmt, k, n), c=p.buffer(m * n),
                 d=p.normal((m, n)) if case["residual"] else None)
        s["out"] = p.view(s["c"], (m, n))
    else:
        gated = kind == "ffn"
        s["stack"] = [(p.normal((k,), 0.1, 1.0) if gated else None, p.weight(fmt, k, 2 * n if gated else n), p.weight(fmt, n, k))
                      for _ in range(case["layers"])]
        s.update(x=[p.normal((m, k))] + [p.buffer(m * k) for _ in s["stack"]], h=p.buffer(m * n * (2 if gated else 1)))
        s["out"] = [p.view(x, (m, k)) for x in s["x"][1:]] + [p.view(s["h"], (m, 2 * n if gated else n))]
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "load":
        w = s["program"].ctx.weight(FMTS[case["fmt"]], s["w"])
        packed = w.export_ref()
        w.free()
        return packed
    m = case["m"]
    if kind == "layers":
        sess = s["sess"]
        sess.set_input("x", s["x"])
        sess.set_input("attn", s["attn"])
        sess.step()
        sess.wait()
        return sess.read_output(m * (case["vocab"] or case["k"]))
    ctx = s["program"].ctx
    if kind == "qkv":
        ctx.matmul_q_batch(s["x"], s["items"], m, capi.PROLOGUE_RMS_NORM, s["norm"], 1e-5)
    elif kind == "gemm":
        (ctx.matmul_q_f16a if case["act"] == "f16" else ctx.matmul_q)(s["a"], s["w"], s["c"], m, s["d"])
    elif kind == "ffn":
        for (norm, up, down), x, y in zip(s["stack"], s["x"], s["x"][1:]):
            ctx.matmul_q_rms_norm(x, norm, 1e-5, up, s["h"], m)
            ctx.matmul_q_swiglu(s["h"], down, y, m, x)
    else:
        for (_, up, down), x, y in zip(s["stack"], s["x"], s["x"][1:]):
            ctx.matmul_q_epilogue(x, up, s["h"], m, [capi.UNARY_SILU])
            ctx.matmul_q(s["h"], down, y, m, x)
    return s["out"]
