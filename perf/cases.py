"""The work this framework is used for, as cases that can be timed: quantized projections of decode and prefill, the
resident runners built on them, and the bulk dequantize of a weight that is loaded.

A case is one of five kinds:

  matmul   one matrix against `tokens` rows of activations through the router (quant.matmul_dev), device buffers in and out
  stack    the projections of a decoder layer (q, k, v, o, gate, up, down) through QwenProjectionStackRunner
  ffn      the FFN half of a decoder layer (add + RMSNorm, gate | up, SwiGLU, down + residual) through FFNSequenceRunner
  head     RMSNorm, vocabulary projection and top-1 through QwenOutputHeadRunner, with or without the logits
  dequant  a raw GGUF tensor to float32 (quant.dequantize_dev)

The runners' decode steps (up to DECODE_TOKENS tokens) are captured once in a HIP graph and replayed, prefills are issued as
they come.
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cogni-ml_amd"))   # the working folder is the root of the tree that is timed

from cogni_ml_amd import hip, quant  # noqa: E402
from cogni_ml_amd.ffn_sequence import FFNSequenceRunner  # noqa: E402
from cogni_ml_amd.output_head import QwenOutputHeadRunner  # noqa: E402
from cogni_ml_amd.output_head import Weights as HeadWeights  # noqa: E402
from cogni_ml_amd.projection_stack import QwenProjectionStackRunner  # noqa: E402
from cogni_ml_amd.projection_stack import Weights as StackWeights  # noqa: E402
from cogni_ml_amd.types import TensorType  # noqa: E402

DECODE_TOKENS = 8


def listed():
    return [
        # the up projection of a small draft model (Q8_0, hidden 1024), one token: the smallest call, all latency
        {"name": "draft_up_1", "kind": "matmul", "type": "Q8_0", "in_dim": 1024, "out_dim": 3584, "tokens": 1},
        # the same model reading a prompt of a couple of hundred tokens
        {"name": "draft_up_200", "kind": "matmul", "type": "Q8_0", "in_dim": 1024, "out_dim": 3584, "tokens": 200},
        # an unquantized (binary16) projection of a file of mixed types, an odd number of tokens
        {"name": "half_33", "kind": "matmul", "type": "F16", "in_dim": 2048, "out_dim": 2048, "tokens": 33},
        # a decoder layer's projections, one token: ordinary decode
        {"name": "stack_1", "kind": "stack", "hidden": 4096, "kv": 1024, "ffn": 12288, "type": "Q4_K", "down": "Q6_K", "tokens": 1},
        # the same for eight sequences in a batch
        {"name": "stack_8", "kind": "stack", "hidden": 4096, "kv": 1024, "ffn": 12288, "type": "Q4_K", "down": "Q6_K", "tokens": 8},
        # a short prompt, a verified draft or a larger batch
        {"name": "stack_48", "kind": "stack", "hidden": 4096, "kv": 1024, "ffn": 12288, "type": "Q4_K", "down": "Q6_K", "tokens": 48},
        # a prompt chunk of the usual size
        {"name": "stack_512", "kind": "stack", "hidden": 4096, "kv": 1024, "ffn": 12288, "type": "Q4_K", "down": "Q6_K", "tokens": 512},
        # the FFN half of a layer for a handful of tokens, an odd number
        {"name": "ffn_13", "kind": "ffn", "hidden": 4096, "ffn": 12288, "down": "Q6_K", "tokens": 13},
        # the same for a long prompt chunk: the largest case
        {"name": "ffn_2048", "kind": "ffn", "hidden": 4096, "ffn": 12288, "down": "Q6_K", "tokens": 2048},
        # the output head of a sampled token: logits and top-1 (510 MB of weights)
        {"name": "head_logits_1", "kind": "head", "type": "Q6_K", "hidden": 4096, "vocab": 151936, "tokens": 1, "logits": True},
        # the output head of a few greedy or verified tokens: top-1 only
        {"name": "head_top1_6", "kind": "head", "type": "Q6_K", "hidden": 4096, "vocab": 151936, "tokens": 6, "logits": False},
        # a weight read to float32
        {"name": "dequant", "kind": "dequant", "type": "Q5_K", "n": 12288 * 4096},
    ]


def _log_uniform(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "matmul", "stack", "ffn", "head", "dequant"])
    if kind == "matmul":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q8_0", "F16", "F32", "IQ4_NL"])
        if t in ("Q4_K", "Q5_K", "Q6_K"):
            return {"kind": kind, "type": t, "in_dim": _log_uniform(rng, 512, 12288, 256), "out_dim": _log_uniform(rng, 256, 12288),
                    "tokens": _log_uniform(rng, 1, 1024)}
        # small models, draft models and single tensors of a mixed file
        return {"kind": kind, "type": t, "in_dim": _log_uniform(rng, 256, 4096, 32), "out_dim": _log_uniform(rng, 256, 4096),
                "tokens": _log_uniform(rng, 1, 256)}
    if kind == "stack":
        hidden = _log_uniform(rng, 1024, 4096, 256)
        return {"kind": kind, "hidden": hidden, "kv": _log_uniform(rng, 256, 1024, 64), "ffn": _log_uniform(rng, 2048, 12288, 256),
                "type": rng.choice(["Q4_K", "Q4_K", "Q5_K"]), "down": rng.choice(["Q6_K", "Q4_K"]), "tokens": _log_uniform(rng, 1, 1024)}
    if kind == "ffn":
        return {"kind": kind, "hidden": _log_uniform(rng, 1024, 4096, 256), "ffn": _log_uniform(rng, 2048, 12288, 256),
                "down": rng.choice(["Q6_K", "Q6_K", "Q4_K"]), "tokens": _log_uniform(rng, 1, 1024)}
    if kind == "head":
        return {"kind": kind, "type": rng.choice(["Q6_K", "Q6_K", "Q4_K"]), "hidden": _log_uniform(rng, 1024, 4096, 256),
                "vocab": _log_uniform(rng, 32000, 151936), "tokens": rng.randint(1, 8), "logits": rng.random() < 0.5}
    return {"kind": kind, "type": rng.choice(["Q4_K", "Q5_K", "Q6_K", "Q8_0", "IQ4_NL", "F16"]),
            "n": _log_uniform(rng, 1 << 16, 12288 * 4096, 256)}


# ---- inputs -------------------------------------------------------------------------------------------------------

_stream = None


def _decode_stream():
    """The one stream this program replays its decode graphs on."""
    global _stream
    if _stream is None:
        _stream = hip.HIPStream()
    return _stream


def _weights(gen, type_name, out_dim, in_dim):
    """Raw bytes of an [out_dim][in_dim] matrix on the GPU: the distributions of cogni_ml_amd.synth."""
    t = TensorType[type_name]

    def scales(n, s):
        return (torch.randn(n, device="cuda", generator=gen).abs() * s).half().view(torch.uint8).view(n, 2)

    if t in (TensorType.F16, TensorType.F32):
        w = torch.randn(out_dim * in_dim, device="cuda", generator=gen) * 0.05
        return (w.half() if t == TensorType.F16 else w).view(torch.uint8)
    nb = out_dim * (-(-in_dim // t.block_elements))
    b = torch.randint(0, 256, (nb, t.block_bytes), dtype=torch.uint8, device="cuda", generator=gen)
    if t == TensorType.Q8_0:
        b[:, 0:2] = scales(nb, 0.01)
        b[:, 2:] = torch.randint(-127, 128, (nb, 32), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
    elif t in (TensorType.Q4_K, TensorType.Q5_K):
        b[:, 0:2] = scales(nb, 0.005)
        b[:, 2:4] = scales(nb, 0.002)
    elif t == TensorType.Q6_K:
        b[:, 192:208] = torch.randint(-32, 32, (nb, 16), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
        b[:, 208:210] = scales(nb, 0.005)
    else:
        b[:, 0:2] = scales(nb, 0.01)
    return b.view(-1)


class _Owner:
    """A runner and its graph; they go when the last that uses them goes (the state, or a tensor over an output)."""

    def __init__(self, runner):
        self.runner, self.graph, self.exec = runner, None, None

    def __del__(self):
        hip.synchronize()
        for o in (self.exec, self.graph, self.runner):
            if o is not None:
                o.close()


class _DeviceArray:
    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner   # a tensor made of this keeps it
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "version": 3}


class _Resident:
    """A runner whose weights and activations are on the GPU, the tensors over its outputs and, for a decode step, its graph."""

    def __init__(self, runner, graph):
        self.runner, self.outputs, self._owner = runner, {}, _Owner(runner)
        runner.upload_weights()
        runner.reset_sequence()
        self._exec = self._stream = None
        if graph:
            self._stream = _decode_stream()
            self._stream.begin_capture()
            with hip.with_stream(self._stream):
                runner.run_sequence()
            self._owner.graph = self._stream.end_capture()
            self._exec = self._owner.exec = self._owner.graph.instantiate()

    def view(self, name, ptr, *shape, typestr="<f4"):
        """A tensor over one of the runner's own output buffers."""
        self.outputs[name] = torch.as_tensor(_DeviceArray(self._owner, ptr, shape, typestr), device="cuda")

    def step(self):
        if self._exec is not None:
            self._exec.launch(self._stream)
        else:
            self.runner.run_sequence()
        return self.outputs


def _init():
    quant.init(0)
    hip.lib().hipGetLastError()   # kernels that init looks up and may not find leave an error behind, which torch would report


def prepare(case, seed):
    _init()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    m = case.get("tokens", 1)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    def host(t):
        return t.cpu().numpy()

    if case["kind"] == "matmul":
        t, i, o = TensorType[case["type"]], case["in_dim"], case["out_dim"]
        nws = quant.gemm_workspace_bytes(t, i, m, o)
        ws = torch.empty(nws, dtype=torch.uint8, device="cuda") if nws else None
        return {"case": case, "type": t, "w": _weights(gen, case["type"], o, i), "x": normal(m, i),
                "out": torch.empty(m, o, device="cuda"), "ws": ws, "nws": nws}
    if case["kind"] == "dequant":
        t, n = TensorType[case["type"]], case["n"]
        return {"case": case, "type": t, "w": _weights(gen, case["type"], 1, n), "out": torch.empty(n, device="cuda")}
    if case["kind"] == "stack":
        h, kv, f, t = case["hidden"], case["kv"], case["ffn"], case["type"]
        layout = [("q", "x", t, h, h), ("k", "x", t, kv, h), ("v", "x", t, kv, h), ("o", "q", t, h, h),
                  ("gate", "x", t, f, h), ("up", "x", t, f, h), ("down", "gate", case["down"], h, f)]
        w = StackWeights(h, [(n, src, TensorType[tt], o, i, host(_weights(gen, tt, o, i))) for n, src, tt, o, i in layout])
        r = _Resident(QwenProjectionStackRunner.from_weights(w, m, host(normal(m * h))), m <= DECODE_TOKENS)
        for n, src, tt, o, i in layout:
            r.view(n, r.runner.device_ptr(n), m, o)
        return r
    if case["kind"] == "ffn":
        h, f = case["hidden"], case["ffn"]
        raw = [host(_weights(gen, "Q4_K", f, h)), host(_weights(gen, "Q4_K", f, h)), host(_weights(gen, case["down"], h, f))]
        # activations that leave silu(gate) * up of order 1, as behind a trained norm
        norm = host(0.02 * (1.0 + 0.1 * normal(h)))
        r = _Resident(FFNSequenceRunner(*raw, h, f, m, host(normal(m * h)), down_type=TensorType[case["down"]], norm=norm,
                                        add=host(normal(m * h))), m <= DECODE_TOKENS)
        r.view("combined", r.runner._act.ptr, m, f)
        r.view("out", r.runner._out.ptr, m, h)
        return r
    h, v = case["hidden"], case["vocab"]
    w = HeadWeights(host(1.0 + 0.1 * normal(h)), host(_weights(gen, case["type"], v, h)), TensorType[case["type"]], h, v)
    r = _Resident(QwenOutputHeadRunner.from_weights(w, m, host(normal(m * h)), 1.0e-6, read_logits=case["logits"]), True)
    r.view("top1_ids", r.runner.top1_ids_device_ptr, m, typestr="<i4")
    r.view("top1_values", r.runner._top1_values.ptr, m)
    if case["logits"]:
        r.view("logits", r.runner._logits.ptr, m, v)
    return r


def run(state):
    if isinstance(state, _Resident):
        return state.step()
    c, out = state["case"], state["out"]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if c["kind"] == "dequant":
        quant.dequantize_dev(state["w"].data_ptr(), state["type"], c["n"], out.data_ptr(), stream)
    else:
        ws = state["ws"]
        quant.matmul_dev(state["w"].data_ptr(), state["type"], state["x"].data_ptr(), out.data_ptr(), c["in_dim"], c["out_dim"],
                         c["tokens"], ws.data_ptr() if ws is not None else 0, state["nws"], 0, stream)
    return out


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def _matrix_bytes(type_name, out_dim, in_dim):
    return TensorType[type_name].data_bytes(in_dim) * out_dim


def work(case):
    m = case.get("tokens", 1)
    if case["kind"] == "dequant":
        return {"bytes": _matrix_bytes(case["type"], 1, case["n"]) + 4 * case["n"], "flops": case["n"]}
    if case["kind"] == "matmul":
        i, o = case["in_dim"], case["out_dim"]
        return {"bytes": _matrix_bytes(case["type"], o, i) + 4 * m * (i + o), "flops": 2 * m * i * o}
    if case["kind"] == "head":
        h, v = case["hidden"], case["vocab"]
        return {"bytes": _matrix_bytes(case["type"], v, h) + 4 * m * h + 4 * h + 8 * m + (4 * m * v if case["logits"] else 0),
                "flops": 2 * m * h * v}
    h, f = case["hidden"], case["ffn"]
    if case["kind"] == "ffn":
        # x, the addend and the norm in; the products and the block's output out
        return {"bytes": 2 * _matrix_bytes("Q4_K", f, h) + _matrix_bytes(case["down"], h, f) + 4 * (2 * m * h + h) + 4 * m * (f + h),
                "flops": 2 * m * 3 * h * f}
    kv, t = case["kv"], case["type"]
    return {"bytes": 2 * _matrix_bytes(t, h, h) + 2 * _matrix_bytes(t, kv, h) + 2 * _matrix_bytes(t, f, h) + _matrix_bytes(case["down"], h, f) +
            4 * m * h + 4 * m * (3 * h + 2 * kv + 2 * f), "flops": 2 * m * (2 * h * h + 2 * kv * h + 3 * f * h)}


def tolerance(case):
    m = case.get("tokens", 1)
    if case["kind"] == "dequant":
        return "exact"
    k_quant = case.get("type") in ("Q4_K", "Q5_K", "Q6_K") or case["kind"] == "ffn"
    if m > DECODE_TOKENS and k_quant and case["kind"] != "head":
        # activations and dequantized weights rounded to binary16, sums in 32 bits (a projection of a projection twice)
        return {"rel": 2.0e-3, "max": 0.04}
    # 32-bit sums of up to 12288 products
    return {"rel": 1.0e-5, "max": 4.0e-4}
