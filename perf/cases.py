"""The work a user of this framework has it do, as measurable cases.

Every case is one pass through the public Python entry points (`QLinear`,
`QTensor`, `hip`, `kir.HipGraph`, `CharLM`) on tensors that are already on the
GPU.  A case's "kind" names the path, the other entries its sizes and options;
`listed()` gives one ordinary case of each, `draw()` others of the same ranges,
odd and ragged sizes among them.

Activations are normal with a few large channels, weights N(0, 0.02) with a few
large columns, which is what makes per-token and per-channel scales differ.
"""

from __future__ import annotations

import math
import types

import numpy as np
import torch

from kansaiml_amd import hip, kir
from kansaiml_amd.charlm import CharLM, CharLMWeights
from kansaiml_amd.device import DeviceTensor
from kansaiml_amd.quantize import QLinear, QTensor

VOCAB, D_MODEL, HEADS, LAYERS, D_FF, BLOCK = 65, 384, 6, 6, 1536, 256  # the char-LM's configuration
HEAD_DIM = 64


def listed():
    return [
        # The smallest int8 Linear the framework is configured for: a batch of 64 rows of a small
        # model's layer with one activation scale, called eagerly (latency and host work count).
        {"name": "linear_small", "kind": "linear", "M": 64, "K": 512, "N": 512, "gran": "tensor"},
        # A decode step's up-projection for eight sequences, one scale per token: the weight stream.
        {"name": "linear_decode", "kind": "linear", "M": 8, "K": 4096, "N": 11008, "gran": "row"},
        # A prompt of 300 tokens through a square layer, one scale per token.
        {"name": "linear_prompt", "kind": "linear", "M": 300, "K": 4096, "N": 4096, "gran": "row"},
        # A layer whose sizes are no multiple of anything, as small classifiers have them.
        {"name": "linear_ragged", "kind": "linear", "M": 1000, "K": 1001, "N": 1250, "gran": "tensor"},
        # A decode step's MLP (up, GELU, down, residual) for four sequences, recorded once and replayed.
        {"name": "mlp_decode", "kind": "mlp", "M": 4, "D": 4096, "F": 11008},
        # The largest product: int8 codes that stay on the device, per-channel weight scales.
        {"name": "gemm_large", "kind": "gemm", "M": 8192, "K": 8192, "N": 8192, "gran": "tensor"},
        # Post-training quantization of an activation dump and back, one scale per row.
        {"name": "quant_round", "kind": "quant", "rows": 16384, "cols": 16384, "gran": "row"},
        # Loading a layer: its fp32 weight quantized per output channel and packed for the product.
        {"name": "weight_load", "kind": "weight", "K": 4096, "N": 11008, "gran": "col"},
        # The reference's own quantized Linear (int8 weight, fp32 product) on a small batch.
        {"name": "weight_only", "kind": "weight_only", "M": 64, "K": 4096, "N": 4096},
        # The fp32 product of a layer that is not quantized.
        {"name": "matmul_f32", "kind": "matmul", "M": 2000, "K": 2048, "N": 4096},
        # Attention over a longer context than the char-LM's, causal.
        {"name": "attention", "kind": "attention", "B": 4, "T": 1000, "H": 12, "mask": "causal"},
        # The whole quantized char-LM on a full batch, recorded once and replayed.
        {"name": "charlm", "kind": "charlm", "batch": 64, "seq": 256, "gran": "tensor"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi, by its logarithm: a multiple of 64, of 8, or any."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(lo, min(hi, (v + step // 2) // step * step))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "mlp", "gemm", "quant", "weight", "weight_only", "matmul",
                       "attention", "charlm"))
    while True:
        c = _draw(rng, kind)
        if c is not None:
            return c


def _draw(rng, kind):
    if kind == "linear":
        c = {"kind": kind, "M": _log(rng, 1, 4096), "K": _size(rng, 64, 11008), "N": _size(rng, 64, 11008),
             "gran": rng.choice(("row", "row", "tensor"))}
        return c if c["M"] * c["K"] * c["N"] <= 1 << 34 else None
    if kind == "mlp":
        return {"kind": kind, "M": _log(rng, 1, 64), "D": _size(rng, 256, 4096), "F": _size(rng, 512, 11008)}
    if kind == "gemm":
        c = {"kind": kind, "M": _size(rng, 512, 8192), "K": _size(rng, 512, 8192), "N": _size(rng, 512, 8192),
             "gran": rng.choice(("tensor", "row"))}
        return c if c["M"] * c["K"] * c["N"] <= 1 << 36 else None
    if kind == "quant":
        c = {"kind": kind, "rows": _log(rng, 1, 16384), "cols": _size(rng, 64, 16384),
             "gran": rng.choice(("row", "tensor"))}
        return c if c["rows"] * c["cols"] <= 1 << 27 else None
    if kind == "weight":
        return {"kind": kind, "K": _size(rng, 64, 8192), "N": _size(rng, 64, 11008),
                "gran": rng.choice(("col", "tensor"))}
    if kind == "weight_only":
        c = {"kind": kind, "M": _log(rng, 1, 2048), "K": _size(rng, 64, 4096), "N": _size(rng, 64, 4096)}
        return c if c["M"] * c["K"] * c["N"] <= 1 << 33 else None
    if kind == "matmul":
        c = {"kind": kind, "M": _log(rng, 1, 4096), "K": _size(rng, 64, 4096), "N": _size(rng, 64, 4096)}
        return c if c["M"] * c["K"] * c["N"] <= 1 << 34 else None
    if kind == "attention":
        c = {"kind": kind, "B": _log(rng, 1, 64), "T": _log(rng, 1, 1500), "H": rng.choice((1, 4, 6, 12)),
             "mask": rng.choice(("causal", "causal", "none", "padding"))}
        return c if c["B"] * c["H"] * c["T"] * c["T"] <= 1 << 26 else None
    seq = rng.choice((BLOCK, _log(rng, 2, BLOCK)))
    return {"kind": kind, "batch": _log(rng, 1, 64), "seq": seq, "gran": rng.choice(("tensor", "row"))}


# ---------------------------------------------------------------------------
# Tensors on the device: torch makes the values, the framework's own buffers
# hold them, and outputs are seen by torch without a copy.
# ---------------------------------------------------------------------------

_TYPESTR = {"float32": "<f4", "int8": "|i1", "int32": "<i4", "float64": "<f8"}


class _Array:
    """A DeviceTensor's memory in the array interface's terms (it keeps the buffer alive)."""

    def __init__(self, t):
        self.t = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": _TYPESTR[t.dtype],
                                         "data": (t.addr, False), "strides": None, "version": 2}


def _see(t):
    return torch.as_tensor(_Array(t), device="cuda")


def _put(x):
    """A torch tensor's values in a buffer of the framework's (its stream is another than torch's)."""
    t = DeviceTensor(list(x.shape), str(x.dtype).replace("torch.", ""))
    torch.cuda.synchronize()
    _see(t).copy_(x)
    torch.cuda.synchronize()
    return t


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(seed * 16 + what)


def _activation(shape, seed, what=0):
    g = _gen(seed, what)
    x = torch.randn(shape, generator=g, device="cuda")
    return x * torch.where(torch.rand(shape[-1], generator=g, device="cuda") < 0.01, 8.0, 1.0)


def _weight(k, n, seed, what=1):
    g = _gen(seed, what)
    w = torch.randn((k, n), generator=g, device="cuda") * 0.02
    return w * torch.where(torch.rand(n, generator=g, device="cuda") < 0.005, 20.0, 1.0)


def _bias(n, seed, what=2):
    return torch.randn(n, generator=_gen(seed, what), device="cuda") * 0.1


def _codes(rows, cols, seed, what):
    """Codes of normal values: the largest of a row is about four sigma."""
    v = torch.randn((rows, cols), generator=_gen(seed, what), device="cuda") * 30.0
    return v.round_().clamp_(-127, 127).to(torch.int8)


def _scales(n, seed, what):
    return (torch.rand(n, generator=_gen(seed, what), device="cuda", dtype=torch.float64) + 0.5) * 1e-3


def _mask(c):
    """Key padding: sequence b ends after its share of the positions (additive, -inf past it)."""
    ends = torch.linspace(1, c["T"], c["B"], device="cuda").long().view(-1, 1, 1, 1)
    m = torch.zeros((c["B"], 1, 1, c["T"]), device="cuda")
    return m.masked_fill_(torch.arange(c["T"], device="cuda") >= ends, -math.inf)


def _linear(k, n, seed, mode="int8", act="tensor", weight="col", what=1):
    weights = types.SimpleNamespace(weight=_put(_weight(k, n, seed, what)), bias=_put(_bias(n, seed, what + 1)))
    return QLinear(weights, mode=mode, act_granularity=act, weight_granularity=weight)


def _charlm_weights(seed):
    """The configuration's own initialisation, the projections that write the residual stream scaled
    down by the square root of their number, as decoders are commonly initialised."""
    w = CharLMWeights(VOCAB, D_MODEL, HEADS, LAYERS, D_FF, BLOCK, seed=seed, bias_std=0.02)
    for block in w.blocks:
        for key in ("w_o", "fc2_w"):
            block[key] *= np.float32(1.0 / math.sqrt(2 * LAYERS))
    return w


def _ids(c, seed):
    return np.random.default_rng(seed).integers(0, VOCAB, (c["batch"], c["seq"]), dtype=np.int32)


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        # One layer of a user's model and its input.
        layer, x = _linear(c["K"], c["N"], seed, act=c["gran"]), _put(_activation((c["M"], c["K"]), seed))
        return lambda: _see(layer(x))
    if kind == "mlp":
        up, down = _linear(c["D"], c["F"], seed, act="row"), _linear(c["F"], c["D"], seed, act="row", what=3)
        x = _put(_activation((c["M"], c["D"]), seed))
        graph = kir.quant_fusion(kir.trace(lambda v: v.add(down(up(v).gelu())), np.zeros(x.shape, np.float32)),
                                 producer_quant="layer_norm", qload=True)
        replay = kir.HipGraph(graph, kir.plan_memory(graph), x)
        torch.cuda.synchronize()
        return lambda: _see(replay(x, to_host=False))
    if kind == "gemm":
        a, b = _put(_codes(c["M"], c["K"], seed, 0)), _put(_codes(c["N"], c["K"], seed, 1))
        sa, sb = _put(_scales(c["M"] if c["gran"] == "row" else 1, seed, 2)), _put(_scales(c["N"], seed, 3))
        bias = _put(_bias(c["N"], seed, 4))
        return lambda: _see(hip.gemm_i8(a, b, sa, sb, bias)[0])
    if kind == "quant":
        x = _put(_activation((c["rows"], c["cols"]), seed))
        there, back = ((hip.quantize_rows, hip.dequantize_rows) if c["gran"] == "row" else
                       (hip.quantize_tensor, hip.dequantize_tensor))

        def both():
            q, s = there(x)
            return _see(q), _see(s), _see(back(q, s))
        return both
    if kind == "weight":
        w = _put(_weight(c["K"], c["N"], seed))

        def load():
            q = QTensor.from_weight(w, c["gran"])
            return _see(q.codes), _see(q.scales)
        return load
    if kind == "weight_only":
        layer = _linear(c["K"], c["N"], seed, mode="weight_only", weight="tensor")
        x = _put(_activation((c["M"], c["K"]), seed))
        return lambda: _see(layer(x))
    if kind == "matmul":
        a, b = _put(_activation((c["M"], c["K"]), seed)), _put(_weight(c["K"], c["N"], seed))
        bias = _put(_bias(c["N"], seed))
        return lambda: _see(hip.matmul(a, b, bias))
    if kind == "attention":
        d = c["H"] * HEAD_DIM
        qkv = _put(torch.randn((c["B"] * c["T"], 3 * d), generator=_gen(seed, 0), device="cuda"))
        mask = _put(_mask(c)) if c["mask"] == "padding" else None
        return lambda: _see(hip.attention(qkv, c["B"], c["T"], c["H"], d, causal=c["mask"] == "causal", mask=mask)[0])
    model = CharLM(_charlm_weights(seed), act_granularity=c["gran"])
    replay = model.capture(c["batch"], c["seq"])
    ids = DeviceTensor.from_host(_ids(c, seed))
    torch.cuda.synchronize()
    return lambda: _see(replay(ids, to_host=False))


def run(state):
    return state()


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * M * K + K * N + 12 * N + 4 * M * N, "flops": 2 * M * K * N}
    if kind == "mlp":
        M, D, F = c["M"], c["D"], c["F"]
        return {"bytes": 8 * M * D + 2 * D * F + 12 * (D + F), "flops": 4 * M * D * F}
    if kind == "gemm":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": M * K + K * N + 4 * M * N + 12 * N + 8 * (M if c["gran"] == "row" else 1),
                "flops": 2 * M * K * N}
    if kind == "quant":
        n = c["rows"] * c["cols"]
        return {"bytes": 9 * n + 8 * (c["rows"] if c["gran"] == "row" else 1), "flops": 4 * n}
    if kind == "weight":
        n = c["K"] * c["N"]
        return {"bytes": 5 * n + 8 * (c["N"] if c["gran"] == "col" else 1), "flops": 3 * n}
    if kind == "weight_only":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * M * K + K * N + 4 * N + 4 * M * N, "flops": 2 * M * K * N}
    if kind == "matmul":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * (M * K + K * N + N + M * N), "flops": 2 * M * K * N}
    if kind == "attention":
        B, T, H = c["B"], c["T"], c["H"]
        pairs = T * (T + 1) // 2 if c["mask"] == "causal" else T * T
        return {"bytes": 16 * B * T * H * HEAD_DIM, "flops": 4 * B * H * HEAD_DIM * pairs}
    rows = c["batch"] * c["seq"]
    weights = LAYERS * (4 * D_MODEL * D_MODEL + 2 * D_MODEL * D_FF) + D_MODEL * VOCAB
    pairs = c["seq"] * (c["seq"] + 1) // 2 if c["seq"] == BLOCK else c["seq"] ** 2
    return {"bytes": 4 * rows + weights + 4 * rows * VOCAB,
            "flops": 2 * rows * weights + LAYERS * 4 * c["batch"] * D_MODEL * pairs}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "weight"):
        return "exact"  # codes, scales and dequantized values are defined to the bit
    # Below: about four times what each path is off `exact`.
    if kind in ("linear", "gemm"):
        return {"rel": 1.5e-7, "max": 1e-6}  # exact int32 sums, rounded to binary32 once and by the bias add
    if kind in ("weight_only", "matmul"):
        return {"rel": 5e-6, "max": 2e-4}  # binary32 sums of up to 4096 products, in any order
    if kind == "attention":
        return {"rel": 2.5e-6, "max": 3e-5}  # binary32 products, sums and exponentials
    # A value whose rounding differs in one bit can take the next code in the quantize that follows;
    # through six layers such codes move the logits by up to 0.026 of their norm (one scale per tensor).
    return {"rel": 1e-4, "max": 4e-3} if kind == "mlp" else {"rel": 3e-2, "max": 0.6}


# ---------------------------------------------------------------------------
# The same in 64 bits, by torch alone
# ---------------------------------------------------------------------------

def _quantized(x, dim=None):
    """quantize -> (codes, scale) in float64; dim: the axis that one scale covers, None for all."""
    m = x.abs().amax() if dim is None else x.abs().amax(dim, keepdim=True)
    s = torch.where(m > 0, m.double() / 127.0, 1.0)
    return (x.double() / s).round().clamp(-127, 127), s


def _linear64(x, w, bias, gran):
    q, sx = _quantized(x, 1 if gran == "row" else None)
    p, sw = _quantized(w, 0)
    y = (q @ p) * (sx * sw)
    return y if bias is None else y + bias.double()


def _gelu64(y):
    return 0.5 * y * (1.0 + torch.erf(y / math.sqrt(2.0)))


def _attention64(qkv, B, T, H, causal, mask):
    q, k, v = (t.contiguous() for t in qkv.double().view(B, T, 3, H, HEAD_DIM).permute(2, 0, 3, 1, 4))
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(HEAD_DIM)
    if causal:
        s = s.masked_fill(torch.ones((T, T), dtype=torch.bool, device=s.device).triu(1), -math.inf)
    if mask is not None:
        s = s + mask.double()
    return torch.matmul(s.softmax(-1), v).permute(0, 2, 1, 3).reshape(B * T, H * HEAD_DIM)


def _layer_norm64(x, w, b):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * w + b


def _charlm64(c, seed):
    w = _charlm_weights(seed)

    def up(a):
        return torch.from_numpy(a).cuda()
    ids = torch.from_numpy(_ids(c, seed)).cuda().long()
    x = (up(w.tok)[ids] + up(w.pos)[: c["seq"]]).reshape(-1, D_MODEL).double()
    for b in w.blocks:
        h = _layer_norm64(x, up(b["ln1_w"]), up(b["ln1_b"]))
        qkv = _linear64(h, torch.cat([up(b["w_q"]), up(b["w_k"]), up(b["w_v"])], 1), None, c["gran"])
        a = _attention64(qkv, c["batch"], c["seq"], HEADS, c["seq"] == BLOCK, None)
        x = x + _linear64(a, up(b["w_o"]), None, c["gran"])
        h = _layer_norm64(x, up(b["ln2_w"]), up(b["ln2_b"]))
        h = _gelu64(_linear64(h, up(b["fc1_w"]), up(b["fc1_b"]), c["gran"]))
        x = x + _linear64(h, up(b["fc2_w"]), up(b["fc2_b"]), c["gran"])
    x = _layer_norm64(x, up(w.lnf_w), up(w.lnf_b))
    return _linear64(x, up(w.head_w), up(w.head_b), c["gran"])


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        return _linear64(_activation((c["M"], c["K"]), seed), _weight(c["K"], c["N"], seed), _bias(c["N"], seed),
                         c["gran"])
    if kind == "mlp":
        x = _activation((c["M"], c["D"]), seed)
        h = _gelu64(_linear64(x, _weight(c["D"], c["F"], seed), _bias(c["F"], seed), "row"))
        return x.double() + _linear64(h, _weight(c["F"], c["D"], seed, 3), _bias(c["D"], seed, 4), "row")
    if kind == "gemm":
        a, b = _codes(c["M"], c["K"], seed, 0).double(), _codes(c["N"], c["K"], seed, 1).double()
        sa = _scales(c["M"] if c["gran"] == "row" else 1, seed, 2).view(-1, 1)
        return (a @ b.T) * (sa * _scales(c["N"], seed, 3)) + _bias(c["N"], seed, 4).double()
    if kind == "quant":
        q, s = _quantized(_activation((c["rows"], c["cols"]), seed), 1 if c["gran"] == "row" else None)
        return q.to(torch.int8), s.reshape(-1), q * s
    if kind == "weight":
        q, s = _quantized(_weight(c["K"], c["N"], seed), 0 if c["gran"] == "col" else None)
        return q.to(torch.int8).T.contiguous(), s.reshape(-1)
    if kind == "weight_only":
        q, s = _quantized(_weight(c["K"], c["N"], seed))
        return _activation((c["M"], c["K"]), seed).double() @ (q * s) + _bias(c["N"], seed).double()
    if kind == "matmul":
        return (_activation((c["M"], c["K"]), seed).double() @ _weight(c["K"], c["N"], seed).double()
                + _bias(c["N"], seed).double())
    if kind == "attention":
        qkv = torch.randn((c["B"] * c["T"], 3 * c["H"] * HEAD_DIM), generator=_gen(seed, 0), device="cuda")
        return _attention64(qkv, c["B"], c["T"], c["H"], c["mask"] == "causal",
                            _mask(c) if c["mask"] == "padding" else None)
    return _charlm64(c, seed)
