"""The calls that a program of this framework makes, as timed cases.

Three kinds, all at the geometry of the routed-expert layer this repository is
built and benchmarked for (128 experts, top-8, hidden 2048, expert
intermediate 768):

* ``layer``  -- router top-k and routed experts of one decoder layer
  (``forward_routed`` of the FP8 or packed backend).  A decode step runs the
  layers of a model back to back for a few tokens, from a hipGraph, as a
  serving loop does (``layers`` > 1: each layer has its own bank); a prefill
  call is one eager layer call on one bank.
* ``linear`` -- the dense W4A16 ``GPTQLinear`` (the attention projections of a
  GPTQ checkpoint).
* ``shared`` -- the dense half of the MoE block: router logits, the gated
  shared expert and the residual adds around given expert outputs
  (``MoeBlock.pre`` and ``MoeBlock.post``).
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "drama3-studio_amd")
for _place in ("drama3-studio_amd", _PACKAGE):  # the tree in the working folder first
    if Path(_place, "drama_moe").is_dir():
        sys.path.insert(0, str(Path(_place).resolve()))
        break

EXPERTS, TOP_K, HIDDEN, INTER = 128, 8, 2048, 768
SHARED_INTER = 768
MODES = {"w4a16": 0, "w4a16-asym": 0, "int8": 1, "w6a8": 2, "w4a8-book": 3, "w4a8-g128": 4, "w6a8-g128": 5}
FP8 = ("fp8-block", "fp8-channel")
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}

# bytes of one expert: codes and scales of w13 and w2
_VALUES = 3 * INTER * HIDDEN
_ROWS = 2 * INTER + HIDDEN
EXPERT_BYTES = {
    "fp8-block": _VALUES + _VALUES // (128 * 128) * 4,
    "fp8-channel": _VALUES + _ROWS * 4,
    "w4a16": _VALUES // 2 + _VALUES // 128 * 2,
    "w4a16-asym": _VALUES // 2 + _VALUES // 128 * 2 + _VALUES // 128 // 2,
    "int8": _VALUES + _ROWS * 4,
    "w6a8": _VALUES * 3 // 4 + _VALUES // 16 + _ROWS * 4,
    "w4a8-book": _VALUES // 2 + _VALUES // 16 + _ROWS * 8,
    "w4a8-g128": _VALUES // 2 + _VALUES // 128 * 2,
    "w6a8-g128": _VALUES * 3 // 4 + _VALUES // 128 * 2,
}


def _layer(name, fmt, tokens, *, layers=1, routing="zipf", x_group="token", dtype="bf16"):
    case = {"kind": "layer", "fmt": fmt, "tokens": tokens, "layers": layers, "routing": routing, "dtype": dtype}
    if fmt in FP8:
        case["x_group"] = x_group
    return {"name": name, **case} if name else case


def listed():
    return [
        # one stream of speech being generated: a decode step, one token through
        # consecutive layers, the FP8 model
        _layer("decode-fp8-1", "fp8-channel", 1, layers=8, routing="uniform", x_group="128"),
        # the same with the smallest model format
        _layer("decode-w4a8-g128-1", "w4a8-g128", 1, layers=8, routing="uniform"),
        # three streams at once from a GPTQ checkpoint
        _layer("decode-w4a16-3", "w4a16", 3, layers=8, routing="uniform"),
        # a batched decode step of 13 streams, official block-scaled FP8 weights
        _layer("decode-fp8-block-13", "fp8-block", 13, layers=4, routing="uniform", x_group="128"),
        # a short prompt and a long one through the FP8 layer
        _layer("prefill-fp8-block-333", "fp8-block", 333, x_group="128"),
        _layer("prefill-fp8-2048", "fp8-channel", 2048),
        # prompts through the packed formats
        _layer("prefill-w4a16-asym-512", "w4a16-asym", 512, routing="uniform"),
        _layer("prefill-int8-197", "int8", 197),
        _layer("prefill-w6a8-512", "w6a8", 512, routing="uniform"),
        _layer("prefill-w6a8-g128-301", "w6a8-g128", 301),
        # an attention projection of a GPTQ checkpoint over a prompt
        {"name": "linear-1024", "kind": "linear", "tokens": 1024, "n": 4096, "k": 2048, "dtype": "bf16"},
        # router, shared expert and residuals of a prompt
        {"name": "shared-509", "kind": "shared", "tokens": 509},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "linear", "shared"])
    routing = rng.choice(["zipf", "uniform"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "linear":
        return {"kind": "linear", "tokens": _log_int(rng, 1, 1024), "n": rng.choice([512, 2048, 4096]),
                "k": rng.choice([1024, 2048]), "dtype": dtype}
    if kind == "shared":
        return {"kind": "shared", "tokens": _log_int(rng, 1, 1024)}
    fmt = rng.choice(list(FP8) + list(MODES))
    x_group = rng.choice(["128", "token"])
    if kind == "decode":
        return _layer(None, fmt, _log_int(rng, 1, 24), layers=rng.choice([2, 3, 4]), routing=routing,
                      x_group=x_group, dtype=dtype)
    return _layer(None, fmt, _log_int(rng, 25, 2000 if fmt in FP8 else 600), routing=routing, x_group=x_group,
                  dtype=dtype)


# --------------------------------------------------------------------- inputs

def _generator(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed))


def _logits(tokens, routing, g, device):
    """Router logits of distinct experts per token: equally likely ones, or
    Zipf(1.1) popularity over a random ranking (log p + Gumbel noise)."""
    if routing == "uniform":
        return torch.randn(tokens, EXPERTS, generator=g, device=device)
    ranks = torch.randperm(EXPERTS, generator=g, device=device).double() + 1
    u = torch.rand(tokens, EXPERTS, generator=g, device=device, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    return (-1.1 * torch.log(ranks) - torch.log(-torch.log(u))).float()


def _bank(fmt, g, device):
    from drama_moe import formats

    if fmt in FP8:
        return formats.random_fp8_bank(EXPERTS, HIDDEN, INTER, layout=fmt[4:], generator=g, device=device)
    return formats.random_quantized_bank(MODES[fmt], EXPERTS, HIDDEN, INTER, asymmetric=fmt.endswith("asym"),
                                         generator=g, device=device)


def _layer_inputs(case, seed, layer):
    """(bank, x, logits) of one layer."""
    device = torch.device("cuda")
    g = _generator(seed * 1000 + layer, device)
    bank = _bank(case["fmt"], g, device)
    x = torch.randn(case["tokens"], HIDDEN, generator=g, device=device).to(DTYPES[case["dtype"]])
    return bank, x, _logits(case["tokens"], case["routing"], g, device)


def _linear_inputs(case, seed):
    device = torch.device("cuda")
    g = _generator(seed, device)
    n, k = case["n"], case["k"]
    words = torch.randint(-(1 << 31), 1 << 31, (k // 8, n), generator=g, device=device, dtype=torch.int64).int()
    scales = ((torch.rand(k // 128, n, generator=g, device=device) * 0.5 + 0.75) * (0.02 * 2.5 / 8)).half()
    x = torch.randn(case["tokens"], k, generator=g, device=device).to(DTYPES[case["dtype"]])
    return words, scales, x


def _shared_inputs(case, seed):
    device = torch.device("cuda")
    g = _generator(seed, device)

    def rand(rows, cols, std):
        return (torch.randn(rows, cols, generator=g, device=device) * std).bfloat16()

    weights = [rand(EXPERTS, HIDDEN, 0.02), rand(1, HIDDEN, 0.02), rand(SHARED_INTER, HIDDEN, 0.02),
               rand(SHARED_INTER, HIDDEN, 0.02), rand(HIDDEN, SHARED_INTER, 0.02)]
    rows = [rand(case["tokens"], HIDDEN, std) for std in (1.0, 0.3, 1.0)]  # x, experts' output, after_mixer
    return weights, rows


def prepare(case, seed):
    if case["kind"] == "linear":
        from drama_moe.quantized import GPTQLinear

        words, scales, x = _linear_inputs(case, seed)
        return {"case": case, "linear": GPTQLinear(words, scales, device=x.device, dtype=x.dtype), "x": x}
    if case["kind"] == "shared":
        from drama_moe.block import MoeBlock

        weights, (x, experts_out, after_mixer) = _shared_inputs(case, seed)
        return {"case": case, "block": MoeBlock(*weights, None, None, top_k=TOP_K), "x": x,
                "experts_out": experts_out, "after_mixer": after_mixer}
    if case["fmt"] in FP8:
        from drama_moe.offload import HipExpertBackend

        backend = HipExpertBackend(x_group=128 if case["x_group"] == "128" else "token")
    else:
        from drama_moe.quantized import QuantizedExpertBackend

        backend = QuantizedExpertBackend(MODES[case["fmt"]])
    state = {"case": case, "backend": backend,
             "layers": [_layer_inputs(case, seed, layer) for layer in range(case["layers"])]}
    if case["layers"] > 1:  # a decode step is captured once and replayed
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _step(state)  # grows the workspace outside the capture
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=stream):
            state["out"] = _step(state)
    return state


def _step(state):
    return [state["backend"].forward_routed(x, logits, TOP_K, bank) for bank, x, logits in state["layers"]]


def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        return state["linear"](state["x"])
    if kind == "shared":
        block = state["block"]
        logits, sgate, act = block.pre(state["x"])
        out = block.post(act, sgate, state["experts_out"], state["after_mixer"])
        return logits, sgate, act, out
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _step(state)


# ----------------------------------------------------------------------- work

def work(case):
    tokens = case["tokens"]
    if case["kind"] == "linear":
        n, k = case["n"], case["k"]
        return {"bytes": n * k // 2 + n * k // 128 * 2 + tokens * (n + k) * 2, "flops": 2 * tokens * n * k}
    if case["kind"] == "shared":
        weights = (EXPERTS + 1 + 3 * SHARED_INTER) * HIDDEN
        # x, experts' output, residual in; logits, gate, act, layer output out
        rows = tokens * (4 * HIDDEN * 2 + EXPERTS * 4 + 2 + SHARED_INTER * 2)
        return {"bytes": weights * 2 + rows, "flops": 2 * tokens * weights}
    g = _generator(17, "cpu")
    picked = _logits(tokens, case["routing"], g, "cpu").topk(TOP_K, dim=-1).indices
    experts = int(torch.unique(picked).numel())  # of one sample of the routing
    rows = tokens * (2 * HIDDEN * 2 + EXPERTS * 4 + TOP_K * (8 + 2))  # x, logits in; output, ids, weights out
    return {"bytes": case["layers"] * (experts * EXPERT_BYTES[case["fmt"]] + rows),
            "flops": case["layers"] * 2 * tokens * TOP_K * _VALUES}


def tolerance(case):
    # About four times what the outputs show against exact(): bf16 roundings
    # (1.7e-3), and for the layers also quantization codes of single hidden
    # values that fall to the other side (up to 3e-3 together).
    return {"rel": 1.2e-2 if case["kind"] == "layer" else 7e-3}


# ---------------------------------------------------------------------- exact
# The same arithmetic in 64 bits: the quantizers and the storage types of the
# formats (they define the result) are kept, every sum, product and SiLU is
# taken in float64.

def _bf16(v):
    return v.to(torch.bfloat16).double()


def _silu(v):
    return v / (1 + torch.exp(-v))


def _fp8_rows(v, group):
    """Rows quantized to E4M3 with one scale per `group` values, decoded.  The
    format fixes the scale, amax * fl(1 / 448), and the quotient as float32
    values: bf16 rows meet E4M3 midpoints often, and they decide those."""
    blocks = v.reshape(v.shape[0], -1, group).float()
    scale = blocks.abs().amax(-1, keepdim=True).clamp_min(1e-10) * torch.tensor(1 / 448, dtype=torch.float32)
    q = (blocks / scale).clamp(-448, 448).to(torch.float8_e4m3fn).double()
    return (q * scale.double()).reshape(v.shape)


def _hadamard(device):
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64,
                      device=device)
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return h / 16


def _int8_rows(v, dtype):
    """Rows rotated by the 256-point Hadamard basis, rounded to their storage
    type and quantized to INT8 per row, decoded."""
    rotated = (v.reshape(-1, 256) @ _hadamard(v.device)).to(dtype).double().reshape(v.shape)
    scale = rotated.abs().amax(-1, keepdim=True).clamp_min(1e-12).float() / 127
    return (rotated.float() / scale).round().clamp(-127, 127).double() * scale.double()


def _nibbles(raw):
    return torch.stack((raw & 15, raw >> 4), -1).flatten(-2)


def _words(words):
    """int32 words -> their eight nibbles, lowest first, along the last axis."""
    w = words.long() & 0xFFFFFFFF
    return ((w[..., None] >> (torch.arange(8, device=w.device) * 4)) & 15).flatten(-2)


def _matrix(fmt, weight, scale, zeros, dtype):
    """float64 weights [N, K] of one expert."""
    if fmt in FP8:
        w = weight.double()
        n, k = w.shape
        rows, cols = n // scale.shape[0], k // scale.shape[1]
        return w * scale.double().repeat_interleave(rows, 0).repeat_interleave(cols, 1)
    mode = MODES[fmt]
    if mode == 0:
        zp = 8.0 if zeros is None else _words(zeros).T.double().repeat_interleave(128, 1)
        return ((_words(weight).double() - zp) * scale.double().repeat_interleave(128, 1)).to(dtype).double()
    if mode == 1:
        return weight.double() * scale.double()
    raw = weight.view(torch.uint8).long()
    if mode in (2, 5):
        k = raw.shape[1] * 4 // 3
        high = ((raw[:, k // 2:, None] >> (torch.arange(4, device=raw.device) * 2)) & 3).flatten(1)
        code = _nibbles(raw[:, :k // 2]) | (high << 4)
    else:
        k = raw.shape[1] * 2
        code = _nibbles(raw)
    if mode in (4, 5):
        return (code.double() - (8 if mode == 4 else 32)) * scale.double().repeat_interleave(128, 1)
    if mode == 3:
        level = scale[:16, k // 16 + 4:].contiguous().view(torch.float32).reshape(16).double()[code]
    else:
        level = code.double() - 32
    relative = scale[:, :k // 16].contiguous().view(torch.float8_e4m3fn).double().repeat_interleave(16, 1)
    channel = scale[:, k // 16:k // 16 + 4].contiguous().view(torch.float32).double()
    return (level * relative).round().clamp(-127, 127) * channel


def _exact_layer(case, bank, x, logits):
    fmt, dtype = case["fmt"], x.dtype
    probabilities = torch.softmax(logits.double(), -1)
    weights, ids = probabilities.topk(TOP_K, -1)
    weights = weights / weights.sum(-1, keepdim=True)
    stored = weights.to(dtype).double()
    mode = MODES.get(fmt)
    if fmt in FP8:
        rows = _fp8_rows(x, 128 if case["x_group"] == "128" else HIDDEN)
    elif mode in (4, 5):
        rows = _fp8_rows(x, HIDDEN)
    elif mode == 0:
        rows = x.double()
    else:
        rows = _int8_rows(x.double(), dtype)
    float8 = fmt in FP8 or mode in (4, 5)
    flat = ids.reshape(-1)
    partial = torch.zeros(flat.numel(), HIDDEN, dtype=torch.float64, device=x.device)
    zeros = (None, None) if float8 else (bank.w13_zeros, bank.w2_zeros)
    for e in torch.unique(flat).tolist():
        pairs = torch.nonzero(flat == e).reshape(-1)
        z13, z2 = (None if z is None else z[e] for z in zeros)
        w13 = _matrix(fmt, bank.w13_weight[e], bank.w13_scale_inv[e], z13, dtype)
        gate, up = (rows[pairs // TOP_K] @ w13.T).chunk(2, -1)
        w2 = _matrix(fmt, bank.w2_weight[e], bank.w2_scale_inv[e], z2, dtype if float8 else torch.bfloat16)
        if float8:
            gate, up = gate.to(dtype).double(), up.to(dtype).double()
            y = _fp8_rows(_silu(gate) * up, 128) @ w2.T
        else:
            act = _bf16(_bf16(_silu(_bf16(gate))) * _bf16(up))
            y = _bf16((act if mode == 0 else _int8_rows(act, torch.bfloat16)) @ w2.T)
        partial[pairs] = y * stored.reshape(-1)[pairs, None]
    return partial.view(-1, TOP_K, HIDDEN).sum(1), weights, ids


def exact(case, seed):
    if case["kind"] == "linear":
        words, scales, x = _linear_inputs(case, seed)
        w = (_words(words.T.contiguous()).double() - 8) * scales.T.double().repeat_interleave(128, 1)
        return x.double() @ w.to(x.dtype).double().T
    if case["kind"] == "shared":
        weights, (x, experts_out, after_mixer) = _shared_inputs(case, seed)
        router, sgate_w, gate_w, up_w, down_w = (w.double() for w in weights)
        rows = x.double()
        sgate = torch.sigmoid(_bf16(rows @ sgate_w.T))
        act = _bf16(_silu(_bf16(rows @ gate_w.T))) * _bf16(rows @ up_w.T)
        shared = _bf16(_bf16(sgate) * _bf16(_bf16(act) @ down_w.T))
        return (rows @ router.T, sgate.reshape(-1), act,
                after_mixer.double() + _bf16(experts_out.double() + shared))
    return [_exact_layer(case, *_layer_inputs(case, seed, layer)) for layer in range(case["layers"])]
