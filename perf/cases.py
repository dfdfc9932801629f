"""What this framework is used for, as cases that can be timed and whose results can be compared.

A user of the library multiplies float16 activations with int4 or int8 weights: token by token (decode, a few rows), for a
batch of sequences (tens of rows) and for whole prompts (hundreds to thousands of rows).  Three ways lead there: the tensor
front end `relax_amd.wq_matmul`, called projection by projection; the runtime modules of an exported model, whose
weights are bound once (`relax_amd.module`); and `relax_amd.wq_dequantize` where a consumer wants the float16 matrix.

The sizes are those of the configurations this repository benchmarks (projections of hidden size 4096 / 11008 and
5120 / 13824, a 152064-row vocabulary) and, in `draw`, the ranges around them.  Weights are uniform over the integer range as
in the configurations; scales are spread by a factor of three around the value that gives a projection of unit
activations unit outputs, so that the layers of a stack can be chained in float16.
"""
import math
import types

import torch

import relax_amd
from relax_amd import lib
from relax_amd import module as wq_module
from relax_amd import vm_harness

# The most that one drawn case may cost: what the largest listed ones (prefill_layer_q4_2048, decode_layers_q8_b16) need.
MAX_FLOPS = 8.2e11
MAX_BYTES = 1.0e9


def listed():
    return [
        # One token through one projection: the smallest call there is, where the launch and the host path count.
        dict(name="decode_one_q4", kind="linear", m=1, n=4096, k=4096, bits=4, group=32, tail="none", tiled=False, workspace=False),
        # One token of one sequence through consecutive decoder layers, weights coming from memory as in a whole model.
        dict(name="decode_layers_q4_b1", kind="layers", m=1, hidden=4096, ffn=11008, layers=8, bits=4, group=32),
        # The same for a small batch of sequences.
        dict(name="decode_layers_q4_b8", kind="layers", m=8, hidden=4096, ffn=11008, layers=8, bits=4, group=32),
        # int8 weights, the larger shapes, the largest decode batch.
        dict(name="decode_layers_q8_b16", kind="layers", m=16, hidden=5120, ffn=13824, layers=3, bits=8, group=128),
        # Next-token scores of three sequences over a vocabulary: few rows, very many columns.
        dict(name="vocabulary_q4", kind="linear", m=3, n=152064, k=4096, bits=4, group=32, tail="none", tiled=False, workspace=False),
        # A serving batch of an odd size: one token of each of 37 sequences.
        dict(name="batch_layers_q4_37", kind="layers", m=37, hidden=4096, ffn=11008, layers=3, bits=4, group=32),
        # An exported model's layer with bound weights (tile-major copy and a workspace of its own), activations [batch, sequence, K].
        dict(name="module_layer_q8", kind="module", batch=3, seq=33, hidden=5120, ffn=13824, bits=8, group=128, tiled=True, workspace=True),
        # A prompt chunk through int8 layers.
        dict(name="prefill_layer_q8_256", kind="layers", m=256, hidden=5120, ffn=13824, layers=1, bits=8, group=128),
        # A projection with bias and gelu at the other common int4 group size, with sizes that are no multiple of a tile.
        dict(name="ragged_gelu_q4_g128", kind="linear", m=333, n=10001, k=4224, bits=4, group=128, tail="bias_gelu", tiled=False, workspace=False),
        # A short prompt, and a long one, through one layer.
        dict(name="prefill_layer_q4_512", kind="layers", m=512, hidden=4096, ffn=11008, layers=1, bits=4, group=32),
        dict(name="prefill_layer_q4_2048", kind="layers", m=2048, hidden=4096, ffn=11008, layers=1, bits=4, group=32),
        # The float16 matrix itself, for a consumer that does not read packed weights.
        dict(name="dequantize_q4", kind="dequantize", n=22016, k=4096, bits=4, group=32),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    while True:
        bits = rng.choice((4, 8))
        standard = 32 if bits == 4 else 128
        kind = rng.choices(("linear", "layers", "module", "dequantize"), (45, 30, 15, 10))[0]
        group = standard
        if kind in ("linear", "dequantize") and rng.random() < 0.3:  # the other group sizes
            group = rng.choice((64, 128) if bits == 4 else (32, 64))
        m = round(_log_uniform(rng, 1, 2048))
        if kind == "linear":
            tiled = group == standard and rng.random() < 0.2  # weights laid out once by wq_tile_weights
            step = 256 if tiled or rng.random() < 0.5 else group
            k = step * max(1, round(_log_uniform(rng, 1024, 14336) / step))
            n = round(_log_uniform(rng, 1024, 32768))
            if rng.random() < 0.5:
                n = 128 * max(1, round(n / 128))
            tails = ("none", "bias", "bias_relu", "bias_gelu", "residual") + (() if tiled else ("silu_mul",))
            tail = rng.choices(tails, (50, 10, 10, 10, 10) + (() if tiled else (10,)))[0]
            if tail == "silu_mul":
                n += n % 2
            case = dict(kind="linear", m=m, n=n, k=k, bits=bits, group=group, tail=tail, tiled=tiled, workspace=rng.random() < 0.3)
        elif kind == "dequantize":
            k = group * max(1, round(_log_uniform(rng, 1024, 14336) / group))
            case = dict(kind="dequantize", n=round(_log_uniform(rng, 1024, 32768)), k=k, bits=bits, group=group)
        else:
            hidden = 256 * round(_log_uniform(rng, 1024, 6144) / 256)
            ffn = 256 * round(hidden * rng.uniform(2.5, 3.5) / 256)
            if kind == "layers":
                case = dict(kind="layers", m=m, hidden=hidden, ffn=ffn, layers=rng.randint(1, 8 if m <= 64 else 2), bits=bits, group=group)
            else:
                batch = rng.randint(1, min(4, m))
                case = dict(kind="module", batch=batch, seq=max(1, m // batch), hidden=hidden, ffn=ffn, bits=bits, group=group,
                            tiled=rng.random() < 0.5, workspace=rng.random() < 0.7)
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


def _rows(case):
    return case["batch"] * case["seq"] if case["kind"] == "module" else case["m"]


def _projections(case):
    """(N, K, fused tail) of one decoder layer: query/key/value, attention output onto the residual stream, gate and up
    with the gated activation, down onto the residual stream."""
    h, f = case["hidden"], case["ffn"]
    return (("qkv", 3 * h, h, "none"), ("out", h, h, "residual"), ("gate_up", 2 * f, h, "silu_mul"), ("down", h, f, "residual"))


def _weight_bytes(n, k, bits, group):
    return n * k * bits // 8 + n * (k // group) * 2


def work(case):
    """Weights, scales, activations and fused operands read once, outputs written once; two operations per weight and row."""
    bits, group = case["bits"], case["group"]
    if case["kind"] == "dequantize":
        n, k = case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, bits, group) + 2 * n * k, "flops": n * k}
    m = _rows(case)
    if case["kind"] == "linear":
        calls = [("", case["n"], case["k"], case["tail"])]
    else:
        calls = _projections(case) * case.get("layers", 1)
    nbytes = flops = 0
    for _, n, k, tail in calls:
        nbytes += _weight_bytes(n, k, bits, group) + 2 * m * k + 2 * m * (n // 2 if tail == "silu_mul" else n)
        nbytes += 2 * m * n if tail == "residual" else 2 * n if tail.startswith("bias") else 0
        flops += 2 * m * n * k
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Unpacking and the one rounding of a dequantized weight are exact; a projection accumulates in float32 and rounds its
    result, and every step of its tail, to float16."""
    return "exact" if case["kind"] == "dequantize" else {"rel": 1e-3}


def _weights(n, k, bits, group, gen):
    """Packed words and scales: int4 fields 0..15 (zero point 7), int8 fields -127..127."""
    if bits == 4:
        wq = torch.randint(-(1 << 31), (1 << 31) - 1, (n, k // 8), dtype=torch.int32, device="cuda", generator=gen)
    else:
        wq = torch.randint(-127, 128, (n, k), dtype=torch.int8, device="cuda", generator=gen).view(torch.int32)
    mean = 1.0 / ((4.63 if bits == 4 else 73.6) * math.sqrt(k))
    scales = torch.rand((n, k // group), device="cuda", generator=gen).add_(0.5).mul_(mean).half()
    return wq, scales


def _normal(shape, gen):
    return torch.randn(shape, dtype=torch.float16, device="cuda", generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = types.SimpleNamespace(kind=case["kind"], bits=case["bits"], group=case["group"])
    if case["kind"] == "dequantize":
        s.wq, s.scales = _weights(case["n"], case["k"], s.bits, s.group, gen)
    elif case["kind"] == "linear":
        _prepare_linear(s, case, gen)
    elif case["kind"] == "layers":
        _prepare_layers(s, case, gen)
    else:
        _prepare_modules(s, case, gen)
    return s


def _prepare_linear(s, case, gen):
    m, n, k, tail = case["m"], case["n"], case["k"], case["tail"]
    s.x = _normal((m, k), gen)
    s.wq, s.scales = _weights(n, k, s.bits, s.group, gen)
    s.options = {}
    if tail.startswith("bias"):
        s.options["bias"] = _normal((n,), gen)
    if tail == "residual":
        s.options["residual"] = _normal((m, n), gen)
    if tail in ("bias_relu", "bias_gelu", "silu_mul"):
        s.options["activation"] = tail.replace("bias_", "")
    if case["tiled"]:
        s.wq, s.scales = relax_amd.wq_tile_weights(s.wq, s.scales, s.bits, s.group)
        s.options["tiled_n"] = n
    if case["workspace"]:
        s.options["workspace"] = relax_amd.wq_workspace(relax_amd.wq_workspace_bytes(s.bits, s.group, n, k, m, case["tiled"]))


def _prepare_layers(s, case, gen):
    """Per layer the four weights and what the parts of a model between the projections hand over: the normalized
    activations of both halves and the attention's output."""
    m, h = case["m"], case["hidden"]
    s.h = _normal((m, h), gen)
    s.layers = []
    for _ in range(case["layers"]):
        weights = [_weights(n, k, s.bits, s.group, gen) for _, n, k, _ in _projections(case)]
        s.layers.append((weights, _normal((m, h), gen), _normal((m, h), gen), _normal((m, h), gen)))


def _prepare_modules(s, case, gen):
    """The modules of one layer's composites, weights bound; activations, residual and outputs in the caller's tensors."""
    b, q, h, f = case["batch"], case["seq"], case["hidden"], case["ffn"]
    vm_harness.set_stream()
    flags = (wq_module.TILE_WEIGHTS if case["tiled"] else 0) | (wq_module.OWN_WORKSPACE if case["workspace"] else 0)
    s.functions, s.modules = {}, []
    for name, n, k, tail in _projections(case):
        fused = tail == "residual"
        spec = vm_harness.CallSpec(op=0, bits=s.bits, group=0, zero_point=7 if s.bits == 4 else 0, arg_wq=0, arg_scales=1, arg_x=2,
                                   arg_residual=3 if fused else -1, arg_out=4 if fused else 3, num_args=5 if fused else 4,
                                   activation=lib.ACT_SILU_MUL if tail == "silu_mul" else lib.ACT_NONE)
        mod = wq_module.SubgraphModule.create(name, spec, ["w", "s"], [0, 1], flags, workspace_rows=b * q if case["workspace"] else 0)
        mod.get_function("__init_" + name)(*_weights(n, k, s.bits, s.group, gen))
        s.modules.append(mod)
        s.functions[name] = mod.get_function(name)
    s.x, s.attention, s.x2, s.h0 = (_normal((b, q, h), gen) for _ in range(4))
    s.qkv, s.h1, s.gated, s.h2 = (torch.empty((b, q, c), dtype=torch.float16, device="cuda") for c in (3 * h, h, f, h))


def run(s):
    if s.kind == "dequantize":
        return relax_amd.wq_dequantize(s.wq, s.scales, s.bits, s.group)
    if s.kind == "linear":
        return relax_amd.wq_matmul(s.x, s.wq, s.scales, s.bits, s.group, **s.options)
    if s.kind == "layers":
        return _run_layers(s)
    f = s.functions
    f["qkv"](s.x, s.qkv)
    f["out"](s.attention, s.h0, s.h1)
    f["gate_up"](s.x2, s.gated)
    f["down"](s.gated, s.h1, s.h2)
    return s.qkv, s.h1, s.gated, s.h2


def _run_layers(s):
    bits, group, h, out = s.bits, s.group, s.h, []
    for ((wqkv, sqkv), (wo, so), (wgu, sgu), (wd, sd)), x, attention, x2 in s.layers:
        out.append(relax_amd.wq_matmul(x, wqkv, sqkv, bits, group))
        h = relax_amd.wq_matmul(attention, wo, so, bits, group, residual=h)
        g = relax_amd.wq_matmul(x2, wgu, sgu, bits, group, activation="silu_mul")
        h = relax_amd.wq_matmul(g, wd, sd, bits, group, residual=h)
    out.append(h)
    return out
