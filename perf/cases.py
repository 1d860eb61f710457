"""The work that users of this framework give it, as cases to be timed and checked.

Every case is one compiled program: the StableHLO text that a jitted JAX function
lowers to (``pjrt_amd.stablehlo_configs`` or the small writers below) or a program
written with ``pjrt_amd.graph``, compiled once by ``Runtime.compile`` and then
launched on device buffers with ``LoadedProgram.enqueue``, as the PJRT plugin's
Execute does.  ``prepare`` holds what such a program keeps between calls: the loaded
program, its inputs and its output buffers.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pjrt-ocl_amd", "python")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from pjrt_amd import configs, graph, lowering, stablehlo_configs, vmprogram  # noqa: E402
from pjrt_amd.runtime import Runtime  # noqa: E402

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i32": torch.int32}
_OF_DT = {vmprogram.DT_F32: "f32", vmprogram.DT_F16: "f16", vmprogram.DT_BF16: "bf16", vmprogram.DT_I32: "i32"}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i32": 4}


def listed():
    return [
        # the smallest call: a small regressor or policy head, one forward per request
        {"name": "mlp_f32_small", "kind": "mlp", "b": 256, "d_in": 128, "h": 512, "d_out": 64},
        # the backward direction: one training step's gradients of an f32 MLP (jax.grad)
        {"name": "mlp_grad_f32", "kind": "mlp_grad", "b": 1024, "d_in": 784, "h": 2048, "d_out": 256},
        # the large dense layer on the matrix cores
        {"name": "matmul_bf16_4096", "kind": "matmul", "m": 4096, "k": 4096, "n": 4096, "dt": "bf16", "out": "f32"},
        # JAX's default type, at sizes nobody rounded up
        {"name": "matmul_f32_odd", "kind": "matmul", "m": 1001, "k": 777, "n": 1130, "dt": "f32", "out": "f32"},
        # logits of a tied embedding: hidden states against the table's rows (x @ wte.T)
        {"name": "tied_head_bf16", "kind": "head", "rows": 512, "d": 768, "vocab": 32000, "dt": "bf16"},
        # prefill attention of a long prompt
        {"name": "attention_causal_bf16", "kind": "attention", "b": 4, "h": 16, "t": 2048, "d": 128, "dt": "bf16",
         "causal": True},
        # an encoder's attention: every position sees every other, a length that fills no block
        {"name": "attention_full_f16", "kind": "attention", "b": 2, "h": 12, "t": 1000, "d": 64, "dt": "f16",
         "causal": False},
        # the bandwidth-bound layer: layer norm, GELU and the cast to bf16 in one pass
        {"name": "ln_gelu_8192x4096", "kind": "ln_gelu", "rows": 8192, "d": 4096},
        # token probabilities over a vocabulary
        {"name": "softmax_vocab_f32", "kind": "softmax", "rows": 512, "d": 32000},
        # one decoder block over a prompt
        {"name": "block_prefill_bf16", "kind": "block", "t": 512, "d": 768, "heads": 12, "mlp": 3072},
        # one token through a small f32 decoder, keys and values appended (latency)
        {"name": "decode_step_f32", "kind": "decode_step", "d": 512, "heads": 8, "mlp": 2048, "layers": 6, "ctx": 256},
        # a whole generation: prompt, then greedy steps in one device loop, with the logits of every step
        {"name": "generate_bf16", "kind": "generate", "layers": 12, "d": 768, "heads": 12, "mlp": 3072,
         "vocab": 32000, "prompt": 512, "steps": 32},
    ]


def _log(rng, lo, hi, of=1):
    """A whole number in [lo, hi], even over its logarithm, a multiple of `of`."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / of)) * of))


def draw(rng):
    kind = rng.choice(["mlp", "mlp_grad", "matmul", "matmul", "head", "attention", "attention", "ln_gelu", "softmax",
                       "block", "decode_step", "generate"])
    even = rng.choice([1, 1, 8, 64])             # sizes that nobody rounded, and rounded ones
    if kind in ("mlp", "mlp_grad"):
        return {"kind": kind, "b": _log(rng, 16, 4096, even), "d_in": _log(rng, 64, 1024, even),
                "h": _log(rng, 64, 2048, even), "d_out": _log(rng, 64, 1024, even) if even > 1 else _log(rng, 4, 1024)}
    if kind == "matmul":
        dt = rng.choice(["bf16", "f16", "f32"])
        most = 2048 if dt == "f32" else 4096
        return {"kind": kind, "m": _log(rng, 64, most, even), "k": _log(rng, 64, most, even),
                "n": _log(rng, 64, most, even), "dt": dt, "out": rng.choice(["f32", dt])}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 512), "d": _log(rng, 128, 1024, 64),
                "vocab": _log(rng, 1000, 32000, even), "dt": rng.choice(["bf16", "f32"])}
    if kind == "attention":
        t, d = _log(rng, 64, 2048, even), rng.choice([32, 64, 64, 80, 128])
        h = rng.choice([4, 8, 12, 16])
        dt = rng.choice(["bf16", "bf16", "f16", "f32"])
        return {"kind": kind, "b": rng.choice([1, 2, 4]) if dt != "f32" else 1, "h": h, "t": t, "d": d, "dt": dt,
                "causal": rng.random() < 0.6}
    if kind == "ln_gelu":
        d = _log(rng, 64, 8192, even)
        return {"kind": kind, "rows": _log(rng, 16, max(16, min(8192, (1 << 25) // d)), even), "d": d}
    if kind == "softmax":
        d = _log(rng, 64, 50000, even)
        return {"kind": kind, "rows": _log(rng, 16, max(16, min(8192, (1 << 24) // d))), "d": d}
    if kind == "block":
        heads = rng.choice([4, 8, 12, 16])
        return {"kind": kind, "t": _log(rng, 32, 1024, even), "d": 64 * heads, "heads": heads,
                "mlp": 256 * heads}
    if kind == "decode_step":
        heads = rng.choice([4, 8, 16])
        return {"kind": kind, "d": 64 * heads, "heads": heads, "mlp": 256 * heads, "layers": rng.choice([2, 4, 6]),
                "ctx": _log(rng, 64, 512, 8)}
    heads = rng.choice([4, 8, 12])
    return {"kind": kind, "layers": rng.choice([2, 4, 6]), "d": 64 * heads, "heads": heads, "mlp": 256 * heads,
            "vocab": _log(rng, 2000, 32000, 8), "prompt": _log(rng, 16, 512), "steps": _log(rng, 4, 32)}


# ---- programs ------------------------------------------------------------------------------

_t = stablehlo_configs._t


def _text_mlp_grad(b, d_in, h, d_out):
    """jax.grad of mean((relu(x @ w1 + b1) @ w2 + b2 - y) ** 2) in the four parameters, with
    the loss's residual o - y (value_and_grad with has_aux)."""
    X, W1, B1, W2, B2 = _t((b, d_in)), _t((d_in, h)), _t((h,)), _t((h, d_out)), _t((d_out,))
    H, HB, Y = _t((b, h)), _t((b, h), "i1"), _t((b, d_out))
    W1T, W2T = _t((h, d_in)), _t((d_out, h))
    return f"""
module @jit_step {{
  func.func public @main(%x: {X}, %y: {Y}, %w1: {W1}, %b1: {B1}, %w2: {W2}, %b2: {B2}) -> ({Y}, {W1}, {B1}, {W2}, {B2}) {{
    %z = stablehlo.constant dense<0.000000e+00> : tensor<f32>
    %zh = stablehlo.broadcast_in_dim %z, dims = [] : (tensor<f32>) -> {H}
    %0 = stablehlo.dot_general %x, %w1, contracting_dims = [1] x [0], precision = [DEFAULT, DEFAULT] : ({X}, {W1}) -> {H}
    %1 = stablehlo.broadcast_in_dim %b1, dims = [1] : ({B1}) -> {H}
    %2 = stablehlo.add %0, %1 : {H}
    %3 = stablehlo.maximum %2, %zh : {H}
    %4 = stablehlo.compare  GT, %2, %zh,  FLOAT : ({H}, {H}) -> {HB}
    %5 = stablehlo.dot_general %3, %w2, contracting_dims = [1] x [0], precision = [DEFAULT, DEFAULT] : ({H}, {W2}) -> {Y}
    %6 = stablehlo.broadcast_in_dim %b2, dims = [1] : ({B2}) -> {Y}
    %7 = stablehlo.add %5, %6 : {Y}
    %8 = stablehlo.subtract %7, %y : {Y}
    %c = stablehlo.constant dense<{2.0 / (b * d_out):.9e}> : tensor<f32>
    %9 = stablehlo.broadcast_in_dim %c, dims = [] : (tensor<f32>) -> {Y}
    %10 = stablehlo.multiply %8, %9 : {Y}
    %11 = stablehlo.reduce(%10 init: %z) applies stablehlo.add across dimensions = [0] : ({Y}, tensor<f32>) -> {B2}
    %12 = stablehlo.dot_general %10, %3, contracting_dims = [0] x [0], precision = [DEFAULT, DEFAULT] : ({Y}, {H}) -> {W2T}
    %13 = stablehlo.transpose %12, dims = [1, 0] : ({W2T}) -> {W2}
    %14 = stablehlo.dot_general %10, %w2, contracting_dims = [1] x [1], precision = [DEFAULT, DEFAULT] : ({Y}, {W2}) -> {H}
    %15 = stablehlo.select %4, %14, %zh : {HB}, {H}
    %16 = stablehlo.reduce(%15 init: %z) applies stablehlo.add across dimensions = [0] : ({H}, tensor<f32>) -> {B1}
    %17 = stablehlo.dot_general %15, %x, contracting_dims = [0] x [0], precision = [DEFAULT, DEFAULT] : ({H}, {X}) -> {W1T}
    %18 = stablehlo.transpose %17, dims = [1, 0] : ({W1T}) -> {W1}
    return %8, %18, %16, %13, %11 : {Y}, {W1}, {B1}, {W2}, {B2}
  }}
}}
"""


def _text_head(rows, d, vocab, dt):
    """def f(x, wte): return jnp.einsum("td,vd->tv", x, wte, preferred_element_type=jnp.float32)"""
    X, W, Y = _t((rows, d), dt), _t((vocab, d), dt), _t((rows, vocab))
    return f"""
module @jit_f {{
  func.func public @main(%arg0: {X}, %arg1: {W}) -> {Y} {{
    %0 = stablehlo.dot_general %arg0, %arg1, contracting_dims = [1] x [1], precision = [DEFAULT, DEFAULT] : ({X}, {W}) -> {Y}
    return %0 : {Y}
  }}
}}
"""


def _text_softmax(rows, d):
    """def f(x): return jax.nn.softmax(x, axis=-1)"""
    X, R, R1 = _t((rows, d)), _t((rows,)), _t((rows, 1))
    return f"""
module @jit_f {{
  func.func public @main(%arg0: {X}) -> {X} {{
    %m = stablehlo.constant dense<0xFF800000> : tensor<f32>
    %0 = stablehlo.reduce(%arg0 init: %m) applies stablehlo.maximum across dimensions = [1] : ({X}, tensor<f32>) -> {R}
    %1 = stablehlo.broadcast_in_dim %0, dims = [0] : ({R}) -> {R1}
    %2 = stablehlo.broadcast_in_dim %1, dims = [0, 1] : ({R1}) -> {X}
    %3 = stablehlo.subtract %arg0, %2 : {X}
    %4 = stablehlo.exponential %3 : {X}
    %z = stablehlo.constant dense<0.000000e+00> : tensor<f32>
    %5 = stablehlo.reduce(%4 init: %z) applies stablehlo.add across dimensions = [1] : ({X}, tensor<f32>) -> {R}
    %6 = stablehlo.broadcast_in_dim %5, dims = [0] : ({R}) -> {R1}
    %7 = stablehlo.broadcast_in_dim %6, dims = [0, 1] : ({R1}) -> {X}
    %8 = stablehlo.divide %4, %7 : {X}
    return %8 : {X}
  }}
}}
"""


_BLOCK = ("ln1_g", "ln1_b", "w_qkv", "b_qkv", "w_o", "b_o", "ln2_g", "ln2_b", "w_fc", "b_fc", "w_proj", "b_proj")


def _block_program(t, d, heads, mlp):
    """One pre-LN decoder block over t tokens: the prefill layer of configs.gpt_c5."""
    g, hd, ADD = graph.Graph(), d // heads, vmprogram.SUB_ADD
    x = g.input((t, d))
    shapes = _block_shapes(d, mlp)
    P = {n: g.input(s, dt) for n, (s, dt) in shapes.items()}
    h = g.layernorm(x, P["ln1_g"], P["ln1_b"], 1e-5, out_dtype="bf16")
    qkv = g.dot(h, P["w_qkv"], out_dtype="bf16", residual=P["b_qkv"], epilogue=[(ADD, 2, 0.0, 0.0)])
    q, k, v = (g.materialize(g.view(qkv, (heads, t, hd), (hd, 3 * d, 1), s * d)) for s in range(3))
    att = g.flash_attention(q, k, v, 1.0 / math.sqrt(hd), True)
    rows = g.reshape(g.transpose_view(att, (1, 0, 2)), (t, d))
    xb = g.add(x, g.broadcast_view(P["b_o"], (t, d), (1,)))
    x = g.dot(rows, P["w_o"], residual=xb, epilogue=[(ADD, 1, 0.0, 0.0)])
    h = g.layernorm(x, P["ln2_g"], P["ln2_b"], 1e-5, out_dtype="bf16")
    f = g.dot(h, P["w_fc"], out_dtype="bf16", residual=P["b_fc"],
              epilogue=[(ADD, 2, 0.0, 0.0), (vmprogram.SUB_GELU, 0, 0.0, 0.0)])
    xb = g.add(x, g.broadcast_view(P["b_proj"], (t, d), (1,)))
    x = g.dot(f, P["w_proj"], residual=xb, epilogue=[(ADD, 1, 0.0, 0.0)])
    g.output(x, k, v)
    return g.build()


def _block_shapes(d, mlp):
    return {"ln1_g": ((d,), "f32"), "ln1_b": ((d,), "f32"), "w_qkv": ((d, 3 * d), "bf16"), "b_qkv": ((3 * d,), "f32"),
            "w_o": ((d, d), "bf16"), "b_o": ((d,), "f32"), "ln2_g": ((d,), "f32"), "ln2_b": ((d,), "f32"),
            "w_fc": ((d, mlp), "bf16"), "b_fc": ((mlp,), "f32"), "w_proj": ((mlp, d), "bf16"), "b_proj": ((d,), "f32")}


def _gpt(c):
    return configs.GptConfig(layers=c["layers"], d=c["d"], heads=c["heads"], mlp=c["mlp"], vocab=c["vocab"],
                             prompt=c["prompt"], steps=c["steps"])


def _step(c):
    return (c["d"], c["heads"], c["mlp"], c["layers"], c["ctx"])


def _program(c):
    """(program, whether Runtime.compile still has to pack its arena)."""
    k = c["kind"]
    if k == "block":
        return _block_program(c["t"], c["d"], c["heads"], c["mlp"]), True
    if k == "generate":
        return configs.gpt_c5(_gpt(c), emit_logits=True), True
    if k == "mlp":
        text = stablehlo_configs.mlp(c["b"], c["d_in"], c["h"], c["d_out"])
    elif k == "mlp_grad":
        text = _text_mlp_grad(c["b"], c["d_in"], c["h"], c["d_out"])
    elif k == "matmul":
        text = stablehlo_configs.matmul(c["m"], c["k"], c["n"], c["dt"], c["out"])
    elif k == "head":
        text = _text_head(c["rows"], c["d"], c["vocab"], c["dt"])
    elif k == "attention":
        text = stablehlo_configs.attention(c["b"], c["h"], c["t"], c["d"], c["dt"], c["causal"])
    elif k == "ln_gelu":
        text = stablehlo_configs.ln_gelu(c["rows"], c["d"])
    elif k == "softmax":
        text = _text_softmax(c["rows"], c["d"])
    else:
        text = stablehlo_configs.decode_step(_step(c))
    return lowering.lower_text(text), False


# ---- inputs --------------------------------------------------------------------------------

def _inputs(c, seed):
    """The program's inputs in order, on the GPU, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)

    def normal(shape, std=1.0, dt="f32"):
        return (torch.randn(shape, generator=gen, device="cuda") * std).to(_TORCH[dt])

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=gen, device="cuda") * (hi - lo) + lo

    k = c["kind"]
    if k in ("mlp", "mlp_grad"):
        x = normal((c["b"], c["d_in"]))
        w1, b1 = normal((c["d_in"], c["h"]), c["d_in"] ** -0.5), normal((c["h"],), 0.1)
        w2, b2 = normal((c["h"], c["d_out"]), c["h"] ** -0.5), normal((c["d_out"],), 0.1)
        return [x, w1, b1, w2, b2] if k == "mlp" else [x, normal((c["b"], c["d_out"])), w1, b1, w2, b2]
    if k == "matmul":
        return [normal((c["m"], c["k"]), 1.0, c["dt"]), normal((c["k"], c["n"]), c["k"] ** -0.5, c["dt"])]
    if k == "head":
        return [normal((c["rows"], c["d"]), 1.0, c["dt"]), normal((c["vocab"], c["d"]), 0.02, c["dt"])]
    if k == "attention":
        return [normal((c["b"], c["h"], c["t"], c["d"]), 1.0, c["dt"]) for _ in range(3)]
    if k == "ln_gelu":
        return [normal((c["rows"], c["d"])), uniform((c["d"],), 0.5, 1.5), normal((c["d"],), 0.1)]
    if k == "softmax":
        return [normal((c["rows"], c["d"]), 3.0)]
    if k == "block":
        out = [normal((c["t"], c["d"]))]
        for n, (s, dt) in _block_shapes(c["d"], c["mlp"]).items():
            out.append(uniform(s, 0.8, 1.2) if n.endswith("_g") else
                       normal(s, 0.02 if n.startswith(("b_", "ln")) else s[0] ** -0.5, dt))
        return out
    if k == "decode_step":
        out = []
        for name, shape in stablehlo_configs.decode_step_params(_step(c)):
            key = name.split(".")[-1]
            out.append(uniform(shape, 0.8, 1.2) if key in ("ln1_g", "ln2_g") else
                       normal(shape, 0.02) if key in ("ln1_b", "ln2_b") else
                       normal(shape, 1.0 if key in ("x", "kc", "vc") else shape[0] ** -0.5))
        return out
    # generate: as in a trained model the token's embedding leads the residual stream, and the
    # head points from it to one next token, by a margin that rounding does not close
    g = _gpt(c)
    ids = torch.randint(0, g.vocab, (g.prompt,), generator=gen, device="cuda", dtype=torch.int32)
    out, wte = [ids], None
    for name, shape, dt in configs.gpt_param_shapes(g):
        base = name.split(".")[-1]
        if base == "wte":
            wte = normal(shape, 1.0, dt)
            out.append(wte)
        elif base == "lm_head":
            nxt = torch.randperm(g.vocab, generator=gen, device="cuda")
            out.append((wte[nxt].t().float() * 0.25).to(_TORCH[dt]).contiguous())
        elif base.endswith("_g"):
            out.append(uniform(shape, 0.9, 1.1))
        elif base.startswith("b_") or base.endswith("_b"):
            out.append(normal(shape, 0.02))
        else:
            out.append(normal(shape, 0.02, dt))
    return out


# ---- a case ----------------------------------------------------------------------------------

_RT = []


def _runtime():
    """The process's client: one device, opened once."""
    if not _RT:
        _RT.append(Runtime(device=0))
    return _RT[0]


def prepare(case, seed):
    prog, pack = _program(case)
    loaded = _runtime().compile(prog, arena_reuse=pack)
    outs = [torch.empty(s.shape, dtype=_TORCH[_OF_DT[s.dtype]], device="cuda") for s in loaded.outputs]
    ins = _inputs(case, seed)
    torch.cuda.synchronize()        # the program runs on the runtime's own stream
    return {"program": loaded, "in": ins, "out": outs}


def run(state):
    state["program"].enqueue(state["in"], state["out"])
    return state["out"]


def work(case):
    c, k = case, case["kind"]
    if k == "mlp":
        b, i, h, o = c["b"], c["d_in"], c["h"], c["d_out"]
        return {"bytes": 4 * (b * i + i * h + h + h * o + o + b * o), "flops": 2 * b * h * (i + o)}
    if k == "mlp_grad":
        b, i, h, o = c["b"], c["d_in"], c["h"], c["d_out"]
        return {"bytes": 4 * (b * i + 2 * b * o + 2 * (i * h + h + h * o + o)), "flops": 2 * b * h * (2 * i + 3 * o)}
    if k == "matmul":
        m, kk, n = c["m"], c["k"], c["n"]
        return {"bytes": _SIZE[c["dt"]] * (m * kk + kk * n) + _SIZE[c["out"]] * m * n, "flops": 2 * m * kk * n}
    if k == "head":
        r, d, v = c["rows"], c["d"], c["vocab"]
        return {"bytes": _SIZE[c["dt"]] * (r * d + v * d) + 4 * r * v, "flops": 2 * r * d * v}
    if k == "attention":
        n, t, d = c["b"] * c["h"], c["t"], c["d"]
        return {"bytes": 4 * n * t * d * _SIZE[c["dt"]], "flops": 4 * n * d * (t * (t + 1) // 2 if c["causal"] else t * t)}
    if k == "ln_gelu":
        return {"bytes": c["rows"] * c["d"] * 6 + 8 * c["d"], "flops": 20 * c["rows"] * c["d"]}
    if k == "softmax":
        return {"bytes": c["rows"] * c["d"] * 8, "flops": 5 * c["rows"] * c["d"]}
    if k == "block":
        t, d, m = c["t"], c["d"], c["mlp"]
        return {"bytes": 8 * t * d + 2 * (4 * d * d + 2 * d * m) + 4 * t * d,
                "flops": 2 * t * (4 * d * d + 2 * d * m) + 4 * d * t * (t + 1) // 2}
    if k == "decode_step":
        d, m, l, n = c["d"], c["mlp"], c["layers"], c["ctx"]
        return {"bytes": 4 * l * (4 * d * d + 2 * d * m + 2 * n * d), "flops": 2 * l * (4 * d * d + 2 * d * m + 2 * n * d)}
    d, m, l, v, p, s = c["d"], c["mlp"], c["layers"], c["vocab"], c["prompt"], c["steps"]
    per = l * (4 * d * d + 2 * d * m)                 # weights of the blocks
    keys = l * d * (p * (p + 1) // 2 + sum(p + i + 1 for i in range(s)))
    # every step reads the blocks, the head and the cache's prefix
    return {"bytes": (s + 1) * 2 * (per + d * v) + 4 * l * d * sum(p + i for i in range(s)) + 4 * (s + 1) * v,
            "flops": 2 * (p + s) * per + 2 * (s + 1) * d * v + 4 * keys}


def tolerance(case):
    """About four times the distance from exact() that was measured."""
    k = case["kind"]
    if k in ("mlp", "mlp_grad", "matmul", "head"):
        out = case.get("out", "f32")
        return {"rel": {"f32": 4e-6, "f16": 1e-3, "bf16": 7e-3}[out]}
    if k == "attention":
        return {"rel": {"f32": 4e-6, "f16": 1.2e-3, "bf16": 8e-3}[case["dt"]]}
    return {"rel": {"ln_gelu": 8e-3, "softmax": 4e-6, "block": 1e-2, "decode_step": 4e-6, "generate": 1.2e-2}[k]}


# ---- the same in 64 bits ------------------------------------------------------------------

def _ln(x, g, b, eps=1e-5):
    mu = x.mean(-1, keepdim=True)
    var = ((x - mu) ** 2).mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(var + eps) * g + b


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _attend(q, k, v, scale, causal):
    """softmax(scale q k^T) v over the leading dims; with `causal` the last query sees every key."""
    s = (q @ k.transpose(-1, -2).contiguous()) * scale
    if causal:
        t, n = s.shape[-2:]
        s = s.masked_fill(torch.ones((t, n), dtype=torch.bool, device=s.device).triu(n - t + 1), -math.inf)
    return torch.softmax(s, -1) @ v


def _layer(x, P, heads, cache=None):
    """One block over the rows of x; `cache`: the earlier rows' (k, v). Returns x, k, v with heads leading."""
    t, d = x.shape
    q, k, v = (y.reshape(t, heads, d // heads).transpose(0, 1)
               for y in (_ln(x, P["ln1_g"], P["ln1_b"]) @ P["w_qkv"] + P["b_qkv"]).split(d, 1))
    if cache:
        k, v = torch.cat([cache[0], k], 1), torch.cat([cache[1], v], 1)
    a = _attend(q, k, v, (d // heads) ** -0.5, True).transpose(0, 1).reshape(t, d)
    x = x + P["b_o"] + a @ P["w_o"]
    return x + P["b_proj"] + _gelu(_ln(x, P["ln2_g"], P["ln2_b"]) @ P["w_fc"] + P["b_fc"]) @ P["w_proj"], k, v


def exact(case, seed):
    c, k = case, case["kind"]
    ins = [x.double() if x.is_floating_point() else x for x in _inputs(case, seed)]
    if k == "mlp":
        x, w1, b1, w2, b2 = ins
        return [(x @ w1 + b1).clamp_min(0) @ w2 + b2]
    if k == "mlp_grad":
        x, y, w1, b1, w2, b2 = ins
        pre = x @ w1 + b1
        h = pre.clamp_min(0)
        r = h @ w2 + b2 - y
        g = r * (2.0 / r.numel())
        gh = (g @ w2.t()) * (pre > 0)
        return [r, x.t() @ gh, gh.sum(0), h.t() @ g, g.sum(0)]
    if k == "matmul":
        return [ins[0] @ ins[1]]
    if k == "head":
        return [ins[0] @ ins[1].t()]
    if k == "attention":
        q, kk, v = ins
        return [torch.stack([_attend(q[i], kk[i], v[i], c["d"] ** -0.5, c["causal"]) for i in range(c["b"])])]
    if k == "ln_gelu":
        return [_gelu(_ln(*ins))]
    if k == "softmax":
        return [torch.softmax(ins[0], -1)]
    if k == "block":
        x, kk, v = _layer(ins[0], dict(zip(_BLOCK, ins[1:])), c["heads"])
        return [x, kk, v]
    if k == "decode_step":
        names = [n for n, _ in stablehlo_configs.decode_step_params(_step(c))]
        P = dict(zip(names, ins))
        x, heads, d = P["x"], c["heads"], c["d"]
        for l in range(c["layers"]):
            p = lambda n: P[f"{l}.{n}"]                                                       # noqa: E731
            h = _ln(x, p("ln1_g"), p("ln1_b"))
            q, kk, v = ((h @ p(w)).reshape(heads, 1, d // heads) for w in ("wq", "wk", "wv"))
            a = _attend(q, torch.cat([P["kc"][l], kk], 1), torch.cat([P["vc"][l], v], 1), (d // heads) ** -0.5, False)
            x = x + a.reshape(1, d) @ p("wo")
            x = x + _gelu(_ln(x, p("ln2_g"), p("ln2_b")) @ p("w1")) @ p("w2")
        return [x]
    g = _gpt(c)
    P = dict(zip(["ids"] + [n for n, _, _ in configs.gpt_param_shapes(g)], ins))
    layers = [{n: P[f"h{l}.{n}"] for n in _BLOCK} for l in range(g.layers)]
    tok, pos, caches, logits = P["ids"].long(), 0, [None] * g.layers, []
    for _ in range(g.steps + 1):
        x = P["wte"][tok] + P["wpe"][pos:pos + tok.numel()]
        for l in range(g.layers):
            x, kk, v = _layer(x, layers[l], g.heads, caches[l])
            caches[l] = (kk, v)
        logits.append((_ln(x[-1:], P["lnf_g"], P["lnf_b"]) @ P["lm_head"])[0])
        pos, tok = pos + tok.numel(), logits[-1].argmax().reshape(1)
    return [None, None, torch.stack(logits)]
