"""The work that programs built on this framework launch, as measurable cases.

A case is one compiled DSL program (``"op"``, a key of
``programs.CONFIG_PROGRAMS``) and the sizes it is launched at. ``run`` is what
a user's program does per call: ``CompiledProgram.launch`` on tensors that are
already on the GPU, into output tensors that the caller owns. The compiled
program is the handle such a program keeps; it is made once per process.

``listed`` holds fixed points of the ranges, ``draw`` any point of them:

  contractions   M from one row to 8192, N and K from 16 to 8192, K- or
                 N-contiguous second operand, f32, bf16 and f16 inputs; half
                 of them with N and K multiples of 64, as weights mostly are,
                 the others odd as they come
  batched        1 to 64 batches of 16 to 1024 square-ish planes, K 32 to 256
  rows           softmax, layernorm and row reductions over rows of 16 to
                 131072 elements, f32, bf16 and u8
  columns        reductions over the non-contiguous axis, f32 and bf16
  maps           elementwise, with broadcast and transposed operands
  chains         a reduction of a reduction
"""
import functools
import math

import torch

from tcacomp_amd import compiler, programs

DEVICE = "cuda"

GEMM = {  # op: (input type, second operand stored [N][K])
    "gemm_f32": (torch.float32, False),
    "gemm_f32_nt": (torch.float32, True),
    "gemm_bf16": (torch.bfloat16, False),
    "gemm_bf16_nt": (torch.bfloat16, True),
    "gemm_f16": (torch.float16, False),
    "gemm_f16_nt": (torch.float16, True),
}
BATCHED = {
    "bmm_f32": (torch.float32, False),
    "bmm_bf16": (torch.bfloat16, False),
    "bmm_bf16_nt": (torch.bfloat16, True),
}
ROWS = {  # op: input type
    "softmax_dyn": torch.float32,
    "layernorm_dyn": torch.float32,
    "softmax_bf16_dyn": torch.bfloat16,
    "row_sum_max_dyn": torch.float32,
    "row_sum_bf16_dyn": torch.bfloat16,
    "row_sum_u8_dyn": torch.uint8,
}
COLUMNS = {
    "col_sum_max_dyn": torch.float32,
    "col_mean_var_dyn": torch.float32,
    "col_mean_var_bf16": torch.bfloat16,
}
EPS = 1e-5
GAIN = 1.5       # the maps' and chains' scalar parameter
U8_SCALE = 0.25


def listed():
    return [
        # The smallest call: one 32 x 32 tile, where the launch is the cost.
        {"name": "gemm_f32_32", "op": "gemm_f32", "m": 32, "n": 32, "k": 32},
        # A projection of a few rows (decode): the weight is read once.
        {"name": "gemm_bf16_decode", "op": "gemm_bf16", "m": 16, "n": 4096, "k": 4096},
        # A projection of a ragged batch of rows, the weight stored [N][K].
        {"name": "gemm_bf16_nt_prefill", "op": "gemm_bf16_nt", "m": 1000, "n": 4096, "k": 1024},
        # The largest contraction, whole tiles everywhere.
        {"name": "gemm_bf16_4096", "op": "gemm_bf16", "m": 4096, "n": 4096, "k": 4096},
        # A 32-bit contraction with odd sizes: ragged tiles, unaligned rows.
        {"name": "gemm_f32_odd", "op": "gemm_f32", "m": 1000, "n": 1500, "k": 1001},
        # Attention scores: many small planes with a short K.
        {"name": "bmm_scores", "op": "bmm_bf16_nt", "b": 32, "m": 500, "n": 500, "k": 64},
        # Softmax over long odd rows (a vocabulary): two reductions and a map.
        {"name": "softmax_long_odd", "op": "softmax_dyn", "r": 4096, "c": 50257},
        # Layernorm of an ordinary activation.
        {"name": "layernorm_768", "op": "layernorm_dyn", "r": 2000, "c": 768},
        # Softmax over 16-bit rows of odd length, computed in 32 bits.
        {"name": "softmax_bf16_odd", "op": "softmax_bf16_dyn", "r": 8192, "c": 2047},
        # Statistics over the leading axis (batch norm).
        {"name": "col_mean_var", "op": "col_mean_var_dyn", "b": 2, "r": 4096, "c": 3000},
        # An elementwise map with broadcast and transposed operands, odd sizes.
        {"name": "map_transposed_odd", "op": "ew_bias_tr", "r": 3001, "c": 2049},
        # A maximum over row sums, per batch.
        {"name": "chain_sum_max", "op": "chain_sum_max", "b": 500, "r": 64, "c": 1000},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "gemm", "batched", "rows", "rows", "columns", "map", "chain"))
    if kind == "gemm":
        op = rng.choice(sorted(GEMM))
        most = 1 << 33 if GEMM[op][0] == torch.float32 else 1 << 36
        whole = rng.random() < 0.5
        while True:
            m, n, k = _log(rng, 1, 8192), _log(rng, 16, 8192), _log(rng, 16, 8192)
            if whole:
                n, k = max(64, n // 64 * 64), max(64, k // 64 * 64)
            if m * n * k <= most:
                return {"op": op, "m": m, "n": n, "k": k}
    if kind == "batched":
        op = rng.choice(sorted(BATCHED))
        m, n = _log(rng, 16, 1024), _log(rng, 16, 1024)
        return {"op": op, "b": _log(rng, 1, 64), "m": m, "n": n, "k": rng.choice((32, 64, 80, 128, rng.randint(32, 256)))}
    if kind == "rows":
        op = rng.choice(sorted(ROWS))
        c = _log(rng, 16, 131072)
        if rng.random() < 0.5:
            c = c // 8 * 8
        return {"op": op, "r": _log(rng, 1, min(65536, (1 << 27) // c)), "c": c}
    if kind == "columns":
        op = rng.choice(sorted(COLUMNS))
        r, c = _log(rng, 16, 65536), _log(rng, 16, 16384)
        if r * c > 1 << 27:
            r = (1 << 27) // c
        case = {"op": op, "r": r, "c": c}
        if op != "col_sum_max_dyn":
            case["b"] = _log(rng, 1, min(16, (1 << 27) // (r * c)))
        return case
    if kind == "map":
        return {"op": rng.choice(("ew_bias_tr", "scale_relu_map")), "r": _log(rng, 16, 8192), "c": _log(rng, 16, 8192)}
    b, r, c = _log(rng, 1, 4096), _log(rng, 4, 1024), _log(rng, 16, 8192)
    while b * r * c > 1 << 27:
        b, r = (b + 1) // 2, (r + 1) // 2
    return {"op": "chain_sum_max", "b": b, "r": r, "c": c}


@functools.lru_cache(maxsize=None)
def _program(op):
    """The compiled program, loaded once: what a user's program holds."""
    return compiler.compile_program(programs.CONFIG_PROGRAMS[op]())


def _inputs(case, seed):
    """The input tensors in declaration order, and the scalars."""
    op = case["op"]
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def normal(shape, dtype=torch.float32, sigma=1.0, mean=0.0):
        return torch.empty(shape, device=DEVICE).normal_(mean, sigma, generator=gen).to(dtype)

    if op in GEMM or op in BATCHED:
        dtype, nt = GEMM.get(op) or BATCHED[op]
        m, n, k = case["m"], case["n"], case["k"]
        lead = (case["b"],) if op in BATCHED else ()
        a = normal(lead + (m, k), dtype)
        w = normal(lead + ((n, k) if nt else (k, n)), dtype, sigma=k ** -0.5)
        return [a, w], ()
    if op in ROWS:
        r, c = case["r"], case["c"]
        if op == "row_sum_u8_dyn":
            return [torch.randint(0, 256, (r, c), device=DEVICE, dtype=torch.uint8, generator=gen)], (U8_SCALE,)
        x = normal((r, c), ROWS[op], sigma=2.0, mean=0.25)
        if op == "layernorm_dyn":
            return [x, normal((c,), sigma=0.1, mean=1.0), normal((c,), sigma=0.1)], (1.0 / c, EPS)
        return [x], ()
    if op in COLUMNS:
        shape = (case["r"], case["c"]) if op == "col_sum_max_dyn" else (case["b"], case["r"], case["c"])
        return [normal(shape, COLUMNS[op], sigma=1.5, mean=0.5)], () if op == "col_sum_max_dyn" else (1.0 / case["r"],)
    if op == "ew_bias_tr":
        r, c = case["r"], case["c"]
        return [normal((r, c)), normal((c, r)), normal((c,)), normal((r,))], ()
    if op == "scale_relu_map":
        r, c = case["r"], case["c"]
        return [normal((r, c)), normal((r, c))], (GAIN,)
    return [normal((case["b"], case["r"], case["c"]))], (GAIN,)


def _output_shapes(case):
    op = case["op"]
    if op in GEMM:
        return [(case["m"], case["n"])]
    if op in BATCHED:
        return [(case["b"], case["m"], case["n"])]
    if op in ("softmax_dyn", "layernorm_dyn", "softmax_bf16_dyn", "ew_bias_tr", "scale_relu_map"):
        return [(case["r"], case["c"])]
    if op in ("row_sum_max_dyn", "row_sum_bf16_dyn"):
        return [(case["r"],)] * 2
    if op == "row_sum_u8_dyn":
        return [(case["r"],)]
    if op == "col_sum_max_dyn":
        return [(case["c"],)] * 2
    if op in COLUMNS:
        return [(case["b"], case["c"])] * 2
    return [(case["b"],)]


def prepare(case, seed):
    tensors, scalars = _inputs(case, seed)
    outputs = [torch.empty(s, device=DEVICE) for s in _output_shapes(case)]
    program = _program(case["op"])
    program.load()
    return {"program": program, "tensors": tensors + outputs, "scalars": scalars, "outputs": outputs}


def run(state):
    state["program"].launch(state["tensors"], scalars=state["scalars"])
    return state["outputs"]


def work(case):
    op = case["op"]
    out = 4 * sum(math.prod(s) for s in _output_shapes(case))
    if op in GEMM or op in BATCHED:
        b, m, n, k = case.get("b", 1), case["m"], case["n"], case["k"]
        size = (GEMM.get(op) or BATCHED[op])[0].itemsize
        return {"bytes": size * b * (m * k + n * k) + out, "flops": 2 * b * m * n * k}
    n = case.get("b", 1) * case["r"] * case["c"]
    if op in ROWS:
        return {"bytes": n * ROWS[op].itemsize + out + (8 * case["c"] if op == "layernorm_dyn" else 0), "flops": 0}
    if op in COLUMNS:
        return {"bytes": n * COLUMNS[op].itemsize + out, "flops": 0}
    if op == "ew_bias_tr":
        return {"bytes": 8 * n + out + 4 * (case["r"] + case["c"]), "flops": 0}
    if op == "scale_relu_map":
        return {"bytes": 8 * n + out, "flops": 0}
    return {"bytes": 4 * n + out, "flops": 0}


def tolerance(case):
    # Bytes are summed in whole numbers, and a map rounds each operation as it
    # is written: both leave no choice.
    if case["op"] in ("row_sum_u8_dyn", "ew_bias_tr", "scale_relu_map"):
        return "exact"
    # Everything else sums in 32 bits, over exact 16-bit products too. About
    # four times the largest distance from the same sums in 64 bits: 5.7e-7
    # for a contraction at K = 1001, growing with the root of K; 9e-8 for the
    # others.
    return {"rel": 4e-6 if case["op"] in GEMM or case["op"] in BATCHED else 1e-6}


def exact(case, seed):
    op = case["op"]
    tensors, scalars = _inputs(case, seed)
    if op in GEMM or op in BATCHED:
        a, w = (t.double() for t in tensors)
        if (GEMM.get(op) or BATCHED[op])[1]:
            w = w.transpose(-1, -2).contiguous()
        return [torch.matmul(a, w)]
    x = tensors[0].double()
    if op in ("softmax_dyn", "softmax_bf16_dyn"):
        x -= x.amax(1, keepdim=True)
        x.exp_()
        return [x.div_(x.sum(1, keepdim=True))]
    if op == "layernorm_dyn":
        x -= x.mean(1, keepdim=True)
        x /= (x.square().mean(1, keepdim=True) + EPS).sqrt()
        return [x * tensors[1].double() + tensors[2].double()]
    if op in ("row_sum_max_dyn", "row_sum_bf16_dyn"):
        return [x.sum(1), x.amax(1)]
    if op == "row_sum_u8_dyn":
        return [x.sum(1) * U8_SCALE]
    if op == "col_sum_max_dyn":
        return [x.sum(0), x.amax(0)]
    if op in COLUMNS:
        mean = x.mean(1)
        return [mean, (x - mean[:, None]).square_().mean(1)]
    if op == "ew_bias_tr":
        z, g, b = (t.double() for t in tensors[1:])
        return [x * g + b[:, None] + z.t()]
    if op == "scale_relu_map":
        return [(GAIN * x + tensors[1].double()).clamp_min(0)]
    return [x.sum(2).amax(1) * GAIN]
