"""Short rows whose length is no multiple of the widest vector: the plan's
lanes per row, and with them the blocks it launches, are those of the body that
runs, and the wide bodies are forms taken by the row length and the number of
elements."""
import ctypes
import re

import numpy as np
import pytest

from helpers import canaries, compiled, host, out_dev, run, to_dev
from tcacomp_amd import _lib, compiler, programs
from tcacomp_amd.compiler import TensorDesc

ROWS = ["softmax_dyn", "layernorm_dyn", "softmax_bf16_dyn", "row_sum_max_dyn", "row_sum_bf16_dyn", "row_sum_u8_dyn",
        "softmax_affine_dyn", "row_stats_shift_dyn", "chain_sum_max"]


def _geometry(plan):
    """{function: elements per lane that the plan packs by} of a program's
    packed kernels and their forms."""
    out, kernel, form = {}, None, None
    for l in plan.split("\n"):
        w = l.split()
        if w and w[0] == "kernel":
            kernel, form = w[1], None
        elif w and w[0] == "pack":
            out[kernel] = int(w[2])
        elif w and w[0] == "form":
            form = w[1]
        elif w and w[0] == "formpack":
            assert out.get(form, int(w[1])) == int(w[1])
            out[form] = int(w[1])
    return out


@pytest.mark.parametrize("name", ROWS)
def test_plan_packs_by_the_body_that_runs(name):
    """Every body that a row kernel calls holds as many elements per lane as
    its plan says (4 vectors when it streams): the device picks the lanes per
    row from its body, the host the blocks from the plan."""
    e = programs.CONFIG_PROGRAMS[name]().emit()
    geometry = _geometry(e.plan)
    seen = 0
    for sym, epl in geometry.items():
        m = re.search(r"__launch_bounds__\(\d+\) %s\(.*?\n}\n" % sym, e.source, re.S)
        bodies = re.findall(r"_rows<(\d+)u, (\d+)u,", m.group(0))
        assert bodies, sym
        for v, nv in bodies:
            seen += 1
            assert int(v) * (int(nv) or 4) == epl, (sym, bodies, epl)
    assert seen > 4


def _selected(name, dtype, R, C, inputs=1, outputs=()):
    e = programs.CONFIG_PROGRAMS[name]().emit()
    h = ctypes.c_void_p()
    assert _lib.lib().tca_program_parse(e.plan.encode(), ctypes.byref(h)) == 0, _lib.last_error()
    arr = compiler._descriptors([TensorDesc(0x1000, (R, C), dtype)] + [TensorDesc(0x1000, s, 0) for s in outputs])
    syms = e.kernel_symbols()
    out, grids = (ctypes.c_uint8 * len(syms))(), (ctypes.c_uint64 * len(syms))()
    rc = _lib.lib().tca_program_selected(h, arr, 1 + len(outputs), None, 0, out, grids, None, len(syms))
    assert rc == 0, _lib.last_error()
    return e.plan, [(s, g) for s, f, g in zip(syms, out, grids) if f]


@pytest.mark.parametrize("name,dtype,R,C,grid", [
    ("row_sum_u8_dyn", 7, 8192, 255, 2048), ("row_sum_u8_dyn", 7, 1024, 511, 512),
    ("softmax_bf16_dyn", 2, 2048, 127, 256), ("softmax_dyn", 0, 8192, 31, 256),
    ("row_sum_bf16_dyn", 2, 100000, 127, 2048)])  # many rows: the blocks walk them
def test_short_rows_fill_the_chip(name, dtype, R, C, grid):
    outs = [(R, C)] if "softmax" in name else [(R,)] * (1 if "u8" in name else 2)
    _, sel = _selected(name, dtype, R, C, outputs=outs)
    assert [g for _, g in sel] == [grid], sel


def _form(plan, sym, R, C):
    lines = plan.split("\n")
    at = next(i for i, l in enumerate(lines) if l.startswith("kernel %s " % sym))
    for l in lines[at + 1:]:
        w = l.split()
        if w[0] in ("kernel", "end"):
            return ""
        if w[0] != "form":
            continue
        pos, ok = 4, True
        for i in range(int(w[3])):
            terms = w[pos + 2:pos + 2 + int(w[pos + 1])]
            if i > 0:  # the first is the grid, of any size
                v = 1
                for t in terms:
                    assert t in ("R/1", "C/1")
                    v *= R if t[0] == "R" else C
                ok = ok and v >= int(w[pos])
            pos += 2 + len(terms)
        if ok:
            return w[1][len(sym):]


@pytest.mark.parametrize("name,dtype,R,C,form", [
    # several passes: wide from 600000 elements on, cached up to 64 vectors
    ("softmax_dyn", 0, 65536, 32 - 1, ""), ("softmax_dyn", 0, 20000, 33, "rc"), ("softmax_dyn", 0, 18000, 33, ""),
    ("softmax_dyn", 0, 65536, 255, "rc"), ("softmax_dyn", 0, 65536, 257, "r"), ("softmax_dyn", 0, 500, 1023, ""),
    ("softmax_dyn", 0, 2000, 1023, "r"), ("softmax_dyn", 0, 1, 2049, "r"), ("softmax_dyn", 0, 1, 2047, ""),
    ("softmax_dyn", 0, 20000, 62, "rc"), ("softmax_dyn", 0, 1, 4098, "r"),
    # one pass: wide always, over 4-element vectors with the narrow body's lanes
    ("row_sum_u8_dyn", 7, 8192, 511, ""), ("row_sum_u8_dyn", 7, 1, 513, "rc"), ("row_sum_u8_dyn", 7, 9, 1025, "r"),
    ("row_sum_bf16_dyn", 2, 1, 129, "rc"), ("row_sum_bf16_dyn", 2, 1, 513, "r"), ("row_sum_max_dyn", 0, 65536, 1023, "rc"),
    ("row_sum_max_dyn", 0, 1, 31, "")])
def test_wide_form_rule(name, dtype, R, C, form):
    outs = [(R, C)] if "softmax" in name else [(R,)] * (1 if "u8" in name else 2)
    plan, sel = _selected(name, dtype, R, C, outputs=outs)
    assert len(sel) == 1
    assert _form(plan, sel[0][0], R, C) == form


PLAN = ("tca-plan 1\nprogram s\ndim R 0\ndim C 0\ntensor x f32 in 2 R C\nkernel k 1024 0 1 R/pack\narg ptr x\n"
        "pack C 4 256\nform k2 0 2 0 1 R/pack 33 1 C/1\nformpack 16\nend\n")


def test_formpack_record():
    def parse(text):
        h = ctypes.c_void_p()
        return _lib.lib().tca_program_parse(text.encode(), ctypes.byref(h)), h
    rc, h = parse(PLAN)
    assert rc == 0, _lib.last_error()
    text = _lib.lib().tca_program_plan_text(h).decode()
    assert "form k2 0 2 0 1 R/pack 33 1 C/1\nformpack 16\n" in text and parse(text)[0] == 0
    for old, new in (("formpack 16", "formpack 0"), ("formpack 16", "formpack"), ("form k2 0 2 0 1 R/pack 33 1 C/1\n", ""),
                     ("pack C 4 256\n", ""), ("33 1 C/1", "33 1 C/pack")):
        assert parse(PLAN.replace(old, new, 1))[0] != 0, (old, new)


# Row lengths on both sides of each switch, with rows for the wide forms (from
# 600000 elements) and for narrow bodies whose blocks walk the rows.
CASES = [(70000, 31), (70001, 30), (18200, 33), (20001, 35), (12801, 47), (9700, 62), (8000, 126), (4801, 127), (2401, 254),
         (2400, 255), (2400, 257), (2399, 258), (1201, 511), (1200, 513), (601, 1021), (300, 2047), (300, 2049), (300, 2050)]


@pytest.mark.gpu
@pytest.mark.parametrize("R,C", CASES)
def test_many_rows(gpu, R, C):
    import torch
    rng = np.random.default_rng(R + C)
    xi = rng.integers(-8, 9, (R, C)).astype(np.float32)
    s, m = out_dev((R,), gpu), out_dev((R,), gpu)
    run(compiled("row_sum_max_dyn"), [to_dev(xi, gpu), s, m])
    assert np.array_equal(host(s), xi.sum(1, dtype=np.float64).astype(np.float32)) and np.array_equal(host(m), xi.max(1))
    run(compiled("row_sum_bf16_dyn"), [to_dev(xi, gpu).to(torch.bfloat16), s, m])
    assert np.array_equal(host(s), xi.sum(1, dtype=np.float64).astype(np.float32)) and np.array_equal(host(m), xi.max(1))
    u = (xi + 8).astype(np.uint8)
    run(compiled("row_sum_u8_dyn"), [to_dev(u, gpu), s], scalars=[0.25])
    assert np.array_equal(host(s), u.sum(1, dtype=np.int64).astype(np.float32) * np.float32(0.25))
    x = (rng.standard_normal((R, C)) * 2 + 0.5).astype(np.float32)
    x[1, C - 1] = 30.0
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    d, y = to_dev(x, gpu), out_dev((R, C), gpu)
    for out in (y, d):  # in place as well: each element is written by the lane that read it
        run(compiled("softmax_dyn"), [d, out])
        got = host(out)
        assert canaries(got) == 0
        assert (np.abs(got - want) <= 5e-6 * want).all()  # as tests/test_gpu_ragged_rows.py derives it
    xb = to_dev(x, gpu).to(torch.bfloat16)
    b64 = host(xb.float()).astype(np.float64)
    e = np.exp(b64 - b64.max(1, keepdims=True))
    run(compiled("softmax_bf16_dyn"), [xb, y])
    assert (np.abs(host(y) - e / e.sum(1, keepdims=True)) <= 5e-6 * e / e.sum(1, keepdims=True)).all()
    g, b = (rng.standard_normal(C) + 1).astype(np.float32), rng.standard_normal(C).astype(np.float32)
    run(compiled("layernorm_dyn"), [to_dev(x, gpu), to_dev(g, gpu), to_dev(b, gpu), y], scalars=[1.0 / C, 1e-5])
    mean, var = x64.mean(1, keepdims=True), x64.var(1, keepdims=True)
    want = (x64 - mean) / np.sqrt(var + 1e-5) * g + b
    bound = 1e-5 * (np.abs(want) + np.abs(g) + np.abs(b)) + 1e-6 * np.abs(g) * np.sqrt((x64 ** 2).mean(1, keepdims=True)) \
        / np.sqrt(var + 1e-5)
    assert (np.abs(host(y) - want) <= bound).all()


# What the narrow body's sums of 4 elements a lane give for these distributions
# (two seeds and more): 2% covers the seed and another order of as many roundings.
@pytest.mark.gpu
@pytest.mark.parametrize("name,R,C,bound", [("softmax_dyn", 20000, 62, 6.42e-8), ("softmax_dyn", 20000, 127, 6.22e-8),
                                            ("softmax_dyn", 8192, 255, 6.35e-8), ("softmax_dyn", 2000, 511, 6.55e-8),
                                            ("softmax_bf16_dyn", 20000, 127, 6.27e-8),
                                            ("softmax_bf16_dyn", 2000, 511, 6.52e-8)])
def test_wide_forms_no_further_from_64_bits(gpu, name, R, C, bound):
    import torch
    gen = torch.Generator(device=gpu)
    gen.manual_seed(C)
    x = torch.empty((R, C), device=gpu).normal_(0.25, 2.0, generator=gen)
    if "bf16" in name:
        x = x.to(torch.bfloat16)
    y = torch.empty((R, C), device=gpu)
    run(compiled(name), [x, y])
    want = torch.softmax(x.double(), 1)
    error = ((y.double() - want).norm() / want.norm()).item()
    print(name, R, C, error, flush=True)
    assert error <= 1.02 * bound
