"""The small contraction's forms: larger tiles as functions of their own, which
the plan's form records put in the 32x32 kernel's place. Host-only: the rule,
the record, and that every compiled function is free of scratch; the results
are tests/test_gemm_any.py's."""
import ctypes
import glob
import os
import re
import subprocess

import pytest

from tcacomp_amd import _lib, compiler, programs
from tcacomp_amd.compiler import TensorDesc

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def _parse(text):
    h = ctypes.c_void_p()
    return _lib.lib().tca_program_parse(text.encode(), ctypes.byref(h)), h


def _form(plan, dims):
    """(function, workgroups) that a launch of the `_s` kernel takes, by the
    plan's text alone; workgroups None for the kernel itself."""
    def term(t):
        prod, div = t.split("/")
        v = 1
        for f in prod.split("*"):
            v *= dims[f]
        return -(-v // int(div))

    lines = plan.split("\n")
    at = next(i for i, l in enumerate(lines) if re.match(r"kernel \S+_k0_s ", l))
    for l in lines[at + 1:]:
        w = l.split()
        if w[0] in ("kernel", "end"):
            return "", None
        if w[0] != "form":
            continue
        pos, grid, ok = 4, None, True
        for _ in range(int(w[3])):
            v = 1
            for t in w[pos + 2:pos + 2 + int(w[pos + 1])]:
                v *= term(t)
            grid = v if grid is None else grid
            ok = ok and v >= int(w[pos])
            pos += 2 + int(w[pos + 1])
        assert pos == len(w), l
        if ok:
            return re.search(r"_s(\d+x\d+)$", w[1]).group(1), min(grid, int(w[2]) or grid)
    raise AssertionError("no end")


@pytest.mark.parametrize("name,dims,form,grid", [
    # 192 workgroups of a tile each, or the next smaller tile
    ("gemm_bf16", (1024, 1024, 4096), "64x64", 256), ("gemm_bf16", (512, 2048, 40), "64x64", 256),
    ("gemm_bf16", (100, 10000, 64), "64x64", 314), ("gemm_f32", (1000, 1000, 512), "64x64", 256),
    ("gemm_bf16", (60, 8001, 64), "64x32", 251), ("gemm_f32", (33, 31775, 64), "64x64", 497),
    ("gemm_bf16", (512, 512, 4096), "", None), ("gemm_f32", (64, 2048, 1024), "", None),
    ("gemm_bf16", (32, 32768, 64), "", None),     # 32 rows: no larger tile has fewer rows to waste
    # rows shorter than a chunk
    ("gemm_bf16", (1000, 1000, 7), "", None), ("gemm_bf16", (1000, 1000, 8), "64x64", 256),
    ("gemm_bf16", (150000, 6, 64), "", None), ("gemm_bf16_nt", (150000, 6, 64), "64x32", 2344),
    ("gemm_f32", (1000, 1000, 3), "", None), ("gemm_f32", (150000, 4, 64), "64x32", 2344),
    ("gemm_bf16", (1000, 1000, 0), "", None),
    # batches: as many tiles together; forms that walk stop at 1024 workgroups
    ("bmm_bf16_nt", (32, 500, 500, 64), "128x128", 512), ("bmm_bf16", (64, 1000, 1000, 64), "128x128", 1024),
    ("bmm_bf16", (64, 64, 1000, 64), "64x64", 1024), ("bmm_bf16", (200, 64, 64, 64), "64x64", 200),
    ("bmm_bf16", (11, 128, 128, 64), "", None), ("bmm_f32", (32, 500, 500, 64), "64x64", 2048),
    ("bmm_f32", (500, 40, 32, 64), "64x32", 500)])
def test_form_rule(name, dims, form, grid):
    plan = programs.CONFIG_PROGRAMS[name]().emit().plan
    names = ("B", "M", "N", "K")[4 - len(dims):]
    assert _form(plan, dict(zip(names, dims))) == (form, grid)


@pytest.mark.parametrize("name", ["gemm_f32", "gemm_f32_nt", "gemm_bf16", "gemm_bf16_nt", "gemm_f16", "bmm_bf16", "bmm_f32",
                                  "bmm_f32_nt_shared_a", "mm_mid"])
def test_forms_compute_the_kernel(name):
    """Every form is a function of the source whose tile is its name's, and no
    form runs where K is split over workgroups (192 tiles are more than 256
    of 32x32)."""
    e = (programs.CONFIG_PROGRAMS.get(name) or programs.SUITE[name][0])().emit()
    for s, m, n in re.findall(r"form (\S+_s(\d+)x(\d+)) ", e.plan):
        assert re.search(r"void [^;{]*\b%s\(" % s, e.source)
        body = e.source[e.source.index(" %s(" % s):]
        body = body[:body.index("\n}\n")]
        assert re.search(r"gemm_small_form<\w+, \w+, %su, %su, \w+>" % (m, n), body) and "gemm_split_chunks" not in body
        assert ("gridDim.x" in body) == ("form %s 1024 " % s in e.plan)
    for M in (33, 64, 65, 96, 97, 128, 129, 1000):
        for N in range(1, 40000, 97):
            if -(-M // 64) * -(-N // 32) >= 192:
                assert -(-M // 32) * -(-N // 32) > 256, (M, N)


PLAN = ("tca-plan 1\nprogram s\ndim M 0\ntensor x f32 in 1 M\nkernel k 64 0 1 M/4\narg ptr x\n"
        "form k2 70 2 10 1 M/8 3 2 M/1 M/1\nend\n")


def test_form_record_survives_the_printed_form():
    rc, h = _parse(PLAN)
    assert rc == 0, _lib.last_error()
    text = _lib.lib().tca_program_plan_text(h).decode()
    assert "form k2 70 2 10 1 M/8 3 2 M/1 M/1\n" in text
    assert _parse(text)[0] == 0
    # a program's selection and arguments are its kernels': forms are no kernels
    arr = compiler._descriptors([TensorDesc(0x1000, (800,), 0)])
    out, grids = (ctypes.c_uint8 * 1)(), (ctypes.c_uint64 * 1)()
    assert _lib.lib().tca_program_selected(h, arr, 1, None, 0, out, grids, None, 1) == 0
    assert grids[0] == 200


@pytest.mark.parametrize("bad", ["form k2", "form k2 0 0", "form k2 0 1 5", "form k2 0 1 5 1", "form k2 0 1 5 1 Q/1",
                                 "form k2 0 1 5 1 M/pack", "form k2 0 1 5 1 M/1 7", "form k2 0 2 5 1 M/1",
                                 "form k2 x 1 5 1 M/1", "form k2 0 1 5 99999999999 M/1"])
def test_form_record_refuses(bad):
    rc, _ = _parse(re.sub(r"form .*", bad, PLAN))
    assert rc != 0


def test_small_functions_have_no_scratch():
    """One function per tile shape: none spills, whatever the others hold."""
    bundler = os.path.join(ROCM, "llvm", "bin", "clang-offload-bundler")
    readelf = os.path.join(ROCM, "llvm", "bin", "llvm-readelf")
    files = [f for f in glob.glob(os.path.join(compiler.KCACHE, "*.hsaco")) if "_sm(" in open(f[:-6] + ".hip").read()]
    if not files or not os.path.exists(bundler):
        pytest.skip("no prebuilt contractions")
    seen = 0
    for f in files:
        r = subprocess.run([bundler, "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + f,
                            "--output=-"], capture_output=True)
        assert r.returncode == 0, r.stderr
        notes = subprocess.run([readelf, "--notes", "-"], input=r.stdout, capture_output=True).stdout.decode()
        for k in notes.split(".agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", k).group(1)
            if re.search(r"_s(m|\d+x\d+)?$", name):
                seen += 1
                assert re.search(r"\.private_segment_fixed_size:\s+(\d+)", k).group(1) == "0", name
    assert seen > 20
