"""LDS that the lanes of one wave exchange (the small contraction's operand
stages): the compiler sees one thread, so a fence must stand between a write
and the next read of it, and between a read and the next write, in the code
that it makes. Host-only: the device code is compiled, not run."""
import os
import re
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


def _unfenced(lines):
    """(accesses, faults): LDS accesses of one block in order, and those of the
    other kind than the last one with no fence between."""
    last, faults, count = "", [], 0
    for line in lines:
        if re.search(r"fence syncscope|s\.barrier", line):
            last = ""
            continue
        if re.match(r"\s*store .*addrspace\(3\)", line):
            kind = "store"
        elif re.search(r"= load .*addrspace\(3\)|ds\.read\.tr", line) and "declare" not in line:
            kind = "load"
        else:
            continue
        count += 1
        if last not in ("", kind):
            faults.append(line.strip())
        last = kind
    return count, faults


def test_the_check_sees_a_missing_fence():
    ir = ["  store <4 x i32> %v, ptr addrspace(3) %p, align 16", "  %x = load <4 x i32>, ptr addrspace(3) %q, align 16"]
    assert _unfenced(ir) == (2, [ir[1].strip()])
    assert _unfenced([ir[0], '  fence syncscope("wavefront") acq_rel, !mmra !1', ir[1]]) == (2, [])


def test_every_exchange_is_fenced(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "w.ll"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-device-only", "-S", "-emit-llvm", "-O2", "-std=c++17",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I",
                        os.path.join(REPO, "tcacomp_amd", "csrc", "include"),
                        os.path.join(REPO, "tests", "c", "wave_exchange.hip"), "-o", str(out)], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"define [^\n]*amdgpu_kernel[^\n]*@(\w+)\((.*?)\n}\n", out.read_text(), re.S)
    assert len(kernels) == 8
    for name, body in kernels:
        blocks = re.split(r"\n(?=\d+:|[\w.]+:)", body)
        seen = 0
        for b in blocks:
            count, faults = _unfenced(b.split("\n"))
            seen += count
            assert not faults, (name, len(faults), faults[0])
        assert seen > 20, name
