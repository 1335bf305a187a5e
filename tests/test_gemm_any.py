"""The contractions' any-shape kernels (gemm16_any, gemm_f32_any) and the small
kernel's tile shapes: which launches take them, and their results at the sizes
where they can go wrong.

Host-only: every tile of a 16-bit plane has exactly one owner. The direct-to-LDS
kernels and the any-shape kernel decide on the device with the same rule
(gemm16_on_whole_tiles, compiled here for the host); the plan's guards may
only skip a launch that the rule leaves idle.

GPU: small-integer operands, so every product and partial sum is exact in
fp32 and every output must equal the float64 product."""
import os
import random
import subprocess
import sys

import numpy as np
import pytest

import oracle
from helpers import canaries, compiled, host, out_dev, run, to_dev
from tcacomp_amd.compiler import TensorDesc

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WHOLE_MIN = 128 << 16


@pytest.fixture(scope="module")
def on_whole_tiles(tmp_path_factory):
    out = tmp_path_factory.mktemp("gemm_edge") / "gemm_edge"
    hipcc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-I",
                        os.path.join(REPO, "tcacomp_amd", "csrc", "include"),
                        os.path.join(REPO, "tests", "c", "gemm_edge.hip"), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]

    def ask(shapes, *args):
        p = subprocess.run([str(out)] + list(args), input="".join("%d %d %d %d\n" % s for s in shapes), capture_output=True,
                           text=True, timeout=60)
        assert p.returncode == 0, p.stderr
        if args == ("steps",):
            return [[int(v) for v in l.split()] for l in p.stdout.splitlines()]
        return [bool(int(v)) for v in p.stdout.split()]
    return ask


def _shapes(rng, count):
    for _ in range(count):
        m, n, k = (max(1, int(2 ** rng.uniform(0, 14))) for _ in range(3))
        if rng.random() < 0.6:
            m, n = max(256, m // 256 * 256), max(256, n // 256 * 256)
        if rng.random() < 0.7:
            k = max(32, k // 32 * 32)
        if rng.random() < 0.3:
            n = max(8, n // 8 * 8)
        b = rng.choice((1, 1, 1, 2, 7))
        if m * n > 1 << 20 and max(m * n, m * k, n * k) * b < 1 << 31:
            yield m, n, k, b


@pytest.mark.parametrize("name", ["bmm_bf16", "bmm_bf16_nt"])
def test_every_tile_has_one_kernel(on_whole_tiles, name):
    from tcacomp_amd import compiler, programs
    prog = compiler.CompiledProgram(name, programs.CONFIG_PROGRAMS[name]().emit(), "")
    shapes = list(_shapes(random.Random(11), 3000))
    shapes += [(2048, 4096, 4096, 1), (2048, 4096 - 256, 4096, 1), (257, 36266, 512, 1), (4096, 4096, 192, 1),
               (4352, 4096, 64, 1), (4100, 4096, 4096, 1), (1024, 1025, 4096, 8), (2048, 2048, 1024, 2)]
    assert len(shapes) > 500
    for (m, n, k, b), whole in zip(shapes, on_whole_tiles(shapes)):
        sel = prog.selected_symbols([TensorDesc(0x1000, (b, m, k), 2),
                                     TensorDesc(0x1000, (b, n, k) if name.endswith("nt") else (b, k, n), 2),
                                     TensorDesc(0x1000, (b, m, n), 0)])
        sel = {s[len("tca_%s_k0" % name):] for s in sel}
        has_whole = whole and m >= 256 and n >= 256
        edges = not has_whole or m % 256 != 0 or n % 256 != 0
        if has_whole:  # the kernel the K rule names
            assert ("_w" if k % 64 == 0 and k >= 256 else "_v") in sel, (m, n, k, b, sel)
        if edges:
            assert "" in sel, (m, n, k, b, sel)
        if m * n * b < WHOLE_MIN:  # no tile is the direct-to-LDS kernels': neither is launched
            assert sel == {""}, (m, n, k, b, sel)
        assert not {"_s", "_sm"} & sel


def test_every_tile_has_one_kernel_without_the_small_kernel(on_whole_tiles):
    """A plan of the tile kernels alone: whole tiles are the direct-to-LDS
    kernels' however few they are."""
    from tcacomp_amd import compiler, programs
    from tcacomp_amd.pkg import EMIT_NO_GEMM_SPLIT
    prog = compiler.CompiledProgram("gemm_bf16", programs.CONFIG_PROGRAMS["gemm_bf16"]().emit(flags=EMIT_NO_GEMM_SPLIT), "")
    shapes = [(256, 256, 256, 1), (256, 256, 32, 1), (300, 256, 64, 1), (255, 4096, 4096, 1), (512, 520, 96, 1),
              (512, 516, 96, 1), (2048, 2048, 4096, 1), (16, 16, 16, 1), (256, 256, 100, 1)]
    for (m, n, k, _), whole in zip(shapes, on_whole_tiles(shapes, "all")):
        sel = {s[len("tca_gemm_bf16_k0"):] for s in prog.selected_symbols(
            [TensorDesc(0x1000, (m, k), 2), TensorDesc(0x1000, (k, n), 2), TensorDesc(0x1000, (m, n), 0)])}
        assert whole == (k % 32 == 0 and n % 8 == 0)
        has_whole = whole and m >= 256 and n >= 256
        assert (("_w" if k % 64 == 0 and k >= 256 else "_v") in sel) == has_whole, (m, n, k, sel)
        assert ("" in sel) == (not has_whole or m % 256 != 0 or n % 256 != 0), (m, n, k, sel)


def test_short_slices_take_no_empty_steps(on_whole_tiles):
    """The fp32 kernel steps through K 8 deep: over all groups of waves as many
    steps as hold any of K (whole 32-deep slices doubled the work at K = 16)."""
    shapes = [(1, 1, k, g) for k in (0, 1, 7, 8, 9, 16, 24, 31, 32, 33, 64, 65, 100, 127, 1000, 1001) for g in (1, 2, 4)]
    for (_, _, k, g), steps in zip(shapes, on_whole_tiles(shapes, "steps")):
        assert sum(steps) == -(-k // 8), (k, g, steps)
        assert steps[0] <= 4 * -(-(-(-k // 32)) // g) and steps[0] - steps[-1] <= 4, (k, g, steps)


# M, N, K: remainders of the 64- and 128-row tiles and of the 64-deep slice, K
# of one element, one chunk and one slice either side, rows of every
# alignment, [K][N] rows shorter than a chunk, few rows, few columns, and
# planes that take the 64-row tile (few 128x128 tiles), the 128-row tile
# (many) and whole 256x256 tiles with edges.
SHAPES = [(1025, 1025, 1), (1025, 1027, 7), (1030, 1029, 8), (1031, 1026, 9), (1089, 1032, 63), (1024, 1032, 64),
          (1152, 1153, 65), (1100, 1101, 127), (1100, 1102, 128), (1100, 1104, 129), (1281, 1031, 200),
          (200001, 6, 70), (210000, 5, 72), (131080, 9, 257), (3, 400000, 65), (64, 16500, 130), (65, 16500, 66),
          (2100, 2300, 333), (2048, 2049, 320), (3100, 3330, 96), (4100, 4104, 256), (3000, 5888, 64)]


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _dev(a, name, gpu):
    import torch
    a = np.ascontiguousarray(a)
    if "_f32" in name:
        return to_dev(a, gpu)
    f16 = "_f16" in name
    if f16:
        return to_dev(a.astype(np.float16), gpu)
    return to_dev(oracle.to_bf16_bits(a).view(np.int16), gpu).view(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("name", ["gemm_bf16", "gemm_bf16_nt", "gemm_f16", "gemm_f32", "gemm_f32_nt"])
def test_any_shape_exact(gpu, M, N, K, name):
    _say("gemm any", name, M, N, K)
    nt, code = name.endswith("_nt"), 0 if "_f32" in name else 1 if "_f16" in name else 2
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a = rng.integers(-4, 5, (M, K)).astype(np.float32)
    b = rng.integers(-4, 5, (K, N)).astype(np.float32)
    p = compiled(name)
    bd = np.ascontiguousarray(b.T) if nt else b
    sel = p.selected_symbols([TensorDesc(0x1000, (M, K), code), TensorDesc(0x1000, bd.shape, code),
                              TensorDesc(0x1000, (M, N), 0)])
    assert "tca_%s_k0%s" % (name, "_v" if code == 0 and min(M, N) >= 4096 else "") in sel, sel
    c = out_dev((M, N), gpu)
    run(p, [_dev(a, name, gpu), _dev(bd, name, gpu), c])
    got = host(c)
    assert canaries(got) == 0
    assert np.array_equal(got, a @ b)  # exact in fp32: partial sums below 2^24


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["bmm_bf16", "bmm_bf16_nt", "bmm_f32"])
@pytest.mark.parametrize("B,M,N,K", [(3, 1025, 1027, 77), (2, 130, 8300, 64), (9, 1024, 1152, 96)])
def test_any_shape_batched_exact(gpu, name, B, M, N, K):
    _say("bmm any", name, B, M, N, K)
    nt = name.endswith("_nt")
    rng = np.random.default_rng(B + M + N + K)
    a = rng.integers(-4, 5, (B, M, K)).astype(np.float32)
    b = rng.integers(-4, 5, (B, K, N)).astype(np.float32)
    c = out_dev((B, M, N), gpu)
    run(compiled(name), [_dev(a, name, gpu), _dev(b.transpose(0, 2, 1) if nt else b, name, gpu), c])
    assert np.array_equal(host(c), np.matmul(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["gemm_bf16", "gemm_bf16_nt", "gemm_f32", "gemm_f32_nt"])
def test_nonfinite_operands_stay_in_their_rows(gpu, name):
    """Infinities and NaN at the ends of rows: a chunk loaded from before the
    end of its row must not bring a neighbour's values in, nor a clamped row
    leave its tile."""
    import torch
    M, N, K = 1030, 1029, 75
    nt = name.endswith("_nt")
    rng = np.random.default_rng(3)
    a = rng.integers(-4, 5, (M, K)).astype(np.float32)
    b = rng.integers(-4, 5, (K, N)).astype(np.float32)
    a[5, K - 1], a[M - 1, 0], b[K - 1, 7], b[0, N - 1] = np.inf, np.nan, -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    c = out_dev((M, N), gpu)
    dtype = torch.float32 if "_f32" in name else torch.bfloat16
    ta = torch.from_numpy(a).to(gpu).to(dtype)
    tb = torch.from_numpy(np.ascontiguousarray(b.T) if nt else b).to(gpu).to(dtype)
    run(compiled(name), [ta, tb, c])
    assert np.array_equal(host(c), want.astype(np.float32), equal_nan=True)


# Planes of at most 2^20 outputs: the small kernel's tile shapes (32x32 with K
# whole and split over workgroups, 64x32, 64x64, 128x128), ragged in M, N and
# K, rows of every alignment, more tiles than workgroups (the grid's stride).
SMALL = [("gemm_bf16", 1, 16, 4096, 4100), ("gemm_bf16", 1, 33, 777, 1001), ("gemm_bf16_nt", 1, 33, 777, 1001),
         ("gemm_f16", 1, 17, 3000, 65), ("gemm_bf16_nt", 1, 5, 9, 3001), ("gemm_bf16", 1, 60, 8001, 129),
         ("gemm_bf16_nt", 1, 60, 8001, 131), ("gemm_bf16", 1, 61, 9000, 8), ("gemm_bf16", 1, 700, 1301, 200),
         ("gemm_bf16_nt", 1, 1000, 1001, 333), ("gemm_f16_nt", 1, 1000, 1001, 1), ("gemm_bf16", 1, 3, 200001, 66),
         ("gemm_bf16", 1, 150001, 5, 66), ("gemm_bf16", 1, 150001, 9, 66), ("bmm_bf16_nt", 32, 500, 500, 64),
         ("bmm_bf16", 20, 500, 501, 77), ("bmm_bf16", 300, 129, 130, 8), ("bmm_bf16_nt", 70, 200, 200, 9),
         ("gemm_f32", 1, 16, 4096, 2050), ("gemm_f32", 1, 33, 777, 1001), ("gemm_f32_nt", 1, 33, 777, 1003),
         ("gemm_f32", 1, 61, 9001, 4), ("gemm_f32_nt", 1, 60, 8001, 67), ("gemm_f32", 1, 1000, 1001, 333),
         ("gemm_f32_nt", 1, 1001, 1000, 130), ("gemm_f32", 1, 1000, 1001, 3), ("gemm_f32", 1, 150001, 3, 66),
         ("gemm_f32", 1, 150001, 6, 35), ("bmm_f32", 32, 500, 501, 66), ("bmm_f32", 2000, 31, 33, 17),
         ("bmm_bf16", 3, 40, 72, 3000), ("bmm_bf16_nt", 500, 65, 33, 40), ("bmm_bf16", 2000, 31, 33, 17)]


@pytest.mark.gpu
@pytest.mark.parametrize("name,B,M,N,K", SMALL)
def test_small_tile_shapes_exact(gpu, name, B, M, N, K):
    _say("small tiles", name, B, M, N, K)
    nt, batched = name.endswith("_nt"), name.startswith("bmm")
    rng = np.random.default_rng(B + M + N + K)
    a = rng.integers(-4, 5, (B, M, K)).astype(np.float32)
    b = rng.integers(-4, 5, (B, K, N)).astype(np.float32)
    bd = b.transpose(0, 2, 1) if nt else b
    c = out_dev((B, M, N) if batched else (M, N), gpu)
    run(compiled(name), [_dev(a if batched else a[0], name, gpu), _dev(bd if batched else bd[0], name, gpu), c])
    assert np.array_equal(host(c).reshape(B, M, N), np.matmul(a, b))


def test_stride_record():
    """`stride n` limits a kernel's workgroups to n after its split record;
    it survives the printed form, and zero or a missing number is refused."""
    import ctypes
    from tcacomp_amd import _lib, compiler
    text = ("tca-plan 1\nprogram s\ndim M 0\ntensor x f32 in 1 M\nkernel k 64 0 1 M/4\narg ptr x\n"
            "split M 10 100000 0 1 M/64\nstride 70\nend\n")
    for t in (text, None):
        if t is None:
            t = _lib.lib().tca_program_plan_text(h).decode()
            assert "stride 70\n" in t
        h = ctypes.c_void_p()
        assert _lib.lib().tca_program_parse(t.encode(), ctypes.byref(h)) == 0, _lib.last_error()
        for m, grid in ((8, 2), (20, 10), (100, 70), (10 ** 6, 70)):
            arr = compiler._descriptors([TensorDesc(0x1000, (m,), 0)])
            out, grids = (ctypes.c_uint8 * 1)(), (ctypes.c_uint64 * 1)()
            assert _lib.lib().tca_program_selected(h, arr, 1, None, 0, out, grids, None, 1) == 0
            assert grids[0] == grid, (m, grids[0])
    for bad in ("stride 0", "stride", "stride x"):
        h = ctypes.c_void_p()
        assert _lib.lib().tca_program_parse(text.replace("stride 70", bad).encode(), ctypes.byref(h)) != 0
        assert "stride <workgroups>" in _lib.last_error()
