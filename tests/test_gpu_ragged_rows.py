"""Rows whose length is no multiple of the widest vector: the streaming
family's narrow-width kernels move whole unaligned vectors and give each
element past the last one to a lane of its own. Row lengths on both sides of
every switch (the narrow body for short rows, the register caches, streamed
rows), every tail length, each element type, against float64 (exact for
integers and maxima)."""
import numpy as np
import pytest

from helpers import canaries, compiled, host, out_dev, run, to_dev

pytestmark = pytest.mark.gpu

# f32 (4 per vector): the narrow body up to 32, the 4-vector cache, the
# lengths the 8-vector variants take, streamed lengths held in registers by
# nests of several passes, streamed rows.
F32 = [1, 3, 31, 33, 35, 63, 255, 1021, 1022, 2047, 4095, 4097, 4098, 8190, 8191, 8193, 8194, 16379, 16382, 16387, 16390,
       33001, 33002]


def _rows(C):
    return 300 if C > 4000 else 700  # above the split's 255 rows


@pytest.mark.parametrize("C", F32)
def test_ragged_sum_max(gpu, C):
    rng = np.random.default_rng(C)
    x = rng.integers(-8, 9, (_rows(C), C)).astype(np.float32)
    s, m = out_dev((len(x),), gpu), out_dev((len(x),), gpu)
    run(compiled("row_sum_max_dyn"), [to_dev(x, gpu), s, m])
    assert np.array_equal(host(s), x.sum(1, dtype=np.float64).astype(np.float32))  # integers: exact
    assert np.array_equal(host(m), x.max(1))


@pytest.mark.parametrize("name", ["softmax_dyn", "layernorm_dyn"])
@pytest.mark.parametrize("C", F32)
def test_ragged_passes(gpu, name, C):
    """In place as well: each element is written by the lane that read it."""
    rng = np.random.default_rng(C + 1)
    R = _rows(C) if C < 16384 else 260
    x = (rng.standard_normal((R, C)) * 2 + 0.5).astype(np.float32)
    x[0, :] = 1.0                       # a constant row
    x[1, C - 1] = 30.0                  # the largest value in the tail
    x64 = x.astype(np.float64)
    y = out_dev((R, C), gpu)
    d = to_dev(x, gpu)
    if name == "softmax_dyn":
        extra, scalars = [], []
        e = np.exp(x64 - x64.max(1, keepdims=True))
        want = e / e.sum(1, keepdims=True)
        bound = 5e-6 * want  # 2.7e-6 of the exponentials, up to 30 roundings of 6e-8 in a lane and its tree, 3e-7 of the map
    else:
        g, b = (rng.standard_normal(C) + 1).astype(np.float32), rng.standard_normal(C).astype(np.float32)
        extra, scalars = [to_dev(g, gpu), to_dev(b, gpu)], [1.0 / C, 1e-5]
        mean, var = x64.mean(1, keepdims=True), x64.var(1, keepdims=True)
        want = (x64 - mean) / np.sqrt(var + 1e-5) * g + b
        # the mean is off by at most 1e-6 of the row's root mean square, which
        # the normalisation scales by up to 1 / sqrt(eps) on a constant row
        bound = 1e-5 * (np.abs(want) + np.abs(g) + np.abs(b)) + 1e-6 * np.abs(g) * np.sqrt((x64 ** 2).mean(1, keepdims=True)) \
            / np.sqrt(var + 1e-5)
    for out in (y, d):
        run(compiled(name), [d] + extra + [out], scalars=scalars)
        got = host(out)
        assert canaries(got) == 0
        assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("C", [5, 127, 129, 131, 1001, 1004, 2047, 4099, 8189, 8196, 16391, 32772, 32774, 65551])
def test_ragged_narrow_types(gpu, C):
    import torch
    rng = np.random.default_rng(C)
    u = rng.integers(0, 256, (300, C)).astype(np.uint8)
    out = out_dev((300,), gpu)
    run(compiled("row_sum_u8_dyn"), [to_dev(u, gpu), out], scalars=[0.25])
    assert np.array_equal(host(out), u.sum(1, dtype=np.int64).astype(np.float32) * np.float32(0.25))
    x = rng.integers(-8, 9, (300, C)).astype(np.float32)
    xb = to_dev(x, gpu).to(torch.bfloat16)
    s, m = out_dev((300,), gpu), out_dev((300,), gpu)
    run(compiled("row_sum_bf16_dyn"), [xb, s, m])
    assert np.array_equal(host(s), x.sum(1, dtype=np.float64).astype(np.float32))
    assert np.array_equal(host(m), x.max(1))
    y = out_dev((300, C), gpu)
    run(compiled("softmax_bf16_dyn"), [xb, y])
    e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    assert (np.abs(host(y) - want) <= 5e-6 * want).all()


@pytest.mark.parametrize("C", [1021, 8193, 33001])
def test_ragged_special_values(gpu, C):
    """-inf, +inf and NaN in a row's tail, and rows of the type's lowest value."""
    x = np.zeros((300, C), np.float32)
    x[0, C - 1], x[1, C - 1], x[2, C - 1] = -np.inf, np.inf, np.nan
    x[3, :], x[4, :] = -np.inf, np.finfo(np.float32).min
    s, m, y = out_dev((300,), gpu), out_dev((300,), gpu), out_dev((300, C), gpu)
    d = to_dev(x, gpu)
    run(compiled("row_sum_max_dyn"), [d, s, m])
    assert host(m)[0] == 0 and host(m)[1] == np.inf and host(m)[3] == -np.inf and host(m)[4] == np.finfo(np.float32).min
    assert host(s)[0] == -np.inf and host(s)[1] == np.inf and np.isnan(host(s)[2])
    run(compiled("softmax_dyn"), [d, y])
    got = host(y)
    assert got[0, C - 1] == 0 and np.allclose(got[0, :-1], 1 / (C - 1), rtol=5e-6)
    assert np.isnan(got[1, C - 1]) and np.isnan(got[2]).all() and np.isnan(got[3]).all()
    assert np.allclose(got[4:], 1 / C, rtol=5e-6)
