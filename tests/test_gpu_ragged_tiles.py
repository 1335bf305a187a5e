"""Maps with a transposed operand whose extents are no multiples of 4: whole
unaligned vectors up to the last, partial one of each row and column, on both
tile sizes. Every extent modulo 4, on either side of a tile's edge, against
numpy (the same float32 operations in the same order: exact)."""
import numpy as np
import pytest

from helpers import canaries, compiled, host, out_dev, run, to_dev
from tcacomp_amd.compiler import compile_program
from tileprog import three_transposed

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 2), (5, 7), (127, 129), (129, 127), (130, 126), (128, 131), (131, 128), (261, 1), (1, 261),
         (257, 514), (1001, 1002), (1003, 999)]


@pytest.fixture(scope="module")
def three():
    return compile_program(three_transposed())


def _check(prog, arrays, want, gpu):
    """Writes exactly want.size elements: the buffer goes on past the output."""
    import torch
    buf = out_dev((want.size + 64,), gpu, torch.float32)
    run(prog, [to_dev(a, gpu) for a in arrays] + [buf[:want.size].view(want.shape)])
    got = host(buf)
    assert np.array_equal(got[:want.size].reshape(want.shape), want)
    assert canaries(got[want.size:]) == 64


# integers, so that a contracted multiply-add rounds nothing
def _ints(rng, *shapes):
    return [rng.integers(-64, 65, s).astype(np.float32) for s in shapes]


@pytest.mark.parametrize("R,C", SIZES)
def test_ragged_transposed_operand(gpu, R, C):
    x, z, g, b = _ints(np.random.default_rng(R * 1000 + C), (R, C), (C, R), (C,), (R,))
    _check(compiled("ew_bias_tr"), [x, z, g, b], x * g + b[:, None] + z.T, gpu)


@pytest.mark.parametrize("R,C", SIZES)
def test_ragged_three_transposed_operands(gpu, three, R, C):
    zs = _ints(np.random.default_rng(R * 1000 + C + 1), *[(C, R)] * 3)
    _check(three, zs, zs[0].T + zs[1].T + zs[2].T, gpu)
