"""The packed tensor descriptors against the fields of include/tca_rt.h: every
rank, dtype code and extent, and the values a packed write does not take."""
import ctypes

import pytest

from tcacomp_amd import _lib, compiler
from tcacomp_amd.compiler import TensorDesc


@pytest.mark.parametrize("rank", range(0, _lib.TCA_MAX_RANK + 3))
def test_fields_of_every_rank(rank):
    shape = tuple(range(3, 3 + rank))
    arr = compiler._descriptors([TensorDesc(0x7f0012345670, shape, 9), TensorDesc(0, (0, 2 ** 32 - 1), 2)])
    assert len(arr) == 2 and ctypes.sizeof(arr) == 2 * ctypes.sizeof(_lib.tca_tensor)
    assert (arr[0].data, arr[0].rank, arr[0].dtype) == (0x7f0012345670, rank, 9)
    assert list(arr[0].dims) == (list(shape) + [0] * 8)[:8]
    assert (arr[1].data, arr[1].rank, arr[1].dtype) == (None, 2, 2)
    assert list(arr[1].dims)[:2] == [0, 2 ** 32 - 1]


def test_values_a_field_takes_alone():
    arr = compiler._descriptors([TensorDesc(None, (2 ** 32 + 5, 7), 0)])
    assert (arr[0].data, arr[0].rank, list(arr[0].dims)[:2], arr[0].dtype) == (None, 2, [5, 7], 0)
    assert len(compiler._descriptors([])) == 1


def test_torch_tensors():
    import torch
    t = torch.zeros(3, 5, dtype=torch.bfloat16)
    arr = compiler._descriptors([t, torch.zeros((), dtype=torch.float32)])
    assert (arr[0].data, arr[0].rank, list(arr[0].dims)[:3], arr[0].dtype) == (t.data_ptr(), 2, [3, 5, 0], 2)
    assert (arr[1].rank, arr[1].dtype) == (0, 0)
    with pytest.raises(ValueError):
        compiler._descriptors([t.t()])
    with pytest.raises(KeyError):
        compiler._descriptors([torch.zeros(2, dtype=torch.float64)])


@pytest.mark.gpu
def test_launch_follows_the_current_stream(gpu):
    import torch
    assert compiler._current_stream() == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert compiler._current_stream() == s.cuda_stream
    assert compiler._current_stream() == torch.cuda.current_stream().cuda_stream
