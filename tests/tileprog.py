"""Programs of tests/test_gpu_ragged_tiles.py that the product does not
register: built beside its own, so a GPU run never compiles."""
from tcacomp_amd.pkg import TF32, At, NewBuilder


def three_transposed():
    """y = z0^T + z1^T + z2^T: three transposed operands take 64x64 tiles."""
    b = NewBuilder("ew_tr3_ragged")
    R, C = b.Dim("R", 0), b.Dim("C", 0)
    zs = [b.Tensor("z%d" % i, TF32, C, R) for i in range(3)]
    y = b.Tensor("y", TF32, R, C)
    b.Stmt().Iter(R, C).Map([At(z, C, R) for z in zs], lambda p, q, r: b.Add(b.Add(p, q), r)).As(R, C).Store(y, R, C)
    return b.Build()


def all_builds():
    """(name, program factory, emit flags), as tests/randprog.py's."""
    return [("ew_tr3_ragged", three_transposed, 0)]
