"""Launch shapes of the band kernels: segments asked for beyond the grid."""
import pytest


@pytest.mark.parametrize("cu,nv,ops,its", [("euler.cu", 4, 2, 2), ("heat.cu", 1, 1, 1)])
@pytest.mark.parametrize("rows", [64, 1000, 10 ** 9, 2 ** 31 - 1])
def test_one_segment_however_long(cu, nv, ops, its, rows):
    """A segment longer than the grid is one segment: every field fits the
    plan's 32-bit members."""
    import ctypes
    from pysweep_amd import kernels
    from pysweep_amd.equations import path as eq_path
    spec = kernels.band_spec(eq_path(cu), nv, ops, its)
    for nx in (1, 6, 7, 64):
        got, shape = kernels.band_launch(spec, nx, 64, rows)
        assert got == rows
        for k, v in shape.items():
            assert ctypes.c_int(v).value == v, (k, v)
        assert shape["rows"] >= nx
