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


@pytest.mark.parametrize("ny,real,wide", [
    (64, "double", False), (2 ** 29, "double", False), (2 ** 29 + 1, "double", True),
    (2 ** 30, "float", False), (2 ** 30 + 8, "float", True)])
def test_rows_of_more_than_32_bits_of_bytes_take_64_bit_offsets(ny, real, wide):
    from pysweep_amd import kernels
    from pysweep_amd.equations import path as eq_path
    size = 8 if real == "double" else 4
    assert ((ny - 1) * size >= 2 ** 32) is wide  # the last column's offset
    for cu, sweep in (("euler.cu", True), ("heat.cu", False)):
        got = kernels.band_defines(eq_path(cu), ny, real, ("EU_EXACT_DIVISION",))
        assert got == ("EU_EXACT_DIVISION",) + (("PS_BAND_WIDE",) if wide and sweep else ())


@pytest.mark.gpu
@pytest.mark.parametrize("cu,real", [("euler.cu", "double"), ("euler_fp32.cu", "float")])
def test_64_bit_offsets_give_the_same_bits(device, cu, real):
    """The form of very long rows, on a grid that the other takes too."""
    import numpy as np
    from pysweep_amd import device as dev, hip, plugins, workloads
    from pysweep_amd.equations import path as eq_path
    cpu = plugins.load_cpu_module(eq_path("euler.py"))
    out = []
    for defines in ((), ("PS_BAND_WIDE",)):
        run = dev.BandRun(eq_path(cu), 4, 2, 2, 66, 131, real=real, defines=defines)
        run.set_globals(cpu, [0.0, 1.0, 0.004, 10 / 66, 10 / 131, 1.4])
        run.upload_ic(workloads.vortex_state(66, 131, 4.0, 1.0, -2.0))
        hip.band_run(run.plan, 1, 7)
        out.append(run.level(8))
        run.close()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])
