"""The Euler standard kernel's 15-row tiles: where they are taken, and results
bitwise equal to 16-row tiles' and to other tiles' on ragged grids."""
import numpy as np
import pytest


@pytest.mark.parametrize("nx,ny,rows", [(16, 16, 15), (240, 256, 15), (256, 256, 16), (352, 352, 16), (384, 384, 15),
                                        (1000, 1500, 15), (2048, 2048, 15), (14, 64, 8), (64, 8, 32)])
def test_rows_of_a_standard_tile(nx, ny, rows):
    from pysweep_amd import kernels
    from pysweep_amd.equations import path as eq_path
    for name, real in (("euler.cu", "double"), ("euler_fp32.cu", "float")):
        spec = kernels.standard_spec(eq_path(name), 4, 2, 2, nx, ny, real=real)
        assert spec.bx == rows and spec.threads == 512
        assert kernels.standard_spec(eq_path(name), 4, 2, 2, nx, ny, real=real, multi=True).bx != 15
    assert kernels.standard_spec(eq_path("heat.cu"), 1, 1, 1, nx, ny).bx != 15


@pytest.mark.gpu
@pytest.mark.parametrize("real", ["double", "float"])
@pytest.mark.parametrize("nx,ny", [(16, 16), (17, 33), (29, 18), (31, 47), (45, 16), (61, 130)])
def test_fifteen_rows_equal_other_tiles(device, nx, ny, real):
    from pysweep_amd import device as dev, plugins, workloads
    from pysweep_amd.equations import path as eq_path
    g = [0.0, 1.0, 0.05 * 10.0 / max(nx, ny), 10.0 / nx, 10.0 / ny, 1.4]
    ic = workloads.vortex_state(nx, ny, 4.0, 1.0, -2.0)
    cpu = plugins.load_cpu_module(eq_path("euler.py"))
    got = []
    for bx, by in ((None, None), (16, 16), (8, 8)):
        r = dev.StandardRun(eq_path("euler.cu" if real == "double" else "euler_fp32.cu"), 4, 2, 2, nx, ny, real=real,
                            bx=bx, by=by)
        r.set_globals(cpu, g)
        r.upload_ic(ic)
        r.run(1, 12)
        got.append((r.spec.bx, r.level(12), r.level(11)))
        r.close()
    assert got[0][0] == 15
    for _, a, b in got[1:]:
        assert np.array_equal(got[0][1], a) and np.array_equal(got[0][2], b)
