"""Small Euler solves on the band kernel: the sizes that take it, what stays on
the phase kernels or is refused, and results bitwise equal to the phases'."""
import numpy as np
import pytest


@pytest.mark.parametrize("nx,ny,band", [
    (16, 16, True), (128, 128, True), (240, 272, True), (16, 4064, True), (1024, 16, True), (4064, 16, False),
    (256, 256, False), (256, 272, False), (288, 288, True), (7680, 16, False), (384, 384, True), (16384, 16, True)])
def test_line_between_band_and_phases(nx, ny, band):
    from pysweep_amd import kernels
    from pysweep_amd.equations import path as eq_path
    for cu in ("euler.cu", "euler_fp32.cu"):
        assert kernels.band_default(eq_path(cu), 4, 2, 2, nx, ny) is band


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,steps,exact", [(16, 16, 9, True), (48, 32, 7, False), (16, 336, 5, True),
                                               (288, 288, 6, False)])
def test_small_solves_equal_the_phases(device, nx, ny, steps, exact):
    from gpu_helpers import gpu_solve
    from pysweep_amd import device as dev, workloads
    ic = workloads.vortex_state(nx, ny, 4.0, 1.0, -2.0)
    g = [0.0, steps * 0.05 * 10.0 / max(nx, ny), 0.05 * 10.0 / max(nx, ny), 10.0 / nx, 10.0 / ny, 1.4]
    a = gpu_solve("euler", ic, g, 2, 2, 16, exact=exact)
    b = gpu_solve("euler", ic, g, 2, 2, 16, exact=exact, tuning={"phases": True})
    assert isinstance(a._run, dev.BandRun) and isinstance(b._run, dev.SweptRun)
    assert np.array_equal(a.result, b.result)
    h = gpu_solve("euler", ic, g, 2, 2, 16, exact=exact, tuning={"threads": 128})
    assert isinstance(h._run, dev.SweptRun) and np.array_equal(a.result, h.result)


@pytest.mark.gpu
@pytest.mark.parametrize("b", [4, 48])
def test_blocks_the_phases_refuse_are_refused(device, b):
    from gpu_helpers import gpu_solve
    from pysweep_amd import workloads
    with pytest.raises(ValueError):
        gpu_solve("euler", workloads.vortex_state(96, 96, 4.0, 1.0, -2.0), [0.0, 0.1, 0.01, 0.1, 0.1, 1.4], 2, 2, b)
