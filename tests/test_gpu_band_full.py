"""Whole launches of the point-update band method (BandFull) against the
standard kernel, bitwise, where rows, columns and parities can go wrong."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("its,scheme", [(1, True), (2, False), (1, False)])  # (1, False): the stage's parity varies
@pytest.mark.parametrize("real", ["double", "float"])
@pytest.mark.parametrize("nx,ny,rows", [
    (1, 2, 3), (3, 7, 1), (5, 104, 2),  # grids smaller than the halo, odd ny
    (29, 105, 4), (40, 112, 7), (64, 209, 16),  # a column past a band, the last segment short
    (31, 313, 31), (33, 96, 40)])
def test_whole_launches_equal_the_standard_kernel(device, nx, ny, rows, real, its, scheme):
    """Two whole launches and a last one of a single step."""
    from pysweep_amd import device as dev, hip, plugins
    from pysweep_amd.equations import path as eq_path
    dx = 1.0 / nx
    g = [0.0, 1.0, 0.1 * dx * dx, dx, 1.0 / ny, 1.0, scheme]
    ic = np.random.default_rng(nx * ny).random((1, nx, ny))
    cpu = plugins.load_cpu_module(eq_path("heat.py"))
    cu = eq_path("heat.cu" if real == "double" else "heat_fp32.cu")
    out = []
    for cls in (dev.StandardRun, dev.BandRun):
        r = cls(cu, 1, 1, its, nx, ny, real=real)
        r.set_globals(cpu, g)
        r.upload_ic(ic)
        out.append(r)
    st, band = out
    assert band.plan.full and band.plan.full_rows >= 1
    band.plan.rows = band.plan.full_rows = rows
    stages = 2 * band.spec.levels + its
    last = its - 1 + stages
    st.run(1, 1 + stages)
    hip.band_run(band.plan, its - 1, stages)
    assert np.array_equal(band.level(last), st.level(last))
    st.close()
    band.close()


@pytest.mark.parametrize("real", ["double", "float"])
def test_full_rows_cover_every_grid(real):
    from pysweep_amd import kernels
    from pysweep_amd.equations import path as eq_path
    spec = kernels.band_spec(eq_path("heat.cu" if real == "double" else "heat_fp32.cu"), 1, 1, 1, real=real)
    for nx, ny in ((1, 2), (64, 64), (100000, 100), (64, 200000), (16384, 65536)):
        assert kernels.band_full_rows(spec, nx, ny) >= 1
