"""Chains of the Euler band sweep (a workgroup's wavefronts handing their
segments' first rows to the segment before) against the standard kernel,
bitwise, where the split of a chain's rows can go wrong."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _runs(nx, ny, real):
    from pysweep_amd import device, plugins, workloads
    from pysweep_amd.equations import path as eq_path
    dx = 10.0 / nx
    g = [0.0, 1.0, 0.05 * dx, dx, 10.0 / ny, 1.4]
    cpu = plugins.load_cpu_module(eq_path("euler.py"))
    cu = eq_path("euler.cu" if real == "double" else "euler_fp32.cu")
    ic = workloads.vortex_state(nx, ny, 4.0, 1.0, -2.0)
    out = []
    for cls in (device.StandardRun, device.BandRun):
        r = cls(cu, 4, 2, 2, nx, ny, real=real)
        r.set_globals(cpu, g)
        r.upload_ic(ic)
        out.append(r)
    return out


@pytest.mark.parametrize("real", ["double", "float"])
@pytest.mark.parametrize("nx,ny,rows", [
    (64, 60, 26),   # chains of 26, 26 and 12 rows: 3, 3 and 1 wavefronts
    (37, 57, 28),   # 4 wavefronts of 8, 8, 7, 5 rows, then 9 rows on one
    (29, 120, 28),  # a last chain of one row
    (14, 64, 14),   # two wavefronts, the whole (periodic) grid in one chain
    (6, 9, 40),     # a chain longer than the grid: one wavefront
    (131, 70, 50), (200, 56, 200)])
def test_chains_equal_the_standard_kernel(device, nx, ny, rows, real):
    """7 stages: whole launches and a last one of a single stage."""
    from pysweep_amd import hip
    st, band = _runs(nx, ny, real)
    st.run(1, 8)
    want = [st.level(7), st.level(8)]
    band.plan.rows, band.plan.chain = rows, 4
    hip.band_run(band.plan, 1, 7)
    assert np.array_equal(band.level(8), want[1])
    band.upload_ic(st_ic(st))
    band.plan.store_all = 1  # every level written: level 7 is a launch's first
    hip.band_run(band.plan, 1, 6)
    assert np.array_equal(band.level(6), level_after(st, 6)) and np.array_equal(band.level(7), want[0])
    assert not band.range_fault()
    st.close()
    band.close()


def st_ic(st):
    from pysweep_amd import workloads
    return workloads.vortex_state(st.nx, st.ny, 4.0, 1.0, -2.0)


def level_after(st, A):
    st.upload_ic(st_ic(st))
    st.run(1, A)
    return st.level(A)


def test_only_chains_of_four_are_taken(device):
    from pysweep_amd import hip
    st, band = _runs(32, 64, "double")
    band.plan.chain = 2
    with pytest.raises(hip.HipError, match="chain"):
        hip.band_run(band.plan, 1, 2)
    st.close()
    band.close()
