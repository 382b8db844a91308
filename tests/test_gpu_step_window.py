"""Windows of the swept phases' per-cell step (turning over by storing cells
twice, or by a copy where the window is short) and the tiles' addresses at the
grid's edge, bitwise against the standard kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _runs(name, nx, ny, b, its, **kw):
    from pysweep_amd import device, plugins, workloads
    from pysweep_amd.equations import path as eq_path
    real = "float" if name.endswith("fp32") else "double"
    if name.startswith("heat"):
        dx, nv, ops = 1.0 / nx, 1, 1
        g = [0.0, 1.0, 0.1 * dx * dx, dx, 1.0 / ny, 1.0, its == 1]
        ic = np.random.default_rng(nx + ny).random((1, nx, ny))
    else:
        dx, nv, ops = 10.0 / nx, 4, 2
        g = [0.0, 1.0, 0.05 * dx, dx, 10.0 / ny, 1.4]
        ic = workloads.vortex_state(nx, ny, 4.0, 1.0, -2.0)
    cpu = plugins.load_cpu_module(eq_path(name.split("_")[0] + ".py"))
    cu = eq_path(name + ".cu")
    out = [device.StandardRun(cu, nv, ops, its, nx, ny, real=real),
           device.SweptRun(cu, nv, ops, its, nx, ny, b, real=real, **kw)]
    for r in out:
        r.set_globals(cpu, g)
        r.upload_ic(ic)
    return ops, out


@pytest.mark.parametrize("name,its,b,slots", [
    ("heat", 1, 8, 2), ("heat", 1, 8, 3), ("heat", 1, 8, 4), ("heat", 1, 8, 7),  # copy, twice (C = 2, 3), full
    ("heat", 1, 32, None), ("heat", 2, 16, 3), ("heat", 2, 16, 4), ("heat", 2, 16, 5), ("heat", 2, 16, 6),
    ("heat_fp32", 1, 16, None), ("euler", 2, 16, 3), ("euler", 2, 16, 4), ("euler", 2, 16, None),
    ("euler_fp32", 2, 16, None), ("euler", 2, 24, None)])
def test_per_cell_windows_equal_the_standard_kernel(device, name, its, b, slots):
    """2 x 3 tiles, every one of them at an edge of the grid or beside one."""
    from pysweep_amd import schedule
    ops, (st, sw) = _runs(name, 2 * b, 3 * b, b, its, slots=slots, generic=True)
    P = b // (2 * ops) - 1
    A = sw.run(schedule.swept_times(max(3 * P // its, 2), b, ops, its, exact=True))
    st.run(1, 1 + A - (its - 1))
    assert np.array_equal(sw.level(A), st.level(A))
    st.close()
    sw.close()


@pytest.mark.parametrize("name,its,b,nx,ny", [("heat", 1, 32, 32, 96), ("heat", 2, 16, 160, 16), ("euler", 2, 16, 16, 64),
                                              ("euler", 2, 8, 80, 72)])
def test_level_update_tiles_at_the_edge(device, name, its, b, nx, ny):
    """One tile across the grid (each its own neighbour), and inner tiles."""
    from pysweep_amd import schedule
    ops, (st, sw) = _runs(name, nx, ny, b, its)
    P = b // (2 * ops) - 1
    A = sw.run(schedule.swept_times(max(3 * P // its, 2), b, ops, its, exact=True))
    st.run(1, 1 + A - (its - 1))
    assert np.array_equal(sw.level(A), st.level(A))
    st.close()
    sw.close()
