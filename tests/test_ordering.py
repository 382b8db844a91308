"""Setting a run up is complete on return: constants, fault flags and initial
levels are in device memory before another context, stream or thread may be
told that they are.  Host logic, checked on a recorded sequence of calls."""
import types

import numpy as np
import pytest


@pytest.fixture
def calls(monkeypatch):
    from pysweep_amd import hip
    log = []
    for name in ("write_bytes", "htod_bytes", "htod", "memset_async", "dtod_async", "synchronize"):
        monkeypatch.setattr(hip, name, lambda *a, _n=name: log.append(_n))
    monkeypatch.setattr(hip, "htod_async", lambda *a: log.append("htod_async"), raising=False)
    return log


def _run(its):
    from pysweep_amd import device
    run = object.__new__(device._Run)
    run.nv, run.its, run.nx, run.ny, run.T = 1, its, 4, 4, its + 1
    run.dtype, run.level_bytes = np.float64, 4 * 4 * 8
    mod = types.SimpleNamespace(get_global=lambda name: (4096, 8), const_owner=None)
    run.modules = [mod, mod]
    return run


def _plugin():
    from pysweep_amd import plugins

    def set_globals(a, b, source_mod=None):
        for name, v in (("A", a), ("B", b)):
            ptr, _ = source_mod.get_global(name)
            plugins.driver.memcpy_htod(ptr, np.float64(v))
    return types.SimpleNamespace(set_globals=set_globals)


def test_constants_are_written_on_return(calls):
    from pysweep_amd import plugins
    run = _run(1)
    run.set_globals(_plugin(), [1.0, 2.0])
    assert calls.count("write_bytes") == 4 and calls[-1] == "synchronize"
    assert calls.count("synchronize") == 1
    del calls[:]
    # through a handle of one's own every copy to the device has waited
    _plugin().set_globals(1.0, 2.0, source_mod=run.facade())
    assert calls.count("write_bytes") == 4 and calls[-1] == "synchronize"
    ptr, _ = plugins.SourceModuleFacade(run.modules).get_global("A")
    del calls[:]
    plugins.driver.memcpy_htod(ptr, np.float64(3.0))
    assert calls[-1] == "synchronize"


def test_cleared_fault_flags_are_cleared_on_return(calls):
    run = _run(2)
    run.range_fault(clear=True)
    assert calls[-1] == "synchronize"
    assert "memset_async" in calls or "htod" in calls


@pytest.mark.parametrize("its", [1, 2, 3])
def test_initial_levels_are_uploaded_on_return(calls, its):
    run = _run(its)
    run.ring = types.SimpleNamespace(ptr=4096, upload=lambda *a: calls.extend(["htod_async", "synchronize"]))
    run.upload_ic(np.zeros((1, 4, 4)))
    assert calls[-1] == "synchronize"
    assert calls.count("dtod_async") == its - 1
