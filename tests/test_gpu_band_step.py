"""Rounds without a BandMulti launch, and counters that move once per run of
rounds: batched results against plain solves, bitwise."""
from types import SimpleNamespace

import numpy as np
import pytest


@pytest.mark.parametrize("h,cs,graph_rounds,want", [
    (2, [1, 5], 0, 2), (2, [1, 2], 0, 0), (2, [], 0, 0), (12, [1, 13, 25], 0, 12), (12, [1, 7], 0, 0),
    (12, [1], 8, 0), (12, [1], 24, 12), (2, [3], 8, 2)])
def test_band_step(h, cs, graph_rounds, want):
    from pysweep_amd.batch import _ClassTable
    table = SimpleNamespace(cls=SimpleNamespace(band_h=h))
    assert _ClassTable._band_step(table, [SimpleNamespace(c=c) for c in cs], graph_rounds) == want


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(), dict(max_rounds_ahead=5), dict(use_graphs=True, graph_rounds=5),
                                dict(use_graphs=True, graph_rounds=12), dict(use_graphs=True, graph_rounds=24),
                                dict(policy="short_first", capacity=20000, max_rounds_ahead=7)])
def test_rounds_equal_plain_solves(device, kw):
    from gpu_helpers import euler_case
    from pysweep_amd import baseline
    from pysweep_amd.batch import Engine, Problem
    probs = []
    for n, steps in ((64, 9), (96, 30), (128, 17)):
        ic, g, _ = euler_case(n, steps)
        for m in ("band", "swept", "standard"):
            probs.append(Problem("euler", ic, g, 2, method=m))
    for i, (n, steps) in enumerate(((64, 7), (96, 12), (128, 50))):
        ic = np.random.default_rng(i).random((1, n, n))
        dt = 0.1 / n / n
        for m in ("band", "swept"):
            probs.append(Problem("heat", ic, [0.0, steps * dt, dt, 1.0 / n, 1.0 / n, 1.0, True], 1, method=m))
    eng = Engine(tuner=None, **kw)
    tickets = [eng.submit(p, arrival=0.0 if i % 3 else 0.002 * i) for i, p in enumerate(probs)]
    eng.run()
    for t in tickets:
        assert np.array_equal(t.result, baseline.solve_plain(t.problem)), (t.problem.plugin, t.problem.method)
