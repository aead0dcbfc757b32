"""Engines driven from several threads at once: each engine's kernel times are its
own.  Two engines (one of them in two parts) step in threads of their own while
small engines are made, stepped and closed beside them; every engine counts one
flight launch per interval, for no longer than its steps took, and its results are
those of a run by itself."""
import threading
import time

import numpy as np
import pytest

import ekmc

pytestmark = pytest.mark.gpu

INTERVALS = 400
# (electrons per condition, E/N, B/N)
LONG = {"one": [(150000, 120.0, 300.0)], "parts": [(250000, 90.0, 300.0), (250000, 200.0, 300.0)]}
SMALL = [(2000, 150.0, 200.0)]


def _engine(batch, precision):
    mix, conds, num = ekmc.workload("cfg3_o2like_batched", conditions=[0] * len(batch))
    for cond, (n, en, bn) in zip(conds, batch):
        cond.n_electrons, cond.reduced_elec_field, cond.reduced_mag_field = n, en, bn
        cond.elec_field_angle = 90.0
    num.precision = precision
    num.seed = 12
    num.n_integration_points = 1e15
    eng = ekmc.Engine(mix, conds, num)
    eng.initialize()
    return eng


def _step(eng, intervals, out):
    t0 = time.perf_counter()
    eng.step(intervals)
    wall = 1e3 * (time.perf_counter() - t0)
    launches, ms = eng.kernel_stats()["advance"]
    st = [eng.status(c) for c in range(len(eng.conditions))]
    out.update(wall=wall, launches=launches, ms=ms,
               state=np.array([[s.time, s.real_collisions, s.null_collisions, s.last_mean_energy] for s in st]))


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
def test_kernel_times_belong_to_their_engine(precision):
    alone, beside = {}, {}
    for name, batch in LONG.items():
        eng = _engine(batch, precision)
        _step(eng, INTERVALS, alone.setdefault(name, {}))
        eng.close()
    engines = {name: _engine(batch, precision) for name, batch in LONG.items()}
    threads = [threading.Thread(target=_step, args=(eng, INTERVALS, beside.setdefault(name, {})))
               for name, eng in engines.items()]
    for t in threads:
        t.start()
    small = []
    while any(t.is_alive() for t in threads) or not small:
        eng = _engine(SMALL, precision)
        small.append({})
        _step(eng, 3, small[-1])
        eng.close()
    for t in threads:
        t.join()
    for eng in engines.values():
        eng.close()
    for name in LONG:
        assert alone[name]["state"].tobytes() == beside[name]["state"].tobytes()
        for run in (alone[name], beside[name]):
            assert run["launches"] == INTERVALS and 0 < run["ms"] < run["wall"]
    for run in small:
        assert run["launches"] == 3 and 0 < run["ms"] < run["wall"]
        assert run["state"].tobytes() == small[0]["state"].tobytes()
