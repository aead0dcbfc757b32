"""The parts of a batch run beside each other whatever streams a program made and freed
before: HIP places a new stream on the hardware queue that has the fewest, so a program
that frees streams of one queue has an engine's next two both put there, where they
run in turn.  The time of a step stays what it is in a fresh program (in turn it was
1.8 times that; a third of it more is allowed for noise), or, where no second stream
beside the first can be had, that of a batch in one part; the results are the same bytes."""
import ctypes
import time

import numpy as np
import pytest

import ekmc

pytestmark = pytest.mark.gpu


def _run(precision):
    mix, conds, num = ekmc.workload("cfg3_o2like_batched", conditions=[0] * 8)
    for k, cond in enumerate(conds):
        cond.n_electrons, cond.elec_field_angle = 100000, 90.0
        cond.reduced_elec_field, cond.reduced_mag_field = 50.0 + 40.0 * k, 100.0 * (1 + k % 3)
    num.precision, num.seed = precision, 4
    num.n_integration_points = 1e15
    eng = ekmc.Engine(mix, conds, num)
    eng.initialize()
    eng.step(32)
    best = 1e9
    for _ in range(8):
        t0 = time.perf_counter()
        eng.step(32)
        best = min(best, time.perf_counter() - t0)
    out = [a for c in (0, 7) for a in eng.electrons(c)]
    eng.close()
    return best, out


@pytest.fixture(scope="module")
def fresh():
    return {p: _run(p) for p in (ekmc.FP64, ekmc.MIXED)}


# streams made, and which of them are freed before the engine is made
PATTERNS = {"held": (8, []), "free2": (8, [1]), "free5": (8, [4]), "free2and6": (8, [1, 5]),
            "queue0": (48, range(0, 48, 4)), "queue1": (48, range(1, 48, 4)),
            "queue2": (48, range(2, 48, 4)), "queue3": (48, range(3, 48, 4))}


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("name", list(PATTERNS))
def test_parts_run_beside_each_other(fresh, name, precision):
    hip = ctypes.CDLL("libamdhip64.so")
    made, freed = PATTERNS[name]
    streams = []
    for _ in range(made):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # non-blocking
        streams.append(s)
    try:
        for k in freed:
            assert hip.hipStreamDestroy(streams[k]) == 0
        best, out = _run(precision)
    finally:
        for k, s in enumerate(streams):
            if k not in freed:
                assert hip.hipStreamDestroy(s) == 0
    for a, b in zip(out, fresh[precision][1]):
        assert np.asarray(a).tobytes() == np.asarray(b).tobytes()
    print("%s: %.2f ms, fresh %.2f ms" % (name, 1e3 * best, 1e3 * fresh[precision][0]))
    assert best < 4.0 / 3.0 * fresh[precision][0]
