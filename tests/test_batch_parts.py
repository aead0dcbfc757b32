"""A batch large enough to run in two parts gives, bit for bit, what it gives in
one (with every kernel timed, EKMC_KERNEL_TIMING=all, an engine runs in one part):
whole jobs whose conditions end at different times, intervals taken in turns of
several lengths, and field cases and sizes on both sides of the cut."""
import numpy as np
import pytest

import ekmc

pytestmark = pytest.mark.gpu

# (electrons, E/N, angle, frequency, B/N) per condition
BATCHES = {
    "cut_after_first": [(390001, 120.0, 90.0, 0.0, 300.0), (5003, 60.0, 180.0, 0.0, 0.0), (10007, 250.0, 90.0, 0.0, 700.0)],
    "cut_before_last": [(101, 100.0, 180.0, 0.0, 0.0), (20000, 200.0, 180.0, 5e7, 0.0), (400000, 150.0, 180.0, 0.0, 0.0)],
    "middle": [(100000, 40.0 + 30.0 * k, 90.0, 0.0, 100.0 * (k % 3)) for k in range(6)],
    "below": [(199999, 90.0, 90.0, 0.0, 200.0), (200000, 150.0, 90.0, 0.0, 200.0)],
}


def _run(batch, precision, form):
    mix, conds, num = ekmc.workload("cfg3_o2like_batched", conditions=[0] * len(batch))
    for cond, (n, en, angle, freq, bn) in zip(conds, batch):
        cond.n_electrons, cond.reduced_elec_field, cond.elec_field_angle = n, en, angle
        cond.excitation_frequency, cond.reduced_mag_field = freq, bn
    num.precision = precision
    num.seed = 91
    num.n_energy_cells = 300
    num.n_integration_phases = 8
    num.n_integration_points = 90 if form == "solve" else 1e15
    eng = ekmc.Engine(mix, conds, num)
    out = []
    if form == "solve":
        eng.solve()
        for c in range(len(conds)):
            out += [np.array(a) for a in eng.eedf(c)] + [np.array(a) for a in eng.process_data(c)]
    else:
        eng.initialize()
        for turns in (1, 2, 37, 1):
            eng.step(turns)
            st = eng.status(len(conds) - 1)
            out.append(np.array([st.time, st.real_collisions, st.null_collisions]))
    for c in range(len(conds)):
        out += [np.array(a) for a in eng.electrons(c)]
        s = eng.series(c)
        out += [s[k] for k in sorted(s)]
    launches, ms = eng.kernel_stats()["advance"]
    out.append(np.array([launches]))
    assert ms > 0
    eng.close()
    return out


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("form", ["step", "solve"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_two_parts_equal_one(monkeypatch, name, form, precision):
    two = _run(BATCHES[name], precision, form)
    monkeypatch.setenv("EKMC_KERNEL_TIMING", "all")
    one = _run(BATCHES[name], precision, form)
    assert len(one) == len(two)
    for a, b in zip(one, two):
        assert a.tobytes() == b.tobytes()
