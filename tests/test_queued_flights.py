"""Flight launches with more chunks than resident waves (chunks taken from the queue,
records stored as whole lines in the mixed form), in one part and in two.

One part: the conditions of a batch below 400,000 electrons fly from the queue, one of
them alone has a wave for every chunk and stores each record by its own lane; its
electrons are the same bytes.  Two parts: each has more chunks than waves, so
both queues, their reset, the stealing between XCDs and the smaller grid are in use;
everything equals the run in one part (EKMC_KERNEL_TIMING=all).  An error in one part
while the other's interval is in flight leaves the other part's conditions whole."""
import numpy as np
import pytest

import ekmc
from helpers import condition, mixture

pytestmark = pytest.mark.gpu

GOLDEN = 0x9E3779B97F4A7C15  # condition c draws with the key seed ^ c GOLDEN
SEED = 2024


def _condition_seed(c):
    """The seed with which condition c alone draws what it draws in a batch."""
    return SEED ^ (c * GOLDEN & 0xFFFFFFFFFFFFFFFF)


def _engine(batch, precision, seed, chunk=64):
    mix, conds, num = ekmc.workload("cfg3_o2like_batched", conditions=[0] * len(batch))
    for cond, (n, en, bn) in zip(conds, batch):
        cond.n_electrons, cond.reduced_elec_field, cond.reduced_mag_field = n, en, bn
        cond.elec_field_angle = 90.0
    num.precision, num.seed, num.work_chunk = precision, seed, chunk
    num.n_energy_cells = 200
    num.n_integration_points = 1e15
    eng = ekmc.Engine(mix, conds, num)
    eng.initialize()
    return eng


def _state(eng, c):
    st = eng.status(c)
    return [*eng.electrons(c), np.array([st.time, st.trial_collision_frequency, st.max_elec_energy]),
            np.array([st.real_collisions, st.null_collisions, st.n_sampling_points])]


def _same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert np.asarray(x).tobytes() == np.asarray(y).tobytes()


# (electrons, E/N, B/N): 4600 chunks of 64 in all, at most 1500 of one condition; from
# attachment (holes and clones) to strong ionization (newborns and removals)
ONE_PART = [(95999, 4.0, 300.0), (65537, 150.0, 700.0), (40001, 600.0, 200.0), (101, 300.0, 400.0),
            (63, 600.0, 400.0), (92161, 350.0, 100.0)]


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("first", range(len(ONE_PART)))
def test_queued_flights_equal_flights_of_a_wave_per_chunk(first, precision):
    # the condition compared comes first in its batch (a clone's variates are keyed
    # by its place in the pool)
    batch = ONE_PART[first:] + ONE_PART[:first]
    assert 3072 < sum(-(-n // 64) for n, *_ in batch) and sum(n for n, *_ in batch) < 400000
    eng = _engine(batch, precision, SEED)
    for turns in (1, 13):
        eng.step(turns)
    queued = _state(eng, 0)
    eng.close()
    eng = _engine(batch[:1], precision, SEED)
    eng.step(14)
    _same(queued, _state(eng, 0))
    eng.close()


TWO_PARTS = {
    "crossed": [(250007, 120.0, 300.0), (20011, 500.0, 200.0), (249989, 30.0, 700.0), (65, 300.0, 100.0)],
    # one part without and one with a magnetic field, flown by the kernel for both
    "sorted": [(250007, 120.0, 0.0), (20011, 400.0, 0.0), (249989, 30.0, 700.0), (65, 300.0, 100.0)],
}


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("name", list(TWO_PARTS))
def test_two_queued_parts_equal_one(monkeypatch, name, precision):
    batch = TWO_PARTS[name]

    def run():
        eng = _engine(batch, precision, SEED)
        for turns in (1, 2, 9):
            eng.step(turns)
        out = [x for c in range(len(batch)) for x in _state(eng, c)]
        for c in range(len(batch)):
            s = eng.series(c)
            out += [s[k] for k in sorted(s)]
        eng.close()
        return out

    two = run()
    monkeypatch.setenv("EKMC_KERNEL_TIMING", "all")
    _same(two, run())


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("failing", [0, 1])
def test_an_error_in_one_part_leaves_the_other_whole(failing, precision):
    top = 60.0  # the tables end here; the condition of the high field passes it
    mix = mixture([
        dict(elastic=True, energy=np.array([0.0, top]), sigma=np.array([1e-19, 1e-19]), mass_amu=40.0),
        dict(threshold=10.0, energy=np.array([10.0, 10.5, top]), sigma=np.array([0.0, 1e-20, 1e-20]), mass_amu=40.0)])
    fields = [(800.0 if c == failing else 5.0) for c in range(2)]

    def engine(conds, seed):
        num = ekmc.numerics_default()
        num.precision, num.seed = precision, seed
        num.initial_elec_temp_over_gas_temp = 11604.5 / 300.0
        num.n_integration_points = 1e15
        eng = ekmc.Engine(mix, [condition(en=fields[c], angle=90.0, bn=100.0, n_e=250000) for c in conds], num)
        eng.initialize()
        return eng

    eng = engine([0, 1], SEED)
    with pytest.raises(ekmc.EngineError) as err:
        eng.step(300)
    assert err.value.status == 3 and "until 60.0" in str(err.value)  # EKMC_ERR_ENERGY_OUT_OF_TABLE
    other = 1 - failing
    whole, intervals = _state(eng, other), eng.status(other).n_sampling_points - 1
    # an interval ahead at most
    assert intervals - (eng.status(failing).n_sampling_points - 1) in (0, 1)
    eng.close()
    eng = engine([other], _condition_seed(other))
    eng.step(intervals)
    _same(whole, _state(eng, 0))
    eng.close()
