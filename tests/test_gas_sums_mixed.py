"""The thermal channel choice of the mixed form against the FP64 oracle with identical
variates, for gas counts around the batches of four gases whose sums are loaded
together and with a gas that is absent.

The two choose alike but where FP32 rounding moves a variate past a boundary: 30
boundaries at most, each known to some 16 units of 2^-24, is 3e-5 of the events, and a
table row that the rounding of energy / step flips (2e-3 of them) shifts a boundary by
1 % at most, 2e-5 more.  That is one event of 20000; the bound is 40, far below what a
wrong index or the sum of another gas moves."""
import numpy as np
import pytest

import ekmc
import oracle_py as O
from helpers import condition, speeds, unit_vectors
from test_gas_sums import _gases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_gas,absent", [(1, -1), (2, 0), (3, 2), (4, -1), (5, 4), (5, 1), (8, 3), (9, 8), (9, -1)])
def test_mixed_thermal_choice_follows_the_oracle(n_gas, absent):
    mix = _gases(n_gas, absent)
    cond = condition(tg=2000.0, n_e=64)
    num = ekmc.numerics_default()
    num.gas_temperature_effect = ekmc.GASTEMP["true"]
    num.n_interp_points = 2000
    num.precision = ekmc.MIXED
    eng = ekmc.Engine(mix, [cond], num)
    num.precision = ekmc.FP64
    model = O.Model(mix, cond, num)
    top = 120.0
    _, _, _, mx, _ = model.tables(top)
    rng = np.random.default_rng(7 * n_gas + absent)
    n = 20000
    energy = np.exp(rng.uniform(np.log(0.02), np.log(100.0), n))
    vel = unit_vectors(rng, n) * speeds(energy)[:, None]
    var = rng.uniform(1e-6, 1.0, (n, ekmc.VARIATES_PER_EVENT))
    nue = np.full(n, 1.2 * mx[-1])
    pid, v, e, *_ = eng.op_collide(0, top, vel, energy, nue, var)
    eng.close()
    _, pid_o, v_o, e_o, *_ = model.collide(vel, energy, nue, var)
    same = pid == pid_o
    assert np.count_nonzero(~same) <= 40
    assert np.any(pid < 0) and np.count_nonzero(np.bincount(pid[pid >= 0], minlength=mix.n_processes)) >= mix.n_processes - 6
    # FP32 velocities: some tens of roundings of 6e-8, against the speed before
    same &= pid >= 0
    off = np.linalg.norm(v.reshape(-1, 3) - v_o.reshape(-1, 3), axis=1)[same]
    before = np.linalg.norm(vel, axis=1)[same]
    assert np.quantile(off / before, 0.99) <= 1e-5
