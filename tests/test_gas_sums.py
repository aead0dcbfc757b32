"""The thermal channel choice on the GPU against the oracle with identical
variates, for gas counts around the batches of four gases whose sums are loaded
together, a gas of one process, and a gas that is absent (fraction 0)."""
import numpy as np
import pytest

import ekmc
import oracle_py as O
from helpers import condition, mixture, speeds, unit_vectors

pytestmark = pytest.mark.gpu

GRID = np.array([0.0, 0.5, 3.0, 12.0, 200.0, 1000.0])


def _gases(n_gas, absent):
    fr = np.array([1.0 + g for g in range(n_gas)])
    if absent >= 0:
        fr[absent] = 0.0
    fr /= fr.sum()
    procs = []
    for g in range(n_gas):
        common = dict(gas=g, mass_amu=4.0 + 9.0 * g)
        procs.append(dict(elastic=True, energy=GRID, sigma=1e-20 * (g + 1) * np.array([1, 3, 5, 4, 2, 1]), **common))
        if g == 1:
            continue  # one process only
        for k, thr in enumerate((0.3, 1.7, 9.0)[: 1 + g % 3]):
            e = np.array([thr, thr + 2.0, 60.0, 1000.0])
            procs.append(dict(threshold=thr, energy=e, sigma=1e-21 * (k + 2) * np.array([0, 4, 6, 3]),
                              scattering=("isotropic", "surendra", "forward")[k], **common))
    return mixture(procs, fractions=tuple(fr))


@pytest.mark.parametrize("n_gas,absent", [(1, -1), (2, 0), (3, 2), (4, -1), (5, 4), (5, 1), (8, 3), (9, 8), (9, -1)])
def test_thermal_choice_matches_oracle(n_gas, absent):
    mix = _gases(n_gas, absent)
    cond = condition(tg=2000.0, n_e=64)
    num = ekmc.numerics_default()
    num.gas_temperature_effect = ekmc.GASTEMP["true"]
    num.n_interp_points = 2000
    eng = ekmc.Engine(mix, [cond], num)
    model = O.Model(mix, cond, num)
    top = 120.0
    _, _, tot, mx, _ = model.tables(top)
    rng = np.random.default_rng(100 * n_gas + absent)
    n = 20000
    energy = np.exp(rng.uniform(np.log(0.02), np.log(100.0), n))
    vel = unit_vectors(rng, n) * speeds(energy)[:, None]
    var = rng.uniform(1e-9, 1.0, (n, ekmc.VARIATES_PER_EVENT))
    nue = np.full(n, 1.2 * mx[-1])
    pid, v, e, *_ = eng.op_collide(0, top, vel, energy, nue, var)
    eng.close()
    _, pid_o, v_o, e_o, *_ = model.collide(vel, energy, nue, var)
    assert np.array_equal(pid, pid_o)
    counts = np.bincount(pid[pid >= 0], minlength=mix.n_processes)
    assert np.any(pid < 0) and np.count_nonzero(counts) >= mix.n_processes - 6
    # the FP64 tolerance of the collision parity tests
    assert np.allclose(v.reshape(-1, 3), v_o.reshape(-1, 3), rtol=1e-12, atol=1e-6)
    assert np.allclose(e, e_o, rtol=1e-12, atol=0)
