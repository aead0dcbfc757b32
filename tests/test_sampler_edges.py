"""Scattering angles at the ends of the samplers' variates on the GPU: the
post-collision velocity is finite, and an elastic collision changes the speed by
no more than the recoil, also where the sampled cos(chi) rounds past 1."""
import numpy as np
import pytest

import ekmc
from helpers import condition, mixture, speeds, unit_vectors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("model,params", [("coulombScreen", (0.0, 1.0)), ("coulombScreen", (1.0, 0.05)),
                                          ("surendra", ()), ("isotropic", ())])
def test_extreme_angles_keep_velocities_finite(precision, model, params):
    mix = mixture([dict(elastic=True, energy=np.array([0.0, 1000.0]), sigma=np.array([1e-19, 1e-19]),
                        mass_amu=28.0, scattering=model, params=params)])
    num = ekmc.numerics_default()
    num.precision = precision
    num.n_interp_points = 1000
    eng = ekmc.Engine(mix, [condition(n_e=64)], num)
    rng = np.random.default_rng(5)
    n = 30000
    energy = np.exp(rng.uniform(np.log(0.05), np.log(400.0), n))
    vel = unit_vectors(rng, n) * speeds(energy)[:, None]
    var = rng.uniform(1e-6, 1.0, (n, ekmc.VARIATES_PER_EVENT))
    # the variate of cos(chi): both ends, one FP32 step from them, and one between
    var[:, 6] = np.resize([0.0, 2.0 ** -24, 0.5, 1.0 - 2.0 ** -24, 1.0 - 2.0 ** -23], n)
    var[:, 5] = 1e-6  # a real collision
    nue = np.full(n, 1e13)
    pid, out, e_out, *_ = eng.op_collide(0, 500.0, vel, energy, nue, var)
    eng.close()
    assert np.all(pid == 0)
    out = out.reshape(-1, 3)
    assert np.all(np.isfinite(out)) and np.all(np.isfinite(e_out))
    # recoil of a 28 amu target: at most 2 m/M of the speed; FP32 rounding of a
    # cos(chi) past 1 adds its few ulp
    ratio = np.linalg.norm(out, axis=1) / np.linalg.norm(vel, axis=1)
    recoil = 2 * ekmc.EMASS / (28.0 * ekmc.AMU)
    assert np.all(ratio <= 1 + 1e-5) and np.all(ratio >= 1 - 1.1 * recoil - 1e-5)
