"""Sampled scattering angles past the ends of cos(chi): a collision neither adds
energy nor loses more than the recoil, however far the sampler's rounding takes the
cosine past 1 (the Surendra quotient in FP32 by 1.4e-3 at 1e-5 eV).  On the CPU with
the device's own functions compiled for the host, on the GPU through the batch
operator."""
import os
import subprocess

import numpy as np
import pytest

import ekmc
from helpers import condition, mixture, speeds, unit_vectors

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_collisions_keep_the_energy_balance_on_the_host(tmp_path):
    exe = str(tmp_path / "scattering_angles")
    native = os.path.join(ROOT, "tests", "native")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I" + os.path.join(native, "host"),
                    os.path.join(native, "scattering_angles.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    bad, n = (int(v) for v in out.stdout.splitlines()[-1].split())
    assert n > 100_000 and bad == 0, out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("precision,ulp", [(ekmc.FP64, 2.0 ** -53), (ekmc.MIXED, 2.0 ** -24)])
@pytest.mark.parametrize("temperature", ["false", "true"])
def test_surendra_from_a_microvolt(precision, ulp, temperature):
    mix = mixture([dict(elastic=True, energy=np.array([0.0, 1000.0]), sigma=np.array([1e-19, 1e-19]),
                        mass_amu=28.0, scattering="surendra")])
    num = ekmc.numerics_default()
    num.precision = precision
    num.gas_temperature_effect = ekmc.GASTEMP[temperature]
    num.n_interp_points = 1000
    cond = condition(n_e=64)
    if temperature == "true":
        cond.gas_temperature = 1e-14  # targets of 2e-6 m/s; the slowest electron has 593
    eng = ekmc.Engine(mix, [cond], num)
    rng = np.random.default_rng(8)
    n = 40000
    energy = np.exp(rng.uniform(np.log(1e-6), np.log(400.0), n))
    vel = unit_vectors(rng, n) * speeds(energy)[:, None]
    var = rng.uniform(1e-6, 1.0, (n, ekmc.VARIATES_PER_EVENT))
    var[:, 6] = np.resize([0.0, 2.0 ** -24, 1e-4, 1e-2, 0.5, 1.0 - 2.0 ** -24, rng.uniform()], n)
    var[:, 5] = 1e-11  # a real collision at every energy
    pid, out, e_out, *_ = eng.op_collide(0, 500.0, vel, energy, np.full(n, 1e13), var)
    eng.close()
    assert np.all(pid == 0)
    out = out.reshape(-1, 3)
    assert np.all(np.isfinite(out)) and np.all(np.isfinite(e_out))
    ratio = np.linalg.norm(out, axis=1) / np.linalg.norm(vel, axis=1)
    recoil = 2 * ekmc.EMASS / (28.0 * ekmc.AMU)  # most of the speed that a target at rest takes
    slack = 64 * ulp + (1e-7 if temperature == "true" else 0.0)  # roundings; the targets' speed
    assert np.all(ratio <= 1 + slack) and np.all(ratio >= 1 - 1.1 * recoil - slack)
