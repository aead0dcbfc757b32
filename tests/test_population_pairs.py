"""Population control of one interval on the GPU, electron by electron: the
pool the flights leave (ekmc_op_interval_pool) against the N electrons after
removals, moves and clones, and the sampled sums against those N electrons.

With more than N electrons alive, every one of the N is a different electron of
the pool; with fewer, every electron of the pool is among the N and the others
are copies of pool electrons.  (A clone and its source of an interval before
are the same in position and velocity until one of them collides, so the pool
is compared with its multiplicities.)  Sizes sit on both sides of the limits where the
removal plan, the pairs and the reductions change their path (32768 electrons;
448 and 4096 chunks of 64)."""
import numpy as np
import pytest

import ekmc

pytestmark = pytest.mark.gpu

# conditions of the 64-condition scan: attachment (holes, then clones), both
# holes and newborns, and strong ionization (removals)
CONDITIONS = [9, 12, 15, 17, 21]


def _key(pos, vel):
    a = np.ascontiguousarray(np.concatenate([pos, vel], axis=1))
    return a.view([("", a.dtype)] * 6).ravel()


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("n,chunk", [(64, 64), (129, 64), (5003, 0), (28672, 64), (28673, 64), (32768, 512),
                                     (32769, 512), (262144, 64), (262145, 64)])
def test_population_control_keeps_the_pool(precision, n, chunk):
    mix, conds, num = ekmc.workload("cfg3_o2like_batched", n_electrons=n, conditions=CONDITIONS)
    num.precision = precision
    num.seed = 77
    num.work_chunk = chunk
    num.n_integration_points = 1e15
    eng = ekmc.Engine(mix, conds, num)
    eng.initialize()
    eng.step(6)
    removed = cloned = 0
    for turn in range(2 * len(conds)):
        c = turn % len(conds)
        pool, _, _ = eng.op_interval_pool(c, capacity=4 * n + 4096)
        pos, vel, energy, _ = eng.electrons(c)
        before, count = np.unique(_key(pool["pos"], pool["vel"]), return_counts=True)
        after, copies = np.unique(_key(pos, vel), return_counts=True)
        assert copies.sum() == n
        at = np.searchsorted(before, after)
        assert np.all(at < len(before)) and np.all(before[at] == after)
        m = len(pool["energy"])
        if m >= n:
            assert np.all(copies <= count[at])
            removed += m - n
        else:
            assert len(after) == len(before) and np.all(copies >= count)
            cloned += n - m
        s = eng.series(c)
        # FP64 sums of n values in two orders
        assert abs(s["mean_energy"][-1] - energy.mean()) <= 1e-12 * energy.mean()
        assert np.allclose(s["mean_position"][-3:], pos.mean(0), rtol=0, atol=1e-12 * np.abs(pos).max())
        assert np.allclose(s["mean_velocity"][-3:], vel.mean(0), rtol=0, atol=1e-12 * np.abs(vel).max())
        flux = (pos.T @ vel / n - np.outer(pos.mean(0), vel.mean(0))).ravel()
        assert np.allclose(s["flux_diffusion"][-9:], flux, rtol=0, atol=1e-12 * np.abs(pos).max() * np.abs(vel).max())
        assert eng.status(c).max_elec_energy >= energy.max()
    if n >= 5000:
        assert removed > 0 and cloned > 0
    eng.close()
