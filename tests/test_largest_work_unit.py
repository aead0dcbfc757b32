"""The largest work units: a unit's EEDF counts are 16-bit, so no unit holds more than
65535 electrons, also where the asked size rounds up to whole waves beyond that.  Every
electron of the condition sits in the lowest of four cells (the grid reaches 1.2 times
the energy of the hot start), so a unit of 65536 would count none."""
import numpy as np
import pytest

import ekmc
from helpers import condition, mixture

pytestmark = pytest.mark.gpu


def _eedf(precision, electrons, work_chunk):
    top = 20000.0
    mix = mixture([
        dict(elastic=True, energy=np.array([0.0, top]), sigma=np.array([1e-19, 1e-19]), mass_amu=40.0),
        dict(threshold=10.0, energy=np.array([10.0, 10.5, top]), sigma=np.array([0.0, 1e-19, 1e-19]), mass_amu=40.0)])
    num = ekmc.numerics_default()
    num.precision = precision
    num.work_chunk = work_chunk
    num.initial_elec_temp_over_gas_temp = 60.0 * 11604.5 / 300.0
    num.n_energy_cells = 4
    num.max_collisions_before_ss = 40.0
    num.n_integration_points = 60
    num.seed = 3
    eng = ekmc.Engine(mix, [condition(en=5.0, angle=90.0, bn=100.0, n_e=electrons)], num)
    eng.solve()
    cells, eedf = eng.eedf(0)
    eng.close()
    return np.array(cells), np.array(eedf)


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("electrons,work_chunk", [(65536, 65535), (65536, 65473), (65536, 65472), (131073, 65535),
                                                  (65535, 65535)])
def test_every_electron_is_counted(precision, electrons, work_chunk):
    cells, eedf = _eedf(precision, electrons, work_chunk)
    _, small = _eedf(precision, electrons, 1024)
    # all counts in one cell: the normalised value is that cell's alone
    assert cells[0] > 20.0 and eedf[0] > 0 and np.all(eedf[1:] == 0)
    assert np.all(small[1:] == 0)
    width = 2.0 * cells[0]
    # normalised: sum of f sqrt(u) du = 1 (a few roundings)
    assert abs(eedf[0] * np.sqrt(cells[0]) * width - 1.0) < 1e-12
