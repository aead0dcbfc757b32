"""The flight kernel's two ways to store records (a lane its own, or whole lines
by four lanes: launches with more chunks than resident waves) leave the same
bytes: a condition's electrons are the same whether it runs alone or beside a
condition large enough to change the way.  Sizes sit at the edges of a wave and of
its groups of four lanes."""
import numpy as np
import pytest

import ekmc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ekmc.FP64, ekmc.MIXED])
@pytest.mark.parametrize("n", [1, 3, 62, 65, 129, 5003])
def test_records_do_not_depend_on_the_launch(precision, n):
    out = []
    for others in ([], [400000]):
        mix, conds, num = ekmc.workload("cfg3_o2like_batched", conditions=[17, 18][: 1 + len(others)])
        for cond, size in zip(conds, [n] + others):
            cond.n_electrons = size
            cond.reduced_elec_field, cond.elec_field_angle, cond.reduced_mag_field = 150.0, 90.0, 400.0
        num.precision = precision
        num.seed = 5
        num.work_chunk = 64  # 6250 chunks of the large condition against 3072 or fewer waves
        num.n_integration_points = 1e15
        eng = ekmc.Engine(mix, conds, num)
        eng.initialize()
        eng.step(12)
        st = eng.status(0)
        out.append([*eng.electrons(0), np.array([st.real_collisions, st.null_collisions])])
        eng.close()
    for a, b in zip(*out):
        assert a.tobytes() == b.tobytes()
