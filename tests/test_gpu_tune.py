"""lbm_tune measures what runs: where the fastest variant of the one-step kernel beats the launches of several
steps that the rule plans, the context keeps to it, until something that the measurement depended on changes."""
import numpy as np
import pytest

from madpac_amd import lbm

pytestmark = pytest.mark.gpu


def _box(size, solids, porosity=False):
    rng = np.random.default_rng(3)
    lat = lbm.Lattice(*size, 0.6, periodic=(True, True, True), force=(1e-6, 0.0, 0.0))
    lat.set_flags(rng.random(lat.n) >= solids)
    if porosity:
        lat.set_porosity(rng.random(lat.n))
    lat.init_equilibrium(u=0.01 * rng.standard_normal((lat.n, 3)))
    return lat


def test_single_steps_where_they_measure_faster():
    # rows of 8 cells, a tenth of them solid: 90 us a step singly, 112 in pairs
    print("[gpu] tune 8 x 8 x 8192", flush=True)
    with _box((8, 8, 8192), 0.1) as lat, _box((8, 8, 8192), 0.1) as plain:
        lat.tune(40)
        assert lat.step_plan() == (1, 0)
        for n in (7, 70):
            lat.step(n, graph=n > 32)
            plain.step(n)
        assert np.array_equal(lat.get_populations(), plain.get_populations())
        # the rule holds again for what was not measured, and the measurement where all is as it was
        plan = plain.step_plan()
        lat.set_porosity(np.full(lat.n, 0.5))
        assert lat.step_plan() == plan
        lat.set_porosity(None)
        assert lat.step_plan() == (1, 0)
        lat.set_boundary_class(3, lbm.BC_MOVING_WALL, mask=1 << 16)
        lat.set_wall_classes(np.full(lat.n, 3))
        lat.init_equilibrium()
        walls = lat.step_plan()
        assert walls == plan
        lat.set_boundary_class(3, lbm.BC_MOVING_WALL, mask=0)
        assert lat.step_plan() == (1, 0)
        lat.set_coupling_cells([5, 900])
        lat.set_flags(np.ones(lat.n))
        assert lat.step_plan()[0] == 2
        lat.init_equilibrium()
        lat.tune(variant=6)
        lat.set_flags(np.random.default_rng(3).random(lat.n) >= 0.1)
        assert lat.step_plan() == plan  # an explicit choice takes the measurement back


def test_pairs_where_they_measure_faster():
    # 74 us a step in pairs, 111 singly
    print("[gpu] tune 128^3", flush=True)
    with lbm.Lattice(128, 128, 128, 0.6, periodic=(True,) * 3) as lat:
        lat.set_flags(np.ones(lat.n))
        lat.init_equilibrium()
        plan = lat.step_plan()
        lat.tune(10)
        assert lat.step_plan() == plan and plan[0] == 2
        before = lat.moments()
        lat.tune(3)  # the state is as it was
        assert np.array_equal(lat.moments(), before)


def test_the_state_survives_the_measurement():
    with _box((64, 64, 64), 0.0) as lat, _box((64, 64, 64), 0.0) as plain:
        lat.step(3)
        lat.tune(5)
        lat.step(4)
        for _ in range(7):
            plain.step(1)
        assert np.array_equal(lat.get_populations(), plain.get_populations())
