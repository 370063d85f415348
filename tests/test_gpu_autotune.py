"""The tuners compare equal work: lanes per body that take a system out of the
steps in registers (a body with its own sites on more than one lane; 20 atoms
on one lane in double precision, beyond the LDS) are not the faster ones."""
import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems
from test_gpu_local_sites import TRIANGLE, with_clusters, with_sites
from test_gpu_local_steps import bodies_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["mixed", "double"])
def test_bodies_with_sites_stay_on_one_lane(hip, precision):
    spec, sites = with_sites(systems.water_box(2000, 0.4, num_free=150, seed=5, rotation_mode=10, free_spacing=0.4), [1])
    cons = with_clusters(spec, [TRIANGLE] * 40)
    c = hip.Context.from_spec(spec, precision=precision, constraints=cons, set_state=False)
    c.set_virtual_sites(sites)
    c.set_positions(spec.positions)
    c.set_velocities(spec.velocities)
    assert "steps=registers" in c.describe()
    c.autotune(reps=3)
    assert "N3x2000:L1 " in c.describe() and "steps=registers" in c.describe()
    c.set_lanes(3, 2)
    assert "steps=launched" in c.describe()


def test_large_bodies_in_double_stay_in_registers(hip):
    c = hip.Context.from_spec(bodies_of(20, 1500, 0, 500), precision="double")
    c.autotune(reps=3)
    assert "N20x1500:L1 " not in c.describe() and "steps=registers" in c.describe()


def test_batch_of_large_bodies_in_double(hip):
    members = [hip.Context.from_spec(bodies_of(20, 700, 0, 100, seed=s), precision="double") for s in (3, 4)]
    x = [m.positions() for m in members]
    b = hip.Batch()
    b.set_members(members)
    b.set_launch(64, 0)
    b.autotune(reps=3)
    assert "N20:L1 " not in b.describe()
    assert all("steps=registers" in m.describe() for m in members)
    for m, p in zip(members, x):
        np.testing.assert_array_equal(m.positions(), p)
