"""Which systems keep their steps in registers: every workgroup of such a launch
reserves the LDS of the largest body, so beside a body of 500 atoms (two waves
per CU in mixed precision) a large box is launched step by step, a small one is
not; either way the trajectory is that of the two-pass steps."""
import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems

pytestmark = pytest.mark.gpu


def water_and(bodies, atoms):
    """`bodies` rigid waters and one body of `atoms` atoms."""
    w = systems.water_box(bodies, 0.3125, seed=12, rotation_mode=10)
    rng = np.random.default_rng(atoms)
    x, m = 5.0 + 0.4 * rng.normal(size=(atoms, 3)), rng.uniform(1.0, 20.0, atoms)
    pos = np.concatenate([w.positions, x])
    return systems.SystemSpec(
        masses=np.concatenate([w.masses, m]),
        body_indices=np.concatenate([w.body_indices, np.full(atoms, bodies + 1, np.int32)]), positions=pos,
        velocities=np.concatenate([w.velocities, systems.maxwell_boltzmann(rng, m, 300.0)]),
        tether_k=np.full(len(pos), 1000.0), tether_r0=pos + 0.01 * rng.normal(size=pos.shape), dt=w.dt, rotation_mode=10)


@pytest.mark.parametrize("bodies,atoms,way", [
    (270000, 500, "launched"), (270000, 400, "registers"), (20000, 500, "registers"), (20000, 600, "launched"),
    (64, 500, "registers")])
def test_large_body_among_waters(hip, bodies, atoms, way):
    spec = water_and(bodies, atoms)
    a, b = hip.Context.from_spec(spec), hip.Context.from_spec(spec)
    assert "steps=" + way in a.describe()
    b.use_fusion(False)
    assert "steps=launched" in b.describe()
    for c in (a, b):
        c.step(6)
    np.testing.assert_array_equal(a.positions()[-3 * 64 - atoms:], b.positions()[-3 * 64 - atoms:])
    np.testing.assert_array_equal(a.velocities()[-3 * 64 - atoms:], b.velocities()[-3 * 64 - atoms:])
