"""The step-by-step launches that remain beside the steps in registers: systems
with bonds, with sites that are no averages and with large clusters of
constraints.  Replayed graphs against the same launches (bit for bit, whole
chunks of 16 boundaries with and without a remainder, several replays with
other work between them), and the fused pass against part 1 and part 2 (bit for
bit in mixed precision, over the body sizes where its branches meet)."""
import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems
from test_gpu_constraints import constrained_spec
from test_gpu_local_steps import bodies_of
from test_gpu_sites import site_spec

pytestmark = pytest.mark.gpu


def assert_equal(a, b):
    for what in ("positions", "velocities", "forces", "kinetic_energies", "potential_energy"):
        np.testing.assert_array_equal(getattr(a, what)(), getattr(b, what)(), err_msg=what)


def contexts(hip, kind, precision, mode):
    out = []
    for _ in range(2):
        if kind == "clusters":
            spec, cons = constrained_spec(mode, seed=16)
            c = hip.Context.from_spec(spec, precision=precision, constraints=cons)
        else:
            spec, sites = site_spec(mode, seed=17)
            c = hip.Context.from_spec(spec, precision=precision, set_state=False)
            c.set_virtual_sites(sites)
            c.set_positions(spec.positions)
            c.set_velocities(spec.velocities)
        assert "steps=launched" in c.describe()
        out.append(c)
    return out


@pytest.mark.parametrize("kind", ["clusters", "sites"])
@pytest.mark.parametrize("precision,mode", [("mixed", 10), ("double", 0)])
def test_replayed_graphs_equal_launches(hip, kind, precision, mode):
    replayed, launched = contexts(hip, kind, precision, mode)
    launched.use_graph(False)
    for steps in (18, 34, 3, 41, 60):
        replayed.step(steps)
        launched.step(steps)
        assert_equal(replayed, launched)


def bond_neighbours(spec, c):
    """Bonds between atoms of consecutive bodies (and free atoms)."""
    a = np.arange(0, spec.num_atoms - 7, 5)
    c.add_bonds(np.stack([a, a + 7], 1), np.linalg.norm(spec.positions[a] - spec.positions[a + 7], axis=1), 200.0)


@pytest.mark.parametrize("mode", [10, 0])
@pytest.mark.parametrize("n,count,lanes", [(2, 65, 1), (3, 130, 1), (4, 64, 1), (5, 63, 1), (6, 100, 1), (8, 70, 1),
                                           (8, 70, 8), (17, 33, 2), (20, 50, 4), (33, 20, 4)])
def test_fused_pass_equals_the_two_passes(hip, mode, n, count, lanes):
    spec = bodies_of(n, count, mode, 9)
    a, b = hip.Context.from_spec(spec), hip.Context.from_spec(spec)
    b.use_fusion(False)
    for c in (a, b):
        c.set_lanes(n, lanes)
        bond_neighbours(spec, c)
        assert "steps=launched" in c.describe()
        c.step(2)
        c.step(9)
    assert_equal(a, b)


@pytest.mark.parametrize("mode", [10, 0])
def test_fused_pass_with_shared_frames(hip, mode):
    spec = systems.water_box(3000, 0.3, num_free=500, seed=9, rotation_mode=mode)
    a, b = hip.Context.from_spec(spec), hip.Context.from_spec(spec)
    b.use_fusion(False)
    for c in (a, b):
        bond_neighbours(spec, c)
        c.step(15)
        assert "sharedShapes=[N3:" in c.describe()
    assert_equal(a, b)
