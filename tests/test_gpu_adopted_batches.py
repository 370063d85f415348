"""Kernels that load several adopted atoms per lane before they store any: the
free atoms of the step kernels and the library's force field, at counts around
the ends of a batch, a wave and a tile.  Both
layouts run the same arithmetic, so results are equal bit for bit."""
import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems
from test_gpu_force_slot import adopted_context, quantized, tether

pytestmark = pytest.mark.gpu

COUNTS = [1, 63, 64, 65, 129, 191, 192, 193, 255, 256, 257, 513, 1025]


def pair(hip, spec, precision, block, tethered):
    g, arr, _ = adopted_context(hip, spec, precision, 10, seed=3, tethered=tethered)
    b = hip.Context(spec.masses, spec.body_indices, spec.dt, 10, precision)
    if tethered:
        b.set_tether(spec.tether_k, spec.tether_r0)
    for c in (g, b):
        c.set_launch(block)
    return g, arr, b


@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("free", COUNTS)
def test_free_atoms_of_the_step_kernels(hip, free, precision, block):
    spec = systems.water_box(5, 0.3125, num_free=free, seed=2, free_spacing=0.3)
    g, arr, b = pair(hip, spec, precision, block, False)
    arr.write_positions(spec.positions)
    f = quantized(tether(spec, spec.positions))[1]
    arr.write_forces(f)
    g.state_changed(g.STATE_POSITIONS)
    arr.write_velocities(spec.velocities)
    g.state_changed(g.STATE_VELOCITIES)
    b.set_positions(arr.positions())
    b.set_velocities(arr.velocities())
    b.set_forces(f)
    for _ in range(3):
        g.part1()
        b.part1()
        f = quantized(tether(spec, arr.positions()))[1]
        arr.write_forces(f)
        b.set_forces(f)
        g.part2()
        b.part2()
    np.testing.assert_array_equal(g.velocities(), b.velocities())
    np.testing.assert_array_equal(g.kinetic_energies(), b.kinetic_energies())
    atoms = spec.body_indices <= 0
    np.testing.assert_array_equal(g.positions()[atoms], b.positions()[atoms])
    arr.check_w_untouched()


@pytest.mark.parametrize("per_atom", [False, True])
@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("free", COUNTS)
def test_the_force_field(hip, free, precision, block, per_atom):
    spec = systems.water_box(0, 0.3, num_free=free, seed=4, free_spacing=0.3)
    spec.tether_r0 = spec.tether_r0 + 0.02
    if per_atom:
        spec.tether_k = np.random.default_rng(1).uniform(500, 2000, free)
    g, arr, b = pair(hip, spec, precision, block, True)
    for c in (g, b):
        c.set_positions(spec.positions)
        c.compute_forces()
    got = arr.force.download()[:, :free]
    want = np.trunc(b.forces()[arr.order] * 2.0 ** 32).astype(np.int64).T
    np.testing.assert_array_equal(got, want)
    assert not arr.force.download()[:, free:].any()
    assert g.potential_energy() == b.potential_energy()
