"""Steps kept in registers (systems whose force on an atom depends on that
atom alone) against the per-step launches of the same steps, fusion off: the
same trajectory bit for bit in mixed precision, and in double precision to
1e-12 of each array's largest value (an ulp per step, 2.2e-16, grown over at
most 131 steps of a stable trajectory).

Sizes where the kernel's branches meet: the unrolled body sizes 2, 3, 4 and 6,
the general loop around its batch of eight, several lanes per body with uneven
shares, one lane for many atoms, bodies too large for the LDS (per-step path),
partly filled tiles, no bodies, no free atoms; step counts around the
boundaries of one launch; uniform, per-atom and no tether; adopted arrays."""
import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems

pytestmark = pytest.mark.gpu


def bodies_of(n, count, mode, free=0, seed=3):
    rng = np.random.default_rng([seed, n])
    side = int(np.ceil((count + free) ** (1 / 3)))
    centres = systems.lattice_points(rng, count + free, side, 0.6, 0.02)
    m = rng.uniform(1.0, 20.0, (count, n))
    local = rng.normal(size=(count, n, 3)) * 0.1
    x = np.concatenate([(centres[:count, None] + local).reshape(-1, 3), centres[count:]])
    m = np.concatenate([m.ravel(), rng.uniform(1.0, 20.0, free)])
    lab = np.concatenate([np.repeat(np.arange(1, count + 1), n), np.zeros(free)]).astype(np.int32)
    return systems.SystemSpec(masses=m, body_indices=lab, positions=x,
                              velocities=systems.maxwell_boltzmann(rng, m, 300.0), tether_k=np.full(m.size, 1000.0),
                              tether_r0=x + 0.01 * rng.normal(size=x.shape), dt=0.001, rotation_mode=mode)


def compare(hip, spec, precision, runs, lanes=None, block=None):
    a = hip.Context.from_spec(spec, precision=precision)
    b = hip.Context.from_spec(spec, precision=precision)
    b.use_fusion(False)
    for c in (a, b):
        if block:
            c.set_launch(block)
        for n, L in (lanes or {}).items():
            c.set_lanes(n, L)
    for steps in runs:
        a.step(steps)
        b.step(steps)
    for what in ("positions", "velocities", "forces", "kinetic_energies", "body_states_array"):
        x, y = getattr(a, what)(), getattr(b, what)()
        if precision == "mixed":
            np.testing.assert_array_equal(x, y, err_msg=what)
        elif x.size:
            np.testing.assert_allclose(x, y, rtol=0, atol=1e-12 * np.abs(y).max(), err_msg=what)
    assert a.potential_energy() == pytest.approx(b.potential_energy(), rel=1e-12)
    assert a.time() == b.time()


@pytest.mark.parametrize("mode", [10, 0, 1])
@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("n,count,free,lanes", [
    (2, 65, 1, 1), (3, 130, 300, 1), (4, 64, 0, 1), (5, 63, 0, 1), (6, 100, 7, 1), (7, 70, 0, 1), (8, 70, 5, 1),
    (8, 70, 5, 8), (9, 40, 0, 2), (17, 33, 0, 2), (20, 50, 0, 4), (20, 50, 0, 1), (33, 20, 0, 4), (300, 3, 0, 2)])
def test_body_sizes(hip, mode, precision, n, count, free, lanes):
    compare(hip, bodies_of(n, count, mode, free), precision, (2, 9), lanes={n: lanes})


@pytest.mark.parametrize("precision,mode", [("mixed", 10), ("mixed", 0), ("double", 10)])
@pytest.mark.parametrize("steps", [1, 2, 64, 65, 66, 130])
def test_step_counts(hip, precision, mode, steps):
    spec = systems.heterogeneous(150, 90, seed=8, rotation_mode=mode)
    spec.tether_r0 = spec.tether_r0 + 0.01
    compare(hip, spec, precision, (steps, 1), block=128)


@pytest.mark.parametrize("tether", ["per atom", "none"])
def test_spring_constants(hip, tether):
    spec = systems.heterogeneous(150, 90, seed=9, rotation_mode=10)
    spec.tether_r0 = spec.tether_r0 + 0.01
    n = spec.num_atoms
    spec.tether_k = np.random.default_rng(1).uniform(500, 2000, n) if tether == "per atom" else np.zeros(n)
    compare(hip, spec, "mixed", (20,))
    if tether == "none":
        a = hip.Context.from_spec(spec, set_state=False)
        free = hip.Context(spec.masses, spec.body_indices, spec.dt, 10, "mixed")   # no force field at all
        for c in (a, free):
            c.set_positions(spec.positions)
            c.set_velocities(spec.velocities)
            c.step(20)
        np.testing.assert_array_equal(a.positions(), free.positions())


def test_free_atoms_alone(hip):
    spec = systems.water_box(0, 0.3, num_free=513, seed=2, free_spacing=0.3)
    spec.tether_r0 = spec.tether_r0 + 0.02
    for precision in ("mixed", "double"):
        compare(hip, spec, precision, (70,))


@pytest.mark.parametrize("precision", ["mixed", "double"])
def test_adopted_arrays(hip, precision):
    from test_gpu_force_slot import adopted_context
    spec = systems.heterogeneous(120, 80, seed=11, rotation_mode=10)
    spec.tether_r0 = spec.tether_r0 + 0.01
    out = []
    for fusion in (True, False):
        g, arr, _ = adopted_context(hip, spec, precision, 10, tethered=True)
        g.set_positions(spec.positions)
        g.set_velocities(spec.velocities)
        g.use_fusion(fusion)
        g.step(70)
        out.append((arr.positions(), arr.velocities(), g.kinetic_energies()))
        arr.check_w_untouched()
    for x, y in zip(*out):
        if precision == "mixed":
            np.testing.assert_array_equal(x, y)
        else:
            # (a force within an ulp of a fixed-point step, 2^-32 kJ/mol/nm, may truncate either way)
            np.testing.assert_allclose(x, y, rtol=0, atol=1e-10 * np.abs(y).max())


def test_batch_equals_members_alone(hip):
    specs = [bodies_of(2, 65, 10, 3), systems.water_box(200, 0.3125, num_free=40, seed=5), bodies_of(20, 30, 10)]
    alone = [hip.Context.from_spec(s) for s in specs]
    members = [hip.Context.from_spec(s) for s in specs]
    b = hip.Batch()
    b.set_members(members)
    b.step(70)
    for c, m in zip(alone, members):
        c.step(70)
        np.testing.assert_array_equal(c.positions(), m.positions())
        np.testing.assert_array_equal(c.velocities(), m.velocities())
