"""Several steps per launch for systems with virtual sites that belong to one
body each and with constraint clusters, against the same steps taken one kernel
after the other.  Mixed precision: equal bit for bit.  Double: the kernels may
round differently in the last bit, and a constraint's convergence test may then
stop a sweep earlier, within the constraint tolerance (1e-10: positions to
1e-10 d, velocities to 1e-10 d / dt)."""
import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems
from test_gpu_local_steps import bodies_of

pytestmark = pytest.mark.gpu


def with_sites(spec, per_body, seed=1):
    """Sites for the bodies of spec, per_body[k % len] for body k: averages of
    two or three of its atoms, some of them sharing parents."""
    rng = np.random.default_rng(seed)
    n = spec.num_atoms
    sites, pos = [], []
    for k, lab in enumerate(np.unique(spec.body_indices[spec.body_indices > 0])):
        atoms = np.flatnonzero(spec.body_indices == lab)
        for _ in range(per_body[k % len(per_body)]):
            np_ = 3 if len(atoms) > 2 and rng.random() < 0.6 else 2
            parents = rng.choice(atoms, np_, replace=False)
            w = rng.uniform(0.1, 1.0, np_)
            w /= w.sum()
            sites.append((2 if np_ == 3 else 1, n + len(sites), [int(a) for a in parents], list(w)))
            pos.append(w @ spec.positions[parents])
    m = len(sites)
    pos = np.array(pos).reshape(m, 3)
    x = np.concatenate([spec.positions, pos])
    return systems.SystemSpec(
        masses=np.concatenate([spec.masses, np.zeros(m)]),
        body_indices=np.concatenate([spec.body_indices, np.zeros(m, np.int32)]), positions=x,
        velocities=np.concatenate([spec.velocities, np.zeros((m, 3))]), tether_k=rng.uniform(500, 1500, n + m),
        tether_r0=x + 0.01 * rng.normal(size=x.shape), dt=spec.dt, rotation_mode=spec.rotation_mode), sites


def with_clusters(spec, shapes, seed=2):
    """The last free atoms of spec moved together into molecules."""
    rng = np.random.default_rng(seed)
    free = np.flatnonzero((spec.body_indices == 0) & (spec.masses > 0))
    base = np.array([[0, 0, 0], [0.12, 0, 0], [-0.03, 0.11, 0], [0.04, 0.03, 0.1]])
    cons, at = [], 0
    for sh in shapes:
        n = max(max(p) for p in sh) + 1
        atoms = free[at:at + n]
        at += n
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        spec.positions[atoms] = spec.positions[atoms[0]] + base[:n] @ q.T
        cons += [(int(atoms[i]), int(atoms[j]), float(np.linalg.norm(spec.positions[atoms[i]] - spec.positions[atoms[j]])))
                 for i, j in sh]
    spec.tether_r0[free] = spec.positions[free] + 0.01 * rng.normal(size=(len(free), 3))
    return cons


def compare(hip, spec, sites, cons, precision, runs, lanes=None):
    ctx = []
    for fusion in (True, False):
        c = hip.Context.from_spec(spec, precision=precision, constraints=cons or None)
        if cons:
            c.set_constraint_tolerance(1e-10)
        if sites:
            c.set_virtual_sites(sites)
        for n, L in (lanes or {}).items():
            c.set_lanes(n, L)
        c.set_positions(spec.positions)
        c.set_velocities(spec.velocities)
        c.use_fusion(fusion)
        for n in runs:
            c.step(n)
        ctx.append(c)
    a, b = ctx
    for what in ("positions", "velocities", "forces", "kinetic_energies", "body_states_array"):
        x, y = getattr(a, what)(), getattr(b, what)()
        if precision == "mixed":
            np.testing.assert_array_equal(x, y, err_msg=what)
        elif x.size:
            rel = 1e-12 if not cons else 1e-9 if what == "positions" else 1e-6
            np.testing.assert_allclose(x, y, rtol=0, atol=rel * np.abs(y).max(), err_msg=what)
    assert a.potential_energy() == pytest.approx(b.potential_energy(), rel=1e-12 if not cons else 1e-6)
    assert a.time() == b.time()
    assert a.constraint_failures() == 0


@pytest.mark.parametrize("mode", [10, 0])
@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("n,count,lanes,per_body", [
    (2, 65, 1, [1]), (3, 64, 1, [1]), (3, 130, 1, [0, 2, 1]), (4, 63, 1, [3]), (5, 20, 1, [1, 0]), (6, 33, 1, [2]),
    (7, 10, 1, [4]), (20, 9, 1, [1, 2]), (20, 9, 4, [1])])
def test_sites_of_bodies(hip, mode, precision, n, count, lanes, per_body):
    spec, sites = with_sites(bodies_of(n, count, mode, 7), per_body)
    compare(hip, spec, sites, None, precision, (2, 9), {n: lanes})


TRIANGLE, PAIR = [(0, 1), (1, 2), (0, 2)], [(0, 1)]
CHAIN, TETRAHEDRON = [(0, 1), (1, 2), (2, 3)], [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]


@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("shapes", [[TRIANGLE] * 65, [PAIR] * 64 + [TRIANGLE[:2]] * 3, [CHAIN, TETRAHEDRON] * 4,
                                    [PAIR, TRIANGLE, CHAIN] * 5])
@pytest.mark.parametrize("steps", [2, 66])
def test_clusters(hip, precision, shapes, steps):
    spec, sites = with_sites(systems.water_box(20, 0.5, num_free=200, seed=5, rotation_mode=10, free_spacing=0.5), [1])
    cons = with_clusters(spec, shapes)
    compare(hip, spec, sites, cons, precision, (steps, 3))
