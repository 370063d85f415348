"""Three constrained atoms whose constraints come in any order and sense, two
or three of them or one given twice: the register kernels take the atoms in an
order of their own, and follow the oracle's sweep constraint by constraint."""
import itertools

import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems
from test_gpu_constraints import TOL, pair

pytestmark = pytest.mark.gpu


def molecules(order_of):
    """A three-atom molecule per entry of order_of (its constraints' pairs)."""
    n = len(order_of)
    spec = systems.water_box(1, 0.5, num_free=3 * n, seed=3, rotation_mode=10, free_spacing=0.5)
    rng = np.random.default_rng(4)
    free = np.flatnonzero(spec.body_indices == 0).reshape(n, 3)
    tri = np.array([[0.0, 0.0, 0.0], [0.14, 0.0, 0.0], [-0.035, 0.13, 0.0]])
    x = spec.positions
    for atoms in free:
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        x[atoms] = x[atoms[0]] + tri @ q.T
    spec.masses[free.ravel()] = rng.uniform(1.0, 20.0, 3 * n)
    spec.tether_r0 = x + 0.02 * rng.normal(size=x.shape)
    cons = [(int(atoms[i]), int(atoms[j]), float(np.linalg.norm(x[atoms[i]] - x[atoms[j]])))
            for atoms, pairs in zip(free, order_of) for i, j in pairs]
    return spec, cons


def orders():
    edges = [(0, 1), (1, 2), (0, 2)]
    out = []
    for k in (2, 3):
        for p in itertools.permutations(edges, k):
            for flip in itertools.product((0, 1), repeat=k):
                out.append([e[::-1] if f else e for e, f in zip(p, flip)])
    return out + [[(0, 1), (1, 0), (1, 2)], [(2, 0), (0, 1), (0, 2)]]


@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("steps", [1, 6])
def test_every_order_matches_the_oracle(hip, oracle, precision, steps):
    spec, cons = molecules(orders())
    o, g = pair(oracle, hip, spec, cons, precision, 1e-10)
    o.step(steps)
    g.step(steps)
    t = TOL[precision]
    np.testing.assert_allclose(g.positions(), o.positions(), rtol=0, atol=t["pos"])
    vo = o.velocities()
    np.testing.assert_allclose(g.velocities(), vo, rtol=0, atol=t["vel"] * np.abs(vo).max())
    x = g.positions()
    for a, b, d in cons:
        assert abs(np.linalg.norm(x[a] - x[b]) - d) <= 1e-8 * d
    assert g.constraint_failures() == 0
