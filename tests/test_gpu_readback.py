"""Read-backs through pinned chunks (2 MiB each, up to four threads): sizes
below, at and above one chunk and several threads' shares hold every atom, as
the anchors set at the same places show, and several threads may read several
systems at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ATOMS_PER_CHUNK = (2 << 20) / 24   # 87381.3


def system(hip, n, seed):
    x = np.random.default_rng(seed).uniform(0.0, 20.0, (n, 3))
    c = hip.Context(np.full(n, 12.0), np.zeros(n, np.int32), 0.001, 0, "double")
    c.set_positions(x)
    return c, x


@pytest.mark.parametrize("n", [1, 87381, 87382, 174762, 174763, 349526, 611671, 1100003])
def test_every_chunk_arrives(hip, n):
    assert int(ATOMS_PER_CHUNK) == 87381
    c, x = system(hip, n, n)
    np.testing.assert_array_equal(c.positions(), x)
    np.testing.assert_array_equal(c.velocities(), np.zeros((n, 3)))


def test_concurrent_readers(hip):
    made = [system(hip, n, 50 + n) for n in (400001, 300007, 90001, 500009, 1000, 250003)]
    got = [None] * len(made)

    def read(i):
        got[i] = [made[i][0].positions() for _ in range(3)]

    team = [threading.Thread(target=read, args=(i,)) for i in range(len(made))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    for (c, x), g in zip(made, got):
        for y in g:
            np.testing.assert_array_equal(x, y)
