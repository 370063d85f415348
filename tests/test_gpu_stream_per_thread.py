"""A context whose stream is the calling thread's own (hipStreamPerThread): its
read-backs, which other threads help to empty, hold the state after the steps
queued before them."""
import ctypes

import numpy as np
import pytest

from openmm_rigidbody_plugin_amd import systems

pytestmark = pytest.mark.gpu
PER_THREAD = ctypes.c_void_p(2)


def test_large_read_backs(hip):
    spec = systems.water_box(80000, 0.3125, num_free=1001, seed=6)       # 5.8 MB of positions
    a, b = hip.Context.from_spec(spec), hip.Context.from_spec(spec)
    assert hip.lib().rbhip_set_stream(a.handle, PER_THREAD) == 0
    for _ in range(4):
        a.step(60)
        b.step(60)
        for what in ("positions", "velocities", "forces"):
            np.testing.assert_array_equal(getattr(a, what)(), getattr(b, what)(), err_msg=what)
    a.close()
