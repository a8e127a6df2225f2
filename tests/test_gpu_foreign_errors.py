"""Errors of a program's own HIP calls stay its own: the runtime keeps the last one per thread, and no
entry point reports it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_callers_hip_error_is_not_an_entry_points(tiny_system):
    from quantom_amd.abi import THERMOSTAT_NONE, RunParams
    from quantom_amd.engine import Engine
    hip = C.CDLL("libamdhip64.so.7")
    e = Engine([tiny_system], RunParams(nlist_interval=10, thermostat=THERMOSTAT_NONE))
    calls = [lambda: e.set_parameters(e.get_parameters()), lambda: e.step(12), e.get_state, e.compute_forces,
             e.rebuild_neighbors, e.energies, lambda: e.adjoint(2, None, [1.0])]
    for call in calls:
        assert hip.hipSetDevice(1 << 20) != 0            # the caller's error
        call()
        hip.hipGetLastError()
    x = e.get_state()
    assert all(np.isfinite(v).all() for v in x)
    e.close()
