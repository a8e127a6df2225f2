"""The all-pairs tiles pad a compound to whole fours with rows of zero constants.  They add nothing
wherever a solvent lies in a large box, 1,000 nm among its coordinates."""
import numpy as np
import pytest

from tests import microsystems as ms
from tests.conftest import rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accumulation", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 6])
def test_solvents_anywhere_in_a_large_box(n, accumulation):
    from oracle.oracle import Oracle
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    x = np.array([1000.0, 1000.0, 1000.5]) + 0.4 * np.arange(n)[:, None] * np.array([0.0, 0.6, 0.8])
    solvents = [(1000.0, 1000.0, 1000.0), (1000.5, 1000.0, 1000.0), (1.0, 1.0, 1.0), (0.0, 0.0, 0.0), (1e3, 0.0, 1e3)]
    s = ms.build(2000.0, [(x, [1] * n)], solvents)
    p = RunParams(accumulation=accumulation, cutoff=20.0)
    e = Engine([s], p)
    got = e.compute_forces()
    energies = e.energies()[0]
    e.close()
    want = Oracle(s, p, precision=32).compute_forces()
    assert np.isfinite(got[1]).all() and all(np.isfinite(v) for v in energies.values())
    # the bar of the force parity tests: both sides are FP32 sums of the same pairs
    assert rel_rms(got[0], want[0]) <= 1e-5 and rel_rms(got[1], want[1]) <= 1e-5
