"""List capacities bound the lists and nothing else: an engine that had to be given larger ones runs the
same trajectory, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accumulation", [0, 1])
def test_capacities_change_no_bit(accumulation):
    """60 compounds and 3,000 solvents: up to 4,260 listed items at the larger capacities, 3,780 at the
    smaller ones, on either side of 4,096, where a system's items stop being summed in parts."""
    from quantom_amd import systems
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    s = systems.build_system(0xCA9, 6, 10, 8.0, 5, 3000, compound_size=33, central_first=True, confine=1.0)
    got = []
    for solvents in (1024, 16384):
        e = Engine([s], RunParams(accumulation=accumulation, nlist_interval=5, max_compound_solvents=solvents))
        f = e.compute_forces()
        assert 32 < e.neighbor_counts()[1].max() <= 1024
        e.step(12)
        got.append((*f, *e.get_state()))
        e.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
