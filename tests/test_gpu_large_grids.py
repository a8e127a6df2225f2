"""Launches of more blocks than one grid dimension takes (2^24 of 256 threads)."""
import numpy as np
import pytest

from tests import microsystems as ms

pytestmark = pytest.mark.gpu


def test_list_build_over_2_to_the_24_blocks():
    """Ten systems of 6,554 one-particle compounds beside one of 526,000 solvents: the build counts 65,540
    compounds x 257 segments of solvents, 16.8 million blocks.  Every system's lists are its own."""
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(*[np.arange(19) * 2.0 + 0.5] * 3, indexing="ij"), -1).reshape(-1, 3)[:6554]
    compounds = ms.build(40.0, [((p[None, :] + rng.uniform(-0.7, 0.7, 3)), [1]) for p in g], [])
    n = 526_000
    m = 81                                              # 81^3 sites, 0.8 nm apart
    sites = rng.permutation(m ** 3)[:n]
    x = (np.stack([sites // m ** 2, sites // m % m, sites % m], 1) + 0.5) * 0.8
    solvents = ms.build(64.8, [], x)
    p = RunParams(max_compound_neighbors=8, max_compound_solvents=8, max_solvent_neighbors=64)
    assert 10 * 6554 * ((n + 2047) // 2048) > 2 ** 24
    both = Engine([compounds] * 10 + [solvents], p)
    got = both.neighbors()
    one, other = Engine([compounds], p), Engine([solvents], p)
    want_cc, want_ss = one.neighbors()[0], other.neighbors()[2]
    for r in (0, 9):
        for c in range(0, 6554, 13):
            assert np.array_equal(got[0][r * 6554 + c] - r * 6554, want_cc[c]), (r, c)
    assert sum(map(len, want_cc)) > 0 and sum(map(len, want_ss[::101])) > 0
    for s in range(0, n, 101):
        assert np.array_equal(got[2][s], want_ss[s]), s
    for e in (both, one, other):
        e.close()
