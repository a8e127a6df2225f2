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


@pytest.mark.parametrize("box,cells", [(200.0, 166 ** 3), (310.0, 256 ** 3)])
def test_list_build_over_many_cells(box, cells):
    """Boxes of 4.6 million cells (over 2^32 threads at 1,024 a cell) and of 16.8 million (at 256, whose
    launch clears the cells' counters for the next build): built twice, the lists are the oracle's."""
    from oracle.oracle import KIND_CS, KIND_SS, Oracle
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    rng = np.random.default_rng(9)
    g = np.stack(np.meshgrid(*[np.arange(8) * 0.5] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = np.mod(np.concatenate([g + c for c in ((0.2, 0.2, 0.2), (box - 2.1, 0.3, box / 2), (box / 2,) * 3)])
               + rng.uniform(-0.05, 0.05, (3 * len(g), 3)), box)
    s = ms.build(box, [([(3.0, 3.0, 5.0), (3.1, 3.0, 5.0)], [1, 2])], x)
    p = RunParams(nlist_interval=0)
    e, o = Engine([s], p), Oracle(s, p, precision=32)
    assert e.config()["n_cells"] == cells
    o.compute_forces()
    for build in range(2):
        _, cs, ss = e.neighbors()
        for got, want in ((cs, o.neighbors(KIND_CS)), (ss, o.neighbors(KIND_SS))):
            assert sum(map(len, want)) > 0
            assert all(np.array_equal(np.sort(a), np.sort(b)) for a, b in zip(got, want)), build
        e.rebuild_neighbors()
    e.close()
