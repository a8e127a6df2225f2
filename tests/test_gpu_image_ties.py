"""Positions exactly half a box apart: neither image is nearer, and the reference's sequence of
re-imagings (each against the next entry, Engine.cu:1111, 706-720) keeps the one that it has.  Coordinates
are multiples of 1/64, so that FP32 and FP64 meet the same ties; the oracle carries the sequence."""
import numpy as np
import pytest

from tests import microsystems as ms
from tests.conftest import rel_rms

pytestmark = pytest.mark.gpu


def _check(s, steps=True, **params):
    from oracle.oracle import KIND_CC, KIND_CS, KIND_SS, Oracle
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    p = RunParams(nlist_interval=0, **params)
    o, e = Oracle(s, p, precision=32), Engine([s], p)
    want = o.compute_forces()
    assert want[2] == 0
    e.set_neighbors(cc=o.neighbors(KIND_CC), cs=o.neighbors(KIND_CS), ss=o.neighbors(KIND_SS))
    got = e.compute_forces()
    # the bar of the force parity tests: both sides are FP32 sums of the same pairs
    assert rel_rms(got[0], want[0]) <= 1e-5 and rel_rms(got[1], want[1]) <= 1e-5
    e.step(1)
    assert o.step(1) == 0
    assert np.array_equal(e.get_state()[3], o.state()[3].astype(np.float32))   # the sequence's last images
    e.close()


@pytest.mark.parametrize("accumulation", [0, 1])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("before", [0, 1, 62, 63, 64, 130])
def test_solvent_half_a_box_from_a_compound(before, axis, accumulation):
    """A solvent that compound 0 moves to its upper image, or not, and `before` compounds later a tie: the
    first, a middle and the last compound of a chunk of 64, and the first of the next; then a tie of ties."""
    roll = lambda p: np.roll(np.asarray(p, float), axis, axis=-1)
    far = lambda k: [(2.625 + 0.375 * (k % 2), 0.3125 * (k // 2 % 12), 2.0 + 0.3125 * (k // 24))]
    # of two particles each: the second 0.9 nm along the axis, where the two images differ by 2 nm and more
    pair = lambda x, y: [(x, y, 1.0), (x + 0.875, y, 1.0)]
    compounds = [(roll(pair(2.625, 0.5)), [1, 1])]
    compounds += [(roll(far(k)), [1]) for k in range(before)]
    compounds += [(roll(pair(2.5, 1.375)), [1, 1]), (roll(pair(2.5, 1.875)), [2, 2])]
    solvents = roll([(0.5, 1.0, 1.0), (0.5, 1.5, 1.5), (0.375, 1.75, 0.5), (0.625, 3.5, 3.5)])
    ignores = {(c, i): [(c, 1 - i)] for c, (p, _) in enumerate(compounds) if len(p) == 2 for i in (0, 1)}
    _check(ms.build(4.0, compounds, solvents, ignores=ignores), accumulation=accumulation)


@pytest.mark.parametrize("accumulation", [0, 1])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", [3, 17, 40])
def test_listed_solvents_half_a_box_apart(n, axis, accumulation):
    """A 2 nm box, whose list radius of 1.2 nm is more than half of it: solvents on a lattice of 1/4 nm,
    each with listed neighbours at exactly 1 nm on an axis, and last entries there."""
    rng = np.random.default_rng(n)
    sites = np.stack(np.meshgrid(*[np.arange(0.125, 2.0, 0.5)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = np.roll(sites[np.sort(rng.permutation(len(sites))[:n])] + [[0.125, 0.0, 0.0]], axis, axis=-1)
    _check(ms.build(2.0, [], x), accumulation=accumulation)
