"""The force launch's roles and the adjoint's against the oracle at the sizes where their splits change,
each case a condition.  Forces: the bar of the force parity tests, 1e-5 of the FP32 oracle's (both sides
are FP32 sums of the same pairs).  Gradients: one frame, whose positions are the given ones, so that
no rounding of a trajectory enters, against differences of the FP64 oracle's loss."""
import numpy as np
import pytest

from quantom_amd.abi import THERMOSTAT_NONE, RunParams
from tests import microsystems as ms
from tests import test_gpu_adjoint_roles as roles
from tests.conftest import rel_rms
from tests.test_adjoint import base_params, with_params
from tests.test_gpu_step_roles import _system

pytestmark = pytest.mark.gpu


def _compare(s, p, lists=False):
    """Forces of an engine and of the FP32 oracle; with `lists` the engine walks the oracle's lists in
    their order, which matters where one image is not enough."""
    from oracle.oracle import KIND_CC, KIND_CS, KIND_SS, Oracle
    from quantom_amd.engine import Engine
    o = Oracle(s, p, precision=32)
    want = o.compute_forces()
    assert want[2] == 0
    e = Engine([s], p)
    if lists:
        e.set_neighbors(cc=o.neighbors(KIND_CC), cs=o.neighbors(KIND_CS), ss=o.neighbors(KIND_SS))
    got = e.compute_forces()
    e.close()
    assert rel_rms(got[0], want[0]) <= 1e-5 and rel_rms(got[1], want[1]) <= 1e-5


@pytest.mark.parametrize("accumulation", [0, 1])
@pytest.mark.parametrize("csize", [12, 16, 17, 20, 31, 32, 33, 64, 65, 100, 128])
def test_each_compound_size(csize, accumulation):
    _compare(_system(csize, csize % 3, 500 + 37 * (csize % 7)), RunParams(accumulation=accumulation))


@pytest.mark.parametrize("accumulation", [0, 1])
@pytest.mark.parametrize("csize", [13, 16, 31, 65, 128])
def test_compounds_a_whole_box_away(csize, accumulation):
    """Stored one box below and above: an image moves by one box at a time, so a solvent two boxes from
    an entry reaches it over several, and its forces depend on the lists' order."""
    from quantom_amd import systems
    s = systems.build_system(0x51A7 + csize, 1, 3, 6.0, 4, 1200, compound_size=csize, central_first=True, confine=1.2)
    off = s.compound_offset
    s.chain_positions[off[0]:off[1]] -= np.float32(s.box_len)
    s.chain_positions[off[2]:off[3], 1] += np.float32(s.box_len)
    _compare(s, RunParams(accumulation=accumulation), lists=True)


@pytest.mark.parametrize("accumulation", [0, 1])
@pytest.mark.parametrize("n_solvents", [1, 2, 15, 63, 257, 1500])
def test_solvents_alone(n_solvents, accumulation):
    """Solvent-solvent forces and energy without compounds, rows below and above a quad's 16 entries.
    The energy is an FP64 sum of FP32 pair energies: 1e-5 of the FP64 oracle's."""
    from oracle.oracle import Oracle
    from quantom_amd import systems
    from quantom_amd.engine import Engine
    s = systems.build_system(0x50 + n_solvents, 0, 1, 4.0, 3, n_solvents)
    p = RunParams(accumulation=accumulation)
    _compare(s, p)
    e, o = Engine([s], p), Oracle(s, p, precision=64)
    o.compute_forces()
    got, want = e.energies()[0]["lj_solvent_solvent"], o.energies()["lj_solvent_solvent"]
    e.close()
    assert abs(got - want) <= 1e-5 * abs(want)


def test_solvent_blocks_of_a_tile_give_each_systems_forces():
    """Over 65,536 solvents the list role takes a tile of 256 a block instead of 64: bit-equal."""
    from quantom_amd.engine import Engine
    kinds = [_system(16, 3, n, compounds=2, box=5.0) for n in (1500, 257, 700)]
    batch = Engine([kinds[k % 3] for k in range(90)], RunParams())
    sim = batch.simulation
    assert sim.n_solvents > 65536
    f = batch.compute_forces()
    for r in (0, 1, 2, 44, 87, 88, 89):
        alone = Engine([kinds[r % 3]], RunParams())
        a = alone.compute_forces()
        alone.close()
        assert np.array_equal(a[0], f[0][sim.chain_begin[r]:sim.chain_begin[r + 1]]), r
        assert np.array_equal(a[1], f[1][sim.solvent_begin[r]:sim.solvent_begin[r + 1]]), r
    batch.close()


@pytest.mark.parametrize("ulps", [-2, -1, 0, 1, 2])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("side", [-1, 1])
def test_image_flag_at_half_a_box(side, axis, ulps):
    """A compound's particle 0, and a listed solvent in a 2 nm box, half a box and a few floats from a
    solvent on either side: beyond half a box the other image is taken, at it and below the stored one."""
    def at(m, L):
        x = np.float32(m + side * L / 2)
        for _ in range(abs(ulps)):
            x = np.nextafter(x, np.float32(x + side * np.sign(ulps)))
        return float(x)
    roll = lambda p: np.roll(np.asarray(p, np.float32), axis, axis=-1)
    m = 1.0 if side > 0 else 3.0
    p0 = at(m, 4.0)
    s = ms.build(4.0, [(roll([(p0, 1.0, 1.0), (p0 + 0.875 * side, 1.0, 1.0)]), [1, 1])], roll([(m, 1.5, 1.0), (m, 1.0, 3.0)]),
                 ignores={(0, 0): [(0, 1)], (0, 1): [(0, 0)]})
    _compare(s, RunParams(nlist_interval=0), lists=True)
    m = 0.5 if side > 0 else 1.5
    s = ms.build(2.0, [], roll([(m, 1.0, 1.0), (at(m, 2.0), 1.25, 1.0)]))
    _compare(s, RunParams(nlist_interval=0), lists=True)


#        chains, compounds a chain, particles, solvents, box, stored across the edge
GRADIENT_CASES = [(1, 3, 16, 63, 3.2, False), (1, 2, 17, 257, 3.2, False), (2, 2, 33, 300, 3.8, False), (1, 2, 65, 130, 4.2, False),
                  (1, 2, 128, 517, 4.6, False), (1, 2, 33, 300, 3.8, True)]


@pytest.mark.parametrize("case", GRADIENT_CASES)
def test_gradient_of_one_frame(case):
    """Every parameter: 2e-3 of the difference and 1e-4 of the largest, the bar of the gradient tests.
    Bonds are off their length, where their FP32 forces have relative accuracy."""
    from oracle.oracle import Oracle
    from quantom_amd.engine import Engine
    s = roles._system(*case)
    rng = np.random.default_rng(case[2])
    s.chain_positions += rng.uniform(-4e-3, 4e-3, s.chain_positions.shape).astype(np.float32)
    p = RunParams(nlist_interval=10, thermostat=THERMOSTAT_NONE)

    def frame(system):
        o = Oracle(system, p, precision=64)
        fc, fs, st = o.compute_forces()
        assert st == 0
        return fc, fs, o.energies()["potential"]

    fc, fs, pot = frame(s)
    fct = (fc * (1 + 0.05 * rng.uniform(-1, 1, fc.shape))).astype(np.float32)
    fst = (fs * (1 + 0.05 * rng.uniform(-1, 1, fs.shape))).astype(np.float32)
    et = pot * 1.03
    alpha, beta = 1.0 / (pot - et) ** 2, 1.0 / float(((fc - fct) ** 2).sum() + ((fs - fst) ** 2).sum())
    e = Engine([s], p)
    _, grad = e.adjoint(1, [alpha], [beta], np.array([[et]]), fct[None], fst[None])
    e.close()
    v0 = base_params(s)

    def loss(i, x):
        v = v0.copy()
        v[i] = x
        c, w, u = frame(with_params(s, v))
        return float(alpha * (u - et) ** 2 + beta * (((c - fct) ** 2).sum() + ((w - fst) ** 2).sum()))

    fd = {}
    for i in [0, 1, 2, 32, 33, 34, 64, 65, 66, 67]:
        h = 1e-4 * max(abs(v0[i]), 1e-3)
        lo, hi = np.float32(v0[i] - h), np.float32(v0[i] + h)
        fd[i] = (loss(i, hi) - loss(i, lo)) / (float(hi) - float(lo))
    scale = max(abs(d) for d in fd.values())
    for i, d in fd.items():
        print(f"case {case} parameter {i}: {grad[0][i]:.6e} {d:.6e}", flush=True)
        assert abs(grad[0][i] - d) <= 2e-3 * abs(d) + 1e-4 * scale, (i, grad[0][i], d)
