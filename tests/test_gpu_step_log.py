"""lima_step_logged's data log against its definition, term by term."""
import ctypes as C

import numpy as np
import pytest

from quantom_amd.abi import RunParams

pytestmark = pytest.mark.gpu


def _repeat_terms(s, kind, times):
    """Every compound's terms of one kind `times` over, each repeat's force constant 10% larger."""
    arr, off = getattr(s, kind + "s"), getattr(s, kind + "_offset")
    key = "k_phi" if kind == "dihedral" else "k_theta"
    parts = []
    for c in range(s.n_compounds):
        for k in range(times):
            t = arr[off[c]:off[c + 1]].copy()
            t[key] *= np.float32(1.0 + 0.1 * k)
            parts.append(t)
    setattr(s, kind + "s", np.concatenate(parts))
    setattr(s, kind + "_offset", (off * times).astype(np.int32))


def _energy(s, kind, t):
    """The oracle's FP32 energy of term t of compound 0 at the initial positions."""
    from oracle.oracle import lib
    fp = lambda v: np.ascontiguousarray(v, np.float32).ctypes.data_as(C.POINTER(C.c_float))
    x = [fp(p) for p in s.chain_positions[:s.compound_offset[1]]]
    out, e = np.zeros(12, np.float32), C.c_double(0.0)
    o = out.ctypes.data_as(C.POINTER(C.c_float))
    d = {"dihedral": s.dihedrals, "angle": s.angles, "bond": s.bonds}[kind][t]
    i = [x[int(k)] for k in d["idx"]]
    if kind == "dihedral":
        lib().oracle_dihedral_f32(*i, C.c_float(d["phi_0"]), C.c_float(d["k_phi"]), int(d["n"]), o, C.byref(e))
    elif kind == "angle":
        lib().oracle_anglebond_f32(*i, C.c_float(d["theta_0"]), C.c_float(d["k_theta"]), o, C.byref(e))
    else:
        lib().oracle_pairbond_f32(*i, C.c_float(d["b0"]), C.c_float(d["kb"]), o, C.byref(e))
    return e.value


# (particles of a compound, repeats): terms of a kind past a wavefront's 64 and within the reference's
# 128 threads, in a compound that fits a wavefront and in one that does not
@pytest.mark.parametrize("csize,times", [(16, 1), (48, 2), (64, 2), (70, 1)])
@pytest.mark.parametrize("kind", ["dihedral", "angle"])
def test_potential_slot_is_thread_0s_terms(kind, csize, times):
    """Thread 0's potE slot: the first dihedral, or without dihedrals the first bond and angle, whatever
    the number of terms and the threads that this engine gives a compound.  The bar is that of the FP32
    term against the oracle's (cosf and acosf differ by ulps): 1e-4 of it."""
    from quantom_amd import systems
    from quantom_amd.engine import Engine
    s = systems.build_system(0x51A7 + csize, 1, 2, 4.6, 4, 200, compound_size=csize, central_first=True)
    # off the equilibrium that the generator builds at
    s.chain_positions += np.random.default_rng(csize).uniform(-4e-3, 4e-3, s.chain_positions.shape).astype(np.float32)
    _repeat_terms(s, kind, times)
    n = np.diff(getattr(s, kind + "_offset"))[0]
    assert times == 1 or 64 < n <= 128
    e = Engine([s], RunParams(nlist_interval=10, enable_dihedrals=1 if kind == "dihedral" else 0))
    log, _ = e.step_logged(1, 0, 128)
    e.close()
    want = _energy(s, "dihedral", 0) if kind == "dihedral" else _energy(s, "bond", 0) + _energy(s, "angle", 0)
    extra = _energy(s, kind, 64) if n > 64 else 0.0
    assert n <= 64 or abs(extra) > 1e-3 * abs(want)     # a sum with term 64 would be seen
    assert abs(log[0, 2] - want) <= 1e-4 * abs(want), (log[0, 2], want, extra)


def test_force_magnitude_is_correctly_rounded(small_system):
    """|F| of the log (Float3::len) is the correctly rounded root of the FP32 sum of squares, as the
    reference's sqrtf and the oracle's are: bit for bit over 64 steps."""
    from quantom_amd.engine import Engine
    p = RunParams(nlist_interval=10)
    a, b = Engine([small_system], p), Engine([small_system], p)
    log, _ = a.step_logged(64, 0, 128, train=False)
    want = []
    for _ in range(64):
        b.step(1)
        f = b.forces()[0][0]
        q = f * f                                        # float32, each operation rounded
        want.append(np.sqrt((q[0] + q[1]) + q[2]))
    a.close()
    b.close()
    assert np.array_equal(log[:, 3], np.array(want, np.float32))
