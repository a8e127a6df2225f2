"""State and forces through the pinned buffer (one system) and straight to the caller's arrays (a batch
over its 4 MB): what is set is what is read, array by array, and leaves types, order and the arrays
that were not given alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 60])
def test_state_round_trip(small_system, count):
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    e = Engine([small_system] * count, RunParams(nlist_interval=0))
    first = e.get_state()
    assert sum(x.nbytes for x in first) > 4 << 20 or count == 1
    forces = [x.copy() for x in e.compute_forces()]
    rng = np.random.default_rng(3)
    new = [(x + rng.uniform(0, 1e-3, x.shape)).astype(np.float32) for x in first]
    for k in range(4):
        args = [None] * 4
        args[k] = new[k]
        e.set_state(*args)
        got = e.get_state()
        for j in range(4):
            assert np.array_equal(got[j], new[j] if j <= k else first[j]), (k, j)
    e.set_state(*first)
    for a, b in zip(e.compute_forces(), forces):    # types and replica marks as before
        assert np.array_equal(a, b)
    for a, b in zip(e.forces(), forces):
        assert np.array_equal(a, b)
    e.close()


def test_large_unpinned_forces_equal_the_small_ones(small_system):
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine
    one, many = Engine([small_system], RunParams()), Engine([small_system] * 120, RunParams())
    (c1, s1), (c, s) = one.compute_forces(), many.compute_forces()
    assert c.nbytes + s.nbytes > 4 << 20
    for r in (0, 59, 119):
        assert np.array_equal(c[r * len(c1):(r + 1) * len(c1)], c1) and np.array_equal(s[r * len(s1):(r + 1) * len(s1)], s1)
    one.close()
    many.close()


def test_state_and_forces_take_no_device_memory(small_system):
    """Reading and setting the state, and forces, work where nothing is left on the device: the first
    call allocates nothing there."""
    import ctypes as C

    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine, load_library
    load_library()
    hip = C.CDLL("libamdhip64.so.7")        # the runtime that the library has loaded

    def free():
        n, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(n), C.byref(total)) == 0
        return n.value

    e = Engine([small_system] * 120, RunParams(nlist_interval=0))
    e.compute_forces()                      # code and pinned buffers loaded
    f = Engine([small_system] * 120, RunParams(nlist_interval=0))
    before = free()
    state = f.get_state()
    f.set_state(*state)
    f.compute_forces()
    assert free() == before
    e.close()
    f.close()


def test_small_engines_keep_small_transfer_buffers(small_system):
    """32 engines of 78 KB of state each: their first reading of it takes less than 1 MB of the
    process's address space an engine (pinned memory is mapped into it)."""
    from quantom_amd.abi import RunParams
    from quantom_amd.engine import Engine

    def mapped():
        with open("/proc/self/status") as f:
            return next(int(line.split()[1]) for line in f if line.startswith("VmSize"))

    first = Engine([small_system], RunParams())
    first.get_state()
    engines = [Engine([small_system], RunParams()) for _ in range(32)]
    before = mapped()
    for e in engines:
        e.get_state()
    grown = mapped() - before
    assert grown < 32 * 1024, grown
    for e in engines + [first]:
        e.close()
