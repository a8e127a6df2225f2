"""The gradient by epsilon of a type whose epsilon is far below the solvent's.  Its geometric credit is
divided by 2 epsilon, so an error of the arithmetic sites must not enter it.

One compound among solvents and one frame, so that the gradient has a closed form: the loss is
sum |F|^2, the forces F are the FP64 oracle's, and dF / d eps follows from each site's own force
(arithmetic: a solvent's from every particle; geometric: a particle's from its listed solvents).
Bar: a force parity of 1e-5 on F and on dF, summed without cancellation."""
import numpy as np
import pytest

from quantom_amd.abi import THERMOSTAT_NONE, RunParams
from tests import microsystems as ms

pytestmark = pytest.mark.gpu


def _lj(d, sigma, e24):
    """Force along d = x_other - x for 24 eps = e24 (calcLJForce's direction and sign)."""
    q = (d ** 2).sum(-1, keepdims=True)
    s6 = (sigma ** 2 / q) ** 3
    return e24 / q * s6 * (1.0 - 2.0 * s6) * d


def _system(ratio, listed, n=17):
    rng = np.random.default_rng(7)
    c = np.array([2.0, 2.0, 2.0]) + rng.uniform(-0.25, 0.25, (n, 3))
    g = np.stack(np.meshgrid(*[np.arange(0.4, 8.0, 0.8)] * 3, indexing="ij"), -1).reshape(-1, 3)
    sol = g + rng.uniform(-0.05, 0.05, g.shape)
    d = np.linalg.norm(sol - 2.0, axis=1)
    sol = sol[(d > 0.75) & (d < 3.9)] if listed else sol[(d > 2.6) & (d < 3.9)]
    every = {(0, i): [(0, j) for j in range(n) if j != i] for i in range(n)}   # no intra-compound pairs
    s = ms.build(8.0, [(c, [1] * n)], sol, ignores=every)
    ff = s.forcefield.copy()
    ff[1, 2] = np.float32(ratio) * ff[0, 2]
    s.forcefield = ff
    return s


@pytest.mark.parametrize("listed", [True, False])
@pytest.mark.parametrize("ratio", [1.0, 1e-2, 1e-4, 1e-6])
def test_gradient_by_a_small_epsilon(ratio, listed):
    from oracle.oracle import KIND_CS, Oracle
    from quantom_amd.engine import Engine
    s = _system(ratio, listed)
    p = RunParams(nlist_interval=10, thermostat=THERMOSTAT_NONE, cutoff=0.5)
    o = Oracle(s, p, precision=64)
    fc, fs, st = o.compute_forces()
    assert st == 0
    near = o.neighbors(KIND_CS)[0]
    assert (len(near) > 0) == listed
    scale = 1.0 / float((fc ** 2).sum() + (fs ** 2).sum())
    e = Engine([s], p)
    _, grad = e.adjoint(1, None, [scale])
    e.close()
    x, y = s.chain_positions.astype(float), s.solvent_positions.astype(float)
    sig0, eps0 = float(s.forcefield[0, 1]), float(s.forcefield[0, 2])
    sig1, eps1 = float(s.forcefield[1, 1]), float(s.forcefield[1, 2])
    sigma = 0.5 * (sig0 + sig1)
    dfs = _lj(x[None, :, :] - y[:, None, :], sigma, 12.0).sum(1)             # 24 (eps0 + eps1) / 2
    dfc = np.zeros_like(fc)
    if listed:
        dfc = _lj(y[None, near, :] - x[:, None, :], sigma, 12.0 * np.sqrt(eps0 / eps1)).sum(1)
    want = 2.0 * scale * ((fs * dfs).sum() + (fc * dfc).sum())
    size = lambda f: np.linalg.norm(f, axis=1)
    bar = 2e-5 * 2.0 * scale * ((size(fs) * size(dfs)).sum() + (size(fc) * size(dfc)).sum())
    print(f"case {ratio} {listed}: {grad[0][33]:.9e} {want:.9e} error {abs(grad[0][33] - want):.1e} bar {bar:.1e}", flush=True)
    assert abs(grad[0][33] - want) <= bar
