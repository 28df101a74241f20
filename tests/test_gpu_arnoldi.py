"""The device Arnoldi step at the vector counts where its kernels change (8
and 16 vectors in registers, more from memory): GMRES iteration by iteration
against a textbook GMRES on the same operator applied on the device."""
import numpy as np
import pytest

from tycho2_amd import mesh as meshmod
from tycho2_amd.quadrature import product_quadrature
from tycho2_amd.sweeper import FP64, NoConvergence, SweeperHIP

pytestmark = pytest.mark.gpu


def textbook(apply, b, steps):
    """Relative residuals and the iterate of `steps` GMRES iterations."""
    V, H, hist = [b / np.linalg.norm(b)], np.zeros((steps + 1, steps)), []
    e = np.zeros(steps + 1)
    e[0] = np.linalg.norm(b)
    for j in range(steps):
        w = apply(V[j])
        for _ in range(2):
            h = np.array([v @ w for v in V])
            H[:j + 1, j] += h
            w = w - sum(hi * v for hi, v in zip(h, V))
        H[j + 1, j] = np.linalg.norm(w)
        y, *_ = np.linalg.lstsq(H[:j + 2, :j + 1], e[:j + 2], rcond=None)
        hist.append(np.linalg.norm(H[:j + 2, :j + 1] @ y - e[:j + 2]) / e[0])
        V.append(w / H[j + 1, j])
    return np.array(hist), sum(yi * v for yi, v in zip(y, V))


@pytest.mark.parametrize("n,ng", [(1, 1), (4, 2), (7, 4)])
def test_history_and_iterate(n, ng):
    steps = 22            # past 8 and 16 vectors in one cycle
    print(f"arnoldi n={n} ng={ng}", flush=True)
    sm = meshmod.kuhn_cube(n, 0.15, seed=2)
    omega, wt = product_quadrature(4)
    rng = np.random.default_rng(4)
    st = rng.uniform(2.0, 40.0, (sm.n_cells, ng))
    q = rng.uniform(0.0, 1.0, (sm.n_cells, 4, ng))
    with SweeperHIP(sm, meshmod.tycho_connectivity(sm), omega, wt, ng, st,
                    0.999 * st, FP64) as s:
        s.set_source_isotropic(q)
        b = s.krylov_rhs().ravel()
        shape = q.shape
        hist, x = textbook(
            lambda v: s.krylov_apply(v.reshape(shape)).ravel(), b, steps)
        try:
            got = s.solve_krylov(steps, 1e-13, 40)
        except NoConvergence as e:
            got = e.result
        phi = s.phi().ravel()
    k = len(got)
    assert k == steps or got[-1] <= 1e-13
    # residuals to round-off of the right-hand side, the iterate to the
    # conditioning of the projected system
    assert np.abs(got - hist[:k]).max() <= 1e-11
    assert np.linalg.norm(phi - x) <= 1e-8 * np.linalg.norm(x)
