"""The level engine's one-block-per-angle form (live values in LDS slots)
against its step launches (T2_NO_GRAPH), bit for bit, at the sizes where the
form's rounds, slots and group chunks change."""
import numpy as np
import pytest

from tycho2_amd import mesh as meshmod
from tycho2_amd.quadrature import product_quadrature
from tycho2_amd.sweeper import FP32, FP64, SweepBatch, SweeperHIP

pytestmark = pytest.mark.gpu


def handle(n, sn, ng, precision, sigma="both", seed=5):
    sm = meshmod.kuhn_cube(n, 0.15, seed=seed)
    omega, wt = product_quadrature(sn)
    rng = np.random.default_rng(seed)
    cell = rng.uniform(0.5, 2.0, (sm.n_cells, 1))
    group = 1.0 + 0.1 * np.arange(ng)[None, :]
    st = np.broadcast_to({"cell": cell, "group": group,
                          "both": cell * group}[sigma], (sm.n_cells, ng))
    s = SweeperHIP(sm, meshmod.tycho_connectivity(sm), omega, wt, ng, st,
                   0.8 * st, precision)
    s.set_source_isotropic(rng.uniform(0.0, 1.0, (sm.n_cells, 4, ng)))
    return s


def states(s, precision):
    """psi after sweeps with an isotropic source, psi and phi after three
    source-iteration steps, and a refined solve's (FP32: the angle-dependent
    source in flux precision, swept in place)."""
    out = []
    for _ in range(3):
        s.sweep_step()
    out += [s.psi(), s.phi()]
    src = np.random.default_rng(9).uniform(0.0, 1.0, out[0].shape)
    if s.info()["n_lagged"] == 0 or precision == FP64:
        out.append(s.sweep(np.zeros_like(src), src).copy())
    if precision == FP32:
        s.solve_refined(100, 1e-5, 1e-4, 20)
        out += [s.psi(), s.phi()]
    return out


@pytest.mark.parametrize("n,sn,ng,sigma", [
    (1, 2, 1, "cell"),       # six cells: every level a part of one round
    (2, 4, 2, "group"),
    (5, 4, 1, "both"),       # one group: contiguous rows
    (6, 6, 1, "cell"),       # angles at 45 degrees: lagged faces
    (5, 6, 4, "both"),       # ... with group chunks
    (7, 8, 8, "group"),      # eight groups a block
    (6, 4, 16, "both"),      # several chunks of groups
    (3, 8, 64, "cell"),      # most groups
    (12, 8, 4, "both"),      # levels of several rounds
])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_equals_step_launches(n, sn, ng, sigma, precision, monkeypatch):
    print(f"angle form n={n} sn={sn} ng={ng} {sigma} {precision}", flush=True)
    with handle(n, sn, ng, precision, sigma) as s:
        got = states(s, precision)
    monkeypatch.setenv("T2_NO_GRAPH", "1")
    with handle(n, sn, ng, precision, sigma) as s:
        ref = states(s, precision)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)


@pytest.mark.parametrize("chains", [0, 1, 2])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_batch_of_both_forms(precision, chains):
    """Members swept with one block per angle beside members that only the
    merged step launches take (a priority schedule): each as by itself."""
    print(f"angle form batch precision={precision} chains={chains}",
          flush=True)
    shapes = [(3, 4, 1, False), (4, 4, 8, True), (5, 8, 2, False),
              (4, 2, 16, False), (3, 4, 8, True), (6, 4, 4, False)]

    def members():
        out = []
        for i, (n, sn, ng, steps) in enumerate(shapes):
            s = handle(n, sn, ng, precision, "both", seed=20 + i)
            if steps:
                s.set_priority(1, 0, 0)
            out.append(s)
        return out

    ref = []
    for s in members():
        with s:
            s.solve_krylov(200, 1e-9 if precision == FP64 else 1e-5, 20)
            s.sweep_step()
            got = [s.phi(), s.psi()]
            if precision == FP32:
                s.solve_refined(100, 1e-5, 1e-4, 20)
                got += [s.phi(), s.psi()]
            ref.append(got)
    mem = members()
    with SweepBatch(mem) as b:
        b.set_concurrent(chains)
        b.solve_krylov(200, 1e-9 if precision == FP64 else 1e-5, 20)
        b.sweep_step()
        b.synchronize()
        got = [[s.phi(), s.psi()] for s in mem]
        if precision == FP32:
            b.solve_refined(100, 1e-5, 1e-4, 20)
            for g, s in zip(got, mem):
                g += [s.phi(), s.psi()]
    for g, r in zip(got, ref):
        for a, c in zip(g, r):
            assert np.array_equal(a, c)
    for s in mem:
        s.close()


def test_levels_after_lagging(monkeypatch):
    """Angles at 45 degrees: the schedule levels the graph left after lagging
    (far fewer steps than the stalling traversal's levels), and step launches
    over it still give the oracle's sweep."""
    import oracle as orc
    from tycho2_amd.sweeper import mesh_geometry, sweep_levels
    print("levels after lagging", flush=True)
    monkeypatch.setenv("T2_NO_GRAPH", "1")
    sm = meshmod.kuhn_cube(6, 0.15, seed=7)
    conn = meshmod.tycho_connectivity(sm)
    omega, wt = product_quadrature(6)
    _, area, normal = mesh_geometry(sm, conn)
    levels, n_lag = sweep_levels(conn.adj_cell, area, normal, omega)
    rng = np.random.default_rng(3)
    st = rng.uniform(0.5, 2.0, (sm.n_cells, 2))
    src = rng.uniform(0.0, 1.0, (sm.n_cells, omega.shape[0], 4, 2))
    with SweeperHIP(sm, conn, omega, wt, 2, st, 0.5 * st, FP64) as s:
        assert s.info()["n_lagged"] == n_lag > 0
        assert s.info()["n_steps"] < (levels.max() + 1) // 2
        psi = s.sweep(np.zeros_like(src), src)
    ref, _ = orc.sweep(orc.build_mesh(sm), omega, 2, st, src)
    assert np.abs(psi - ref).max() <= 1e-12 * np.abs(ref).max()
