"""Device memory: whatever a handle needs besides the one-launch form's tables
comes before them, at creation and after it."""
import numpy as np
import pytest

from test_gpu_angle_form import handle
from tycho2_amd.sweeper import (FORM_STEPS, FP32, FP64, SweepBatch, T2Error,
                                set_alloc_fail)

pytestmark = pytest.mark.gpu


def created(nth, precision):
    """The form of a handle whose nth allocation fails, None without one."""
    set_alloc_fail(nth)
    try:
        with handle_without_source(precision) as s:
            set_alloc_fail(0)
            return s.form()
    except T2Error as e:
        assert e.code == -3
        return None
    finally:
        set_alloc_fail(0)


def handle_without_source(precision):
    from tycho2_amd import mesh as meshmod
    from tycho2_amd.quadrature import product_quadrature
    from tycho2_amd.sweeper import SweeperHIP
    sm = meshmod.kuhn_cube(3, 0.15, seed=3)
    omega, wt = product_quadrature(4)
    st = np.ones((sm.n_cells, 2))
    return SweeperHIP(sm, meshmod.tycho_connectivity(sm), omega, wt, 2, st,
                      0.5 * st, precision)


@pytest.mark.parametrize("precision", [FP64, FP32])
def test_tables_are_created_last(precision, monkeypatch):
    print(f"form tables last precision={precision}", flush=True)
    monkeypatch.setenv("T2_NO_GRAPH", "1")       # no tables
    need = 1
    while created(need, precision) is None:
        need += 1
    monkeypatch.delenv("T2_NO_GRAPH")
    forms = [created(nth, precision) for nth in range(1, need + 8)]
    assert forms[:need - 1] == [None] * (need - 1)
    assert forms[need - 1] == 0                  # tables' allocations
    assert None not in forms[need - 1:]
    assert forms[-1] > 0                         # none of them failed


@pytest.mark.parametrize("precision", [FP64, FP32])
def test_tables_make_room(precision):
    print(f"form tables make room precision={precision}", flush=True)

    def calls(s):
        s.sweep_step()
        yield s.phi()
        set_alloc_fail(arm)
        s.solve_krylov(100, 1e-6, 20)            # Krylov space
        yield s.phi()
        if precision == FP32:
            s.set_order(0)                       # the tables again
            s.set_order(1)
            set_alloc_fail(arm)
            s.solve_refined(100, 1e-5, 1e-4, 20)  # residual
            yield s.phi()
        yield s.psi()

    arm = 0
    with handle(5, 4, 4, precision) as s:
        s.set_form(FORM_STEPS)
        want = list(calls(s))
    arm = 1
    try:
        with handle(5, 4, 4, precision) as s:
            assert s.form() > 0
            got = list(calls(s))
            set_alloc_fail(0)
            assert s.form() == 0
            used = s.info()["device_bytes"]
            s.set_order(0)
            s.set_order(1)
            assert s.form() > 0
            assert s.info()["device_bytes"] > used
    finally:
        set_alloc_fail(0)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", [FP64, FP32])
def test_member_of_a_batch_makes_room(precision):
    print(f"form tables make room in a batch {precision}", flush=True)
    shapes = [(5, 4, 4), (4, 6, 2), (3, 4, 16)]

    def members():
        return [handle(n, sn, ng, precision) for n, sn, ng in shapes]

    mem = members()
    for m in mem:
        m.solve_krylov(100, 1e-6, 20)
    want = [m.phi() for m in mem]
    for m in mem:
        m.close()
    mem = members()
    with SweepBatch(mem) as b:
        b.sweep_step()
        b.synchronize()
        assert b.form() == 3
        set_alloc_fail(2)                        # the second member's space
        try:
            b.solve_krylov(100, 1e-6, 20)
        finally:
            set_alloc_fail(0)
        assert b.form() == 2 and mem[1].form() == 0
        assert all(np.array_equal(m.phi(), w) for m, w in zip(mem, want))
        b.sweep_step()                           # not refused
        b.synchronize()
    for m in mem:
        m.close()


def test_steps_give_the_tables_back():
    print("form tables given back", flush=True)
    with handle(5, 4, 4, FP64) as s:
        s.sweep_step()
        ref, full = s.phi(), s.info()["device_bytes"]
        items = s.nc * s.na
        for _ in range(2):
            s.set_form(FORM_STEPS)
            assert s.form() == 0
            assert s.info()["device_bytes"] <= full - 32 * items
            s.set_order(0)                       # none built either
            s.set_order(1)
            assert s.info()["device_bytes"] <= full - 32 * items
            s.set_phi(np.zeros_like(ref))
            s.sweep_step()
            assert np.array_equal(s.phi(), ref)
            s.set_form(0)
            assert s.form() > 0
            assert s.info()["device_bytes"] == full
            s.set_phi(np.zeros_like(ref))
            s.sweep_step()
            assert np.array_equal(s.phi(), ref)
