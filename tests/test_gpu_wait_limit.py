"""A wait of the one-launch form that runs out is reported: with a poll limit
of 1 some wait of every sweep does, each kernel still runs to its end, and
later sweeps are exact again."""
import numpy as np
import pytest

from test_gpu_angle_form import handle
from tycho2_amd.sweeper import (ERR_TIMEOUT, FORM_STEPS, FP32, FP64,
                                SweepBatch, T2Error)

pytestmark = pytest.mark.gpu


def timeouts(calls):
    n = 0
    for call in calls:
        try:
            call()
        except T2Error as e:
            assert e.code == ERR_TIMEOUT and "one-launch" in str(e)
            n += 1
    return n


@pytest.mark.parametrize("ng", [1, 4])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_handle_reports_abandoned_sweeps(precision, ng):
    print(f"wait limit ng={ng} precision={precision}", flush=True)
    with handle(8, 4, ng, precision) as s:
        s.sweep_step()
        ref = s.phi(), s.psi()
        phi0 = np.zeros_like(ref[0])

        def swept_then(read):
            def call():
                s.sweep_only()
                read()
            return call

        s.set_wait_limit(1)
        assert s.form() > 0
        calls = [swept_then(s.synchronize), swept_then(s.phi),
                 swept_then(s.psi), swept_then(lambda: s.psi_angle(0)),
                 lambda: s.solve_source_iteration(3, 1e-12),
                 lambda: s.solve_krylov(3, 1e-12, 3)]
        assert timeouts(calls * 2) == 2 * len(calls)
        s.synchronize()                  # reported once
        s.set_wait_limit(0)
        s.set_phi(phi0)
        s.sweep_step()
        s.synchronize()
        # (lagged faces none: a sweep does not read the former psi)
        assert np.array_equal(s.phi(), ref[0])
        assert np.array_equal(s.psi(), ref[1])
        s.set_wait_limit(1)              # of no meaning to step launches
        s.set_form(FORM_STEPS)
        s.set_phi(phi0)
        s.sweep_step()
        s.synchronize()
        assert np.array_equal(s.phi(), ref[0])
        with pytest.raises(T2Error):
            s.set_wait_limit(-1)


@pytest.mark.parametrize("precision", [FP64, FP32])
def test_batch_reports_abandoned_sweeps(precision):
    print(f"wait limit, batch precision={precision}", flush=True)
    shapes = [(6, 4, 1), (8, 4, 4), (7, 2, 16)]
    mem = [handle(n, sn, ng, precision) for n, sn, ng in shapes]
    for m in mem:
        m.sweep_step()
    ref = [m.phi() for m in mem]
    for m in mem:
        m.set_phi(np.zeros_like(m.phi()))
    with SweepBatch(mem) as b:
        b.sweep_step()
        b.synchronize()
        for m, r in zip(mem, ref):
            assert np.array_equal(m.phi(), r)
        mem[1].set_wait_limit(1)

        def swept():
            b.sweep_only()
            b.synchronize()

        calls = [swept, lambda: b.solve_source_iteration(3, 1e-12),
                 lambda: b.solve_krylov(3, 1e-12, 3)]
        assert timeouts(calls * 2) == 2 * len(calls)
        b.synchronize()
        mem[1].set_wait_limit(0)
        for m, r in zip(mem, ref):
            m.set_phi(np.zeros_like(r))
        b.sweep_step()
        b.synchronize()
        for m, r in zip(mem, ref):
            assert np.array_equal(m.phi(), r)
    for m in mem:
        m.close()
