"""A batch whose member rebuilt its schedule refuses the next call, also where
the new tables lie at the old ones' addresses with the old ones' sizes."""
import numpy as np
import pytest

from test_gpu_angle_form import handle
from tycho2_amd.sweeper import (FP32, FP64, ORDER_CELL, ORDER_FACES,
                                SweepBatch, T2Error)

pytestmark = pytest.mark.gpu


def reorder(s):
    s.set_order(ORDER_CELL)
    s.set_order(ORDER_FACES)


def other_rule(s):
    s.set_dependency_tolerance(1e-10)


def other_rule_and_back(s):
    s.set_dependency_tolerance(1e-10)
    s.set_dependency_tolerance(-1.0)


@pytest.mark.parametrize("change", [reorder, other_rule, other_rule_and_back])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_rebuilt_member_is_refused(change, precision):
    print(f"stale batch {change.__name__} precision={precision}", flush=True)
    mem = [handle(4, 6, 2, precision, seed=3), handle(3, 4, 4, precision)]
    with SweepBatch(mem) as b:
        b.sweep_step()
        b.synchronize()
        change(mem[0])
        for call in (b.sweep_step, b.sweep_only, b.solve_krylov):
            with pytest.raises(T2Error) as e:
                call()
            assert e.value.code == -4 and "member 0" in str(e.value)
    with SweepBatch(mem) as b:       # a new batch takes the member as it is
        b.sweep_step()
        b.synchronize()
    assert all(np.isfinite(m.phi()).all() for m in mem)
    for m in mem:
        m.close()
