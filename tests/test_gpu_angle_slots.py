"""The one-block-per-angle form where a cell takes over the slot of the one
it alone reads last, and where the form is chosen for rows in several parts of
two or more groups: bit for bit the step launches (T2_NO_GRAPH)."""
import numpy as np
import pytest

from test_gpu_angle_form import handle, states
from tycho2_amd.sweeper import FP32, FP64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sn,ng,precision", [
    (1, 2, 4, FP64),        # readers in one level only
    (9, 8, 16, FP32),       # wide levels, sixteen-byte parts
    (14, 6, 8, FP32),       # lagged faces beside handed-on slots
    (16, 8, 4, FP64),       # two parts a row
    (23, 4, 16, FP32),      # four parts a row: the rule's wider side
])
def test_equals_step_launches(n, sn, ng, precision, monkeypatch):
    print(f"slots n={n} sn={sn} ng={ng} {precision}", flush=True)
    with handle(n, sn, ng, precision) as s:
        got = states(s, precision)
    monkeypatch.setenv("T2_NO_GRAPH", "1")
    with handle(n, sn, ng, precision) as s:
        ref = states(s, precision)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
