"""Step launches where the lanes of an item trade values for 16-byte accesses
(vertex rows of 8 to 32 bytes) and where they do not, bit for bit the ready
queue's one value per lane and access."""
import numpy as np
import pytest

from test_gpu_angle_form import handle, states
from tycho2_amd.sweeper import ENGINE_QUEUE, FP32, FP64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n,sn", [(1, 2), (5, 6), (6, 4)])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_equals_queue(n, sn, ng, precision, monkeypatch):
    print(f"step pieces n={n} sn={sn} ng={ng} {precision}", flush=True)
    with handle(n, sn, ng, precision) as s:
        s.set_engine(ENGINE_QUEUE)
        ref = states(s, precision)
    monkeypatch.setenv("T2_NO_GRAPH", "1")
    with handle(n, sn, ng, precision) as s:
        got = states(s, precision)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
