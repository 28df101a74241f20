"""Which form a level-engine sweep takes: one launch with a block per angle,
or step launches, which every knob of theirs asks for."""
import numpy as np
import pytest

from test_gpu_angle_form import handle
from tycho2_amd import autotune
from tycho2_amd.sweeper import (ENGINE_LEVELS, ENGINE_QUEUE, FORM_AUTO,
                                FORM_STEPS, FP32, FP64, T2Error)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sn,ng,gc64,gc32", [
    (1, 2, 1, 1, 1),
    (2, 4, 2, 1, 1),         # more blocks rather than whole rows
    (5, 4, 1, 1, 1),
    (6, 6, 1, 1, 1),         # lagged faces
    (5, 6, 4, 2, 2),         # ... with group chunks
    (7, 8, 8, 8, 8),         # eight groups a block
    (6, 4, 16, 4, 4),        # four chunks of groups
    (3, 8, 64, 8, 8),        # most groups
    (12, 8, 4, 4, 4),        # levels of several rounds
    (1, 2, 4, 1, 2),
    (9, 8, 16, 8, 8),
    (14, 6, 8, 4, 4),
    (16, 8, 4, 4, 4),
    (23, 4, 16, None, 4),    # sixteen-byte parts of a row
    (23, 8, 16, 0, None),    # the step launches are taken to be faster
])
def test_groups_per_block(n, sn, ng, gc64, gc32):
    """The shapes at which the one launch is compared with step launches."""
    print(f"form n={n} sn={sn} ng={ng}", flush=True)
    for precision, want in ((FP64, gc64), (FP32, gc32)):
        if want is not None:
            with handle(n, sn, ng, precision) as s:
                assert s.form() == want


def test_knobs_of_step_launches_ask_for_them(monkeypatch):
    print("form knobs", flush=True)
    ng = 16
    with handle(4, 4, ng, FP64) as s:
        assert s.form() > 0
        for items in (4, 8, 16):             # 64, 128 and 256 threads
            s.set_form(FORM_AUTO)
            assert s.form() > 0
            s.set_launch(items, 1)
            assert s.form() == 0
        s.set_launch(0, 1)                   # keeps what is set
        assert s.form() == 0
        s.set_form(FORM_AUTO)
        for on, off in ((lambda: s.set_launch(0, 2), lambda: s.set_launch(0, 1)),
                        (lambda: s.set_items_per_lane(2),
                         lambda: s.set_items_per_lane(1)),
                        (lambda: s.set_schedule(2), lambda: s.set_schedule(1)),
                        (lambda: s.set_concurrent_batches(True),
                         lambda: s.set_concurrent_batches(False)),
                        (lambda: s.set_priority(1, 0, 0),
                         lambda: s.set_priority(-1)),
                        (lambda: s.set_engine(ENGINE_QUEUE),
                         lambda: s.set_engine(ENGINE_LEVELS)),
                        (lambda: s.set_form(FORM_STEPS),
                         lambda: s.set_form(FORM_AUTO))):
            on()
            assert s.form() == 0
            off()
            assert s.form() > 0
        with pytest.raises(T2Error):
            s.set_form(2)
    monkeypatch.setenv("T2_NO_GRAPH", "1")
    with handle(4, 4, ng, FP64) as s:
        assert s.form() == 0


@pytest.mark.parametrize("n,sn,ng", [(4, 4, 16), (6, 6, 4), (5, 8, 1)])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_step_graph_equals_one_launch(n, sn, ng, precision):
    """Replays of the captured step launches at each block size."""
    print(f"step graph n={n} sn={sn} ng={ng} {precision}", flush=True)
    with handle(n, sn, ng, precision) as s:
        assert s.form() > 0
        for _ in range(3):
            s.sweep_step()
        ref = s.phi(), s.psi()
    for block in (64, 128, 256):
        with handle(n, sn, ng, precision) as s:
            s.set_launch(block // ng, 1)
            assert s.form() == 0
            for _ in range(3):
                s.sweep_step()
            assert np.array_equal(s.phi(), ref[0])
            assert np.array_equal(s.psi(), ref[1])


def test_tuner_times_both_forms():
    print("tuner, both forms", flush=True)
    with handle(4, 4, 4, FP64) as s:
        best, trials = autotune.tune(s, reps=1, batches=(1,),
                                     engines=(ENGINE_LEVELS,))
        assert [t["one_launch"] for t in trials].count(True) == 1
        assert {t["block"] for t in trials if not t["one_launch"]} == \
            set(autotune.BLOCKS)
        assert best == min(trials, key=lambda t: t["ms"])
        assert (s.form() > 0) == best["one_launch"]
