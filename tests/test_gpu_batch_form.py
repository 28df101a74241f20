"""Which members a batch's level form sweeps with one block per angle, and the
merged steps of the same members when a block size or a member asks for them:
each as by itself, bit for bit."""
import numpy as np
import pytest

from test_gpu_angle_form import handle
from tycho2_amd import autotune
from tycho2_amd.sweeper import (ENGINE_LEVELS, ENGINE_QUEUE, FORM_AUTO,
                                FORM_STEPS, FP32, FP64, SweepBatch, T2Error)

pytestmark = pytest.mark.gpu

SHAPES = [(3, 4, 1), (4, 4, 8), (5, 6, 8), (4, 2, 16)]


def members(precision, form=FORM_AUTO):
    out = [handle(n, sn, ng, precision, seed=30 + i)
           for i, (n, sn, ng) in enumerate(SHAPES)]
    for m in out:
        m.set_form(form)
    return out


def close(mem):
    for m in mem:
        m.close()


@pytest.fixture(scope="module", params=[FP64, FP32])
def alone(request):
    """Each member's own solve and step, in step launches."""
    mem = members(request.param, FORM_STEPS)
    want = []
    for m in mem:
        m.solve_krylov(200, 1e-6, 20)
        m.sweep_step()
        want.append((m.phi(), m.psi()))
    close(mem)
    return request.param, want


def same(b, mem, want):
    b.solve_krylov(200, 1e-6, 20)
    b.sweep_step()
    b.synchronize()
    for m, (phi, psi) in zip(mem, want):
        assert np.array_equal(m.phi(), phi)
        assert np.array_equal(m.psi(), psi)


@pytest.mark.parametrize("block,chains", [(64, 0), (128, 1), (256, 0),
                                          (256, 2)])
def test_block_size_asks_for_merged_steps(alone, block, chains):
    precision, want = alone
    print(f"batch form block={block} chains={chains} precision={precision}",
          flush=True)
    mem = members(precision)
    with SweepBatch(mem) as b:
        assert b.form() == len(SHAPES)
        b.set_concurrent(chains)
        b.set_launch(block)
        assert b.form() == 0
        same(b, mem, want)
        b.set_form(FORM_AUTO)        # the tables are built anew
        assert b.form() == len(SHAPES)
        same(b, mem, want)
        b.set_engine(ENGINE_QUEUE, 1 << 20)
        assert b.form() == 0
    close(mem)


def test_members_knobs_count(alone, monkeypatch):
    precision, want = alone
    print(f"batch form, members' knobs precision={precision}", flush=True)
    mem = members(precision)
    with SweepBatch(mem) as b:
        same(b, mem, want)
        mem[1].set_launch(64 // mem[1].ng, 1)
        mem[3].set_items_per_lane(2)
        mem[2].set_engine(ENGINE_QUEUE)     # of its own sweeps only
        assert b.form() == 2
        same(b, mem, want)
        mem[1].set_form(FORM_AUTO)
        assert b.form() == 3
        same(b, mem, want)
    close(mem)
    monkeypatch.setenv("T2_NO_GRAPH", "1")
    mem = members(precision)
    with SweepBatch(mem) as b:
        assert b.form() == 0
        same(b, mem, want)
        with pytest.raises(T2Error):
            b.set_form(2)
    close(mem)


def test_tuner_times_both_forms():
    print("batch tuner, both forms", flush=True)
    mem = members(FP64)
    with SweepBatch(mem) as b:
        best, trials = autotune.tune_batch(b, reps=1)
        level = [t for t in trials if t["engine"] == ENGINE_LEVELS]
        assert [t["by_angle"] for t in level].count(len(SHAPES)) == 1
        assert {t["block"] for t in level if not t["by_angle"]} == \
            set(autotune.BLOCKS)
        assert b.form() == best["by_angle"]
    close(mem)
