"""The form calls refuse bad arguments without a GPU."""
import ctypes

from tycho2_amd import sweeper


def test_null_handles():
    lib = sweeper.lib()
    n = ctypes.c_int()
    assert lib.t2_set_form(None, 0) == -1
    assert lib.t2_get_form(None, ctypes.byref(n)) == -1
    assert lib.t2_set_wait_limit(None, 0) == -1
    assert lib.t2_batch_set_form(None, 0) == -1
    assert lib.t2_batch_get_form(None, ctypes.byref(n)) == -1
    assert b"bad argument" in lib.t2_last_error()
