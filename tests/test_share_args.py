"""fr_share refuses a missing plan before any HIP call."""
from tomocupy_amd import _lib


def test_null_plan():
    assert _lib.lib().fr_share(None, 5) != 0
    assert 'plan is NULL' in _lib.last_error()
