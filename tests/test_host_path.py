"""The calls' way through cuv_amd/dia.py, the Python module and the library's dispatch, on a runtime without a GPU
(tests/cxx/fake_hip.c), so that waits and launches can fail and calls can be held where they are."""
import _fake_hip


def test_a_wait_that_cannot_begin_leaves_the_call_undone(tmp_path):
    _fake_hip.run(tmp_path, """
A, x, y = matrix(64, 64, [-1, 0, 1]), tensor(4, 64), tensor(4, 64)
flag("fake_fail_event_create", 1)
assert D._native.product(y, A, x, "n", 1.0, 0.0, None, 0, 0, True) is False and flag("fake_launches") == 0
flag("fake_fail_event_create", 0)
assert D._native.product(y, A, x, "n", 1.0, 0.0, None, 0, 0, True) is True and flag("fake_launches") == 1
""")
