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


def test_a_device_without_an_event_leaves_the_other_devices_wait_alone(tmp_path):
    _fake_hip.run(tmp_path, """
event = L["_ZN6cuvdia12launch_eventEv"]                  # cuvdia::launch_event()
event.restype = ctypes.c_void_p
wait_begin, wait_end = L.cuvdia_wait_begin, L.cuvdia_wait_end
wait_end.argtypes = [ctypes.c_void_p]
assert wait_begin() == 0
first = event()
assert first and wait_end(None) == 0 and flag("fake_waited_event", kind=ctypes.c_void_p) == first
flag("fake_device", 1)
flag("fake_fail_event_create", 1)
assert wait_begin() == _lib.EHIP
flag("fake_device", 0)
assert wait_begin() == 0
assert event() == first and wait_end(None) == 0
flag("fake_fail_event_create", 0)
flag("fake_device", 1)
assert wait_begin() == 0
second = event()
assert second and second != first and wait_end(None) == 0 and flag("fake_waited_event", kind=ctypes.c_void_p) == second
""")
