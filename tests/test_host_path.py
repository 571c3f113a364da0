"""The calls' way through cuv_amd/dia.py, the Python module and the library's dispatch, on a runtime without a GPU
(tests/cxx/fake_hip.c), so that waits and launches can fail and calls can be held where they are."""
import pytest

import _fake_hip


CALLS = """
A, G = matrix(64, 64, [-1, 0, 1]), matrix(64, 64, [-1, 0, 1])
x, y, w, m, d = tensor(4, 64), tensor(4, 64), tensor(100), tensor(100), tensor(100)
CALLS = [lambda sync: D.prod(y, A, x, "n", "n", 1.0, 0.5, sync=sync),
         lambda sync: D.prod_bias_act(y, A, x, "n", 1.0, 0.5, act=1, sync=sync),
         lambda sync: D.densedense_to_dia(G, None, x, y, 1.0, 1.0, sync=sync),
         lambda sync: D.learn_step_weight_decay(w, d, 0.1, sync=sync),
         lambda sync: D.learn_step_weight_decay_momentum(w, m, d, 0.1, sync=sync)]
for call in CALLS:
    call(True)
    call(False)
assert flag("fake_launches") == 10
"""


def test_a_call_that_fails_after_its_launch_is_raised_and_not_done_again(tmp_path):
    _fake_hip.run(tmp_path, CALLS + """
general = []
real, _lib.lib = _lib.lib, lambda: general.append(1) or real()
for fail in ("fake_fail_wait", "fake_fail_launch"):
    for k, call in enumerate(CALLS):
        for sync in (True, False):
            if fail == "fake_fail_wait" and not sync: continue
            before = flag("fake_launches")
            flag(fail, 1)
            try:
                call(sync)
                raise SystemExit("no error: %s of call %d" % (fail, k))
            except _lib.CuvDiaError as e:
                assert e.code == _lib.EHIP and "a failure asked for" in str(e), e
            finally:
                flag(fail, 0)
            assert flag("fake_launches") == before + 1, (fail, k, sync)
            call(sync)                                   # and the next call is an ordinary one
            assert flag("fake_launches") == before + 2
""")


def test_a_wait_that_cannot_begin_leaves_the_call_undone(tmp_path):
    _fake_hip.run(tmp_path, """
A, x, y = matrix(64, 64, [-1, 0, 1]), tensor(4, 64), tensor(4, 64)
flag("fake_fail_event_create", 1)
assert D._native.product(y, A, x, "n", 1.0, 0.0, None, 0, 0, True) is False and flag("fake_launches") == 0
flag("fake_fail_event_create", 0)
assert D._native.product(y, A, x, "n", 1.0, 0.0, None, 0, 0, True) is True and flag("fake_launches") == 1
flag("fake_fail_capturing", 1)                           # the stream cannot be asked whether it is being captured
assert D._native.product(y, A, x, "n", 1.0, 0.0, None, 0, 0, True) is False and flag("fake_launches") == 1
flag("fake_fail_capturing", 0)
assert D._native.product(y, A, x, "n", 1.0, 0.0, None, 0, 0, True) is True and flag("fake_launches") == 2
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


def test_tensors_without_memory_are_left_to_the_general_way(tmp_path):
    """Wrappers that torch hands out inside a transform, and fake tensors: a Python exception, as the general way words it."""
    _fake_hip.run(tmp_path, """
import torch._subclasses.fake_tensor as ft
ft.init_gpu_context = lambda *a: None
A, x, v = matrix(64, 64, [-1, 0, 1]), tensor(4, 64), tensor(100)
with ft.FakeTensorMode():
    fake, fake_v = torch.empty(4, 64, device="cuda:0"), torch.empty(100, device="cuda:0")
assert fake.is_cuda
N = D._native
def calls(t, u):
    return [(lambda: N.product(t, A, x, "n", 1.0, 0.0, None, 0, 0, True), lambda: D.prod(t, A, x)),
            (lambda: N.product(x, A, t, "n", 1.0, 0.0, None, 0, 0, True), lambda: D.prod(x, A, t)),
            (lambda: N.product(x, A, x, "n", 1.0, 0.0, u[:64], 0, 0, True), lambda: D.prod_bias_act(x, A, x, bias=u[:64])),
            (lambda: N.projection(A, t, x, 1.0, 0.0, True), lambda: D.densedense_to_dia(A, None, t, x)),
            (lambda: N.projection(A, x, t, 1.0, 0.0, True), lambda: D.densedense_to_dia(A, None, x, t)),
            (lambda: N.weight_step(u, None, v, 0.1, 0.0, 0.0, True), lambda: D.learn_step_weight_decay(u, v, 0.1)),
            (lambda: N.weight_step(v, u, v, 0.1, 0.9, 0.0, True), lambda: D.learn_step_weight_decay_momentum(v, u, v, 0.1)),
            (lambda: N.weight_step(v, None, u, 0.1, 0.0, 0.0, True), lambda: D.learn_step_weight_decay(v, u, 0.1))]
assert not any(direct() for direct, _ in calls(fake, fake_v))
def check(t, u):
    for k, (direct, whole) in enumerate(calls(t, u)):
        assert direct() is False
        try:
            whole()
            raise SystemExit("no error: call %d" % k)
        except (RuntimeError, TypeError):
            pass
    return torch.zeros(1)
torch.func.vmap(check)(tensor(3, 4, 64), tensor(3, 100))
torch.func.functionalize(lambda t, u: any(direct() for direct, _ in calls(t, u)) and 1 / 0)(x, v)
class Holder: pass
h = Holder()                                             # a matrix whose values are such a tensor
h.h, h.w, h._desc_ptr, h.vec = 64, 64, A._desc_ptr, fake_v
assert N.product(x, h, x, "n", 1.0, 0.0, None, 0, 0, True) is False and N.projection(h, x, x, 1.0, 0.0, True) is False
assert flag("fake_launches") == 0
""")


def test_other_threads_run_during_launches_and_waits(tmp_path):
    _fake_hip.run(tmp_path, CALLS + """
import threading, time
for call in CALLS:
    for sync in (True, False):
        flag("fake_hold_launch", 1)                      # the call stays in its launch until the other thread lets it go on
        other = threading.Thread(target=lambda: (time.sleep(0.02), flag("fake_hold_launch", 0)))
        other.start()
        call(sync)
        other.join()
assert flag("fake_held") == 0
""")


def test_the_planned_window_projection_is_the_one_that_runs(tmp_path):
    """cuvdia_plan_window_launch against what a call on packed operands takes, over maps, windows and batches on both sides
    of its rules, operands above 2 GiB among them."""
    _fake_hip.run(tmp_path, """
import random
rng, seen = random.Random(2), set()
cases = [(500, 500, 7, 1, 1, b) for b in (4, 8, 9)] + [(512, 512, 7, 1, 1, 4), (1024, 1024, 5, 1, 1, 700), (1000, 1000, 5, 1, 1, 700)]
for _ in range(400):
    px = rng.choice([rng.randint(15, 160) * 4, rng.randint(1, 10) * 64, rng.randint(60, 640)])
    maps = rng.choice([(1, 1), (1, 1), (2, 2), (1, 4)])
    cases.append((px, rng.randint(16, 600), rng.choice([3, 5, 7, 8, 9, 10, 11, 13]), *maps, rng.choice([rng.randint(1, 12), rng.randint(13, 700)])))
for px, py, fs, maps_in, maps_out, batch in cases:
    h, w = px * py * maps_in, px * py * maps_out
    C = matrix(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets())
    plan = L.cuvdia_plan_window_launch(C._offsets.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), C.num_dia, C.stride, h, w, batch)
    D.densedense_to_dia(C, None, tensor(batch, h, bytes_at=1 << 41), tensor(batch, w, bytes_at=1 << 42), 1.0, 0.0)
    ran = L.cuvdia_last_path()
    what = (px, py, fs, maps_in, maps_out, batch, plan, L.cuvdia_last_kernel())
    assert (plan > 0) == (ran in (_lib.PATH_WINDOW, _lib.PATH_PLANE)), what
    assert ran != _lib.PATH_WINDOW or plan == flag("fake_grid"), what
    seen.add(L.cuvdia_last_kernel().split(b"<")[0])
assert seen >= {b"dd2dia_window_kernel", b"dd2dia_window_long_kernel", b"dd2dia_rows_kernel", b"dd2dia_tiled_kernel"}, seen
""")


def test_the_projections_that_run_with_rows_along_the_lanes(tmp_path):
    """Both sides of every limit of the choice on operands that any kernel could take."""
    _fake_hip.run(tmp_path, """
def rows(M, batch):
    D.densedense_to_dia(M, None, tensor(batch, M.h, bytes_at=1 << 41), tensor(batch, M.w, bytes_at=1 << 42), 1.0, 0.0)
    return L.cuvdia_last_kernel().startswith(b"dd2dia_rows_kernel")
def window(px, py, fs, maps_in=1, maps_out=1):
    return matrix(px * py * maps_in, px * py * maps_out, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets())
for M, yes, no in [
    (window(64, 64, 7), [1, 2, 4, 128, 257, 2048], [3, 129, 256, 2049, 8192]),       # 112 tiles of 256 rows and a chunk
    (window(64, 64, 5), [96, 257], [97]),
    (window(64, 64, 7, 1, 2), [64, 300], [65]),                                      # 14 chunks
    (window(120, 120, 7), [3, 48], [49, 300]),                                       # 399 tiles
    (window(128, 128, 5), [3, 16], [17, 300]),                                       # 320
    (matrix(262 * 262, 262 * 262, list(range(-7, 8))), [64], [65, 300]),             # 538, two chunks
    (window(280, 280, 7), [16], [17]),                                               # 2149
    (window(356, 356, 5), [12], [13]),                                               # 2480
    (window(416, 217, 5, 1, 2), [16], [17]),                                         # ..., two maps
    (window(408, 408, 3), [8], [9]),
    (window(480, 293, 3, 1, 2), [16], [17]),
    (matrix(504 * 732, 504 * 732, list(range(-3, 4))), [], [1, 8]),                  # one chunk
    (window(500, 500, 7), [8], [9]),                                                 # window rows staged for the whole window
    (window(500, 500, 9), [20], [21]),
]:
    for batch in yes + no:
        assert rows(M, batch) == (batch in yes), (M.h, M.w, M.num_dia, batch, L.cuvdia_last_kernel())
""")


def test_the_products_of_few_columns_that_run_with_rows_along_the_lanes(tmp_path):
    """Both sides of every limit of the choice on many tiles."""
    _fake_hip.run(tmp_path, """
def thin(M, trans, batch):
    out, inner = (M.w, M.h) if trans == "t" else (M.h, M.w)
    D.prod(tensor(batch, out, bytes_at=1 << 41), M, tensor(batch, inner, bytes_at=1 << 42), trans)
    return L.cuvdia_last_kernel().startswith(b"spmm_thin_kernel")
def window(px, py, fs, maps_in=1, maps_out=1):
    return matrix(px * py * maps_in, px * py * maps_out, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets())
for M, trans, yes, no in [
    (window(201, 260, 7), "n", [24, 32, 35], [36]),          # 4 columns per lane
    (window(152, 152, 3, 4, 4), "n", [24, 35], [36]),        # 8
    (window(332, 332, 7, 2, 2), "n", [24, 32], [33]),
    (window(340, 340, 6, 2, 5), "t", [], [24, 25, 32]),      # 8, window rows of 6 and of 13 diagonals
    (window(90, 90, 13, 1, 16), "t", [], [24, 32]),
    (window(420, 420, 6), "n", [24, 35], [36]),              # 4
    (window(32, 410, 8, 1, 8), "t", [24], [25, 30]),         # 15 chunks' rows, of which a row block meets 8
    (window(164, 234, 8, 1, 8), "t", [24, 32], [33]),        # ..., on more than 1000 tiles
    (window(57, 152, 7, 1, 8), "t", [28], [29]),
    (window(96, 260, 5, 1, 8), "t", [24, 35], [36]),
]:
    for batch in yes + no:
        assert thin(M, trans, batch) == (batch in yes), (M.h, M.w, M.num_dia, batch, L.cuvdia_last_kernel())
""")


def test_the_planned_walk_is_the_one_that_runs(tmp_path):
    """cuvdia_plan_walk_launch against the kernel and the grid of the product, over maps, windows and batches on both sides of
    its rules."""
    _fake_hip.run(tmp_path, """
import random
rng, seen = random.Random(3), set()
for _ in range(400):
    px, py = rng.choice([rng.randint(1, 10) * 64, rng.randint(40, 640)]), rng.randint(16, 700)
    fs, maps = rng.choice([3, 5, 7, 7, 9]), rng.choice([(1, 1), (1, 1), (2, 2), (1, 4)])
    batch, trans = rng.choice([rng.randint(1, 40), rng.randint(41, 700)]), rng.choice("nt")
    h, w = px * py * maps[0], px * py * maps[1]
    A = matrix(h, w, D.filter_factory_float(px, py, fs, *maps).offsets())
    plan = L.cuvdia_plan_walk_launch(A._offsets.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), A.num_dia, A.stride, h, w, trans == "t", batch)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    D.prod_bias_act(tensor(batch, n_out, bytes_at=1 << 41), A, tensor(batch, n_in, bytes_at=1 << 42), trans, act=rng.choice([0, 1, 2]))
    ran = L.cuvdia_last_path()
    assert (plan > 0) == (ran == _lib.PATH_WALK), (px, py, fs, maps, batch, trans, plan, L.cuvdia_last_kernel())
    assert ran != _lib.PATH_WALK or plan == flag("fake_grid")
    seen.add(L.cuvdia_last_kernel().split(b"<")[0])
assert seen >= {b"spmm_walk_kernel", b"spmm_plane_kernel", b"spmm_thin_kernel", b"spmm_tiled_kernel"}, seen
""")


def test_sampled_layers_of_one_map_leave_the_plane_earlier(tmp_path):
    """9 x 9 windows: a sample at every block's exit with one map, at every second or fourth with more."""
    _fake_hip.run(tmp_path, """
def ran(px, py, maps, batch, act):
    n = px * py * maps
    A = matrix(n, n, D.filter_factory_float(px, py, 9, maps, maps).offsets())
    D.prod_bias_act(tensor(batch, n, bytes_at=1 << 41), A, tensor(batch, n, bytes_at=1 << 42), "n", act=act)
    return L.cuvdia_last_path() == _lib.PATH_PLANE
assert ran(396, 396, 1, 576, _lib.ACT_SIGMOID), L.cuvdia_last_kernel()
assert not ran(396, 396, 1, 576, _lib.ACT_SIGMOID_SAMPLE)
assert ran(345, 345, 2, 128, _lib.ACT_SIGMOID_SAMPLE), L.cuvdia_last_kernel()
assert ran(509, 444, 1, 329, _lib.ACT_SIGMOID_SAMPLE)
""")


def test_layers_on_either_side_of_the_planes_lines(tmp_path):
    """Samples of several maps, a sigmoid on tiles that the width fills badly, samples of a few columns more than a tile."""
    _fake_hip.run(tmp_path, """
def ran(px, py, fs, maps_in, maps_out, batch, trans, act):
    h, w = px * py * maps_in, px * py * maps_out
    A = matrix(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets())
    out, inner = (w, h) if trans == "t" else (h, w)
    D.prod_bias_act(tensor(batch, out, bytes_at=1 << 41), A, tensor(batch, inner, bytes_at=1 << 42), trans, act=act)
    return L.cuvdia_last_kernel().decode().split("<")[0]
for call, kernel in [
    ((150, 150, 7, 4, 6, 200, "n", _lib.ACT_NONE), "spmm_plane_kernel"),
    ((56, 152, 7, 1, 1, 897, "n", _lib.ACT_NONE), "spmm_tiled_kernel"),                  # segments of few map rows
    ((272, 60, 7, 1, 2, 569, "n", _lib.ACT_NONE), "spmm_tiled_kernel"),
    ((288, 318, 11, 4, 4, 154, "t", _lib.ACT_SIGMOID_SAMPLE), "spmm_plane_kernel"),
    ((520, 520, 11, 1, 1, 537, "n", _lib.ACT_SIGMOID), "spmm_plane_kernel"),
    ((171, 270, 7, 2, 5, 94, "t", _lib.ACT_SIGMOID), "spmm_plane_kernel"),
    ((261, 261, 7, 4, 4, 128, "n", _lib.ACT_SIGMOID_SAMPLE), "spmm_plane_kernel"),
    ((310, 310, 5, 3, 4, 71, "n", _lib.ACT_SIGMOID), "spmm_plane_kernel"),
    ((310, 310, 5, 3, 4, 71, "n", _lib.ACT_SIGMOID_SAMPLE), "spmm_thin_kernel"),
    ((310, 310, 5, 3, 4, 77, "n", _lib.ACT_SIGMOID_SAMPLE), "spmm_plane_kernel"),
    ((160, 189, 7, 1, 16, 70, "t", _lib.ACT_SIGMOID_SAMPLE), "spmm_plane_kernel"),       # 7 chunks a tile
]:
    assert ran(*call) == kernel, (call, L.cuvdia_last_kernel())
""")


def test_an_empty_batch_is_launched_for_the_projection_alone(tmp_path):
    _fake_hip.run(tmp_path, """
A = matrix(4096, 4096, [64 * dy + dx for dy in range(-2, 3) for dx in range(-2, 3)])
D.prod(tensor(0, 4096, bytes_at=1 << 41), A, tensor(0, 4096, bytes_at=1 << 42))
assert flag("fake_launches") == 0                        # a product of no columns has no result
for path in (_lib.PATH_AUTO, _lib.PATH_TILED):
    L.cuvdia_set_path(path)
    D.densedense_to_dia(A, None, tensor(0, 4096, bytes_at=1 << 41), tensor(0, 4096, bytes_at=1 << 42), 1.0, 0.5)
assert flag("fake_launches") == 2 and L.cuvdia_last_kernel() == b"dd2dia_generic_kernel"
""")


def test_forced_families(tmp_path):
    """CUVDIA_PATH_TILED runs the kernels that stage operands, at every batch, or nothing; CUVDIA_PATH_THIN is a product's
    choice alone."""
    _fake_hip.run(tmp_path, """
A = matrix(4099, 4099, [64 * dy + dx for dy in range(-2, 3) for dx in range(-2, 3)])
huge = matrix(1 << 24, 1 << 24, list(range(-20, 20)))    # 2.5 GiB of values
def ran(path, M, batch):
    x, y = tensor(batch, M.w, bytes_at=1 << 41), tensor(batch, M.h, bytes_at=1 << 42)
    L.cuvdia_set_path(path)
    names = []
    for call in (lambda: D.prod(y, M, x), lambda: D.densedense_to_dia(M, None, y, x)):
        try:
            call()
            names.append(L.cuvdia_last_kernel().decode().split("<")[0])
        except _lib.CuvDiaError as e:
            names.append(e.code)
    return names
for batch in (1, 4, 23, 24, 100):
    assert ran(_lib.PATH_TILED, A, batch) == ["spmm_tiled_kernel", "dd2dia_tiled_kernel"], (batch, L.cuvdia_last_kernel())
    assert ran(_lib.PATH_AUTO, A, batch)[1] == ran(_lib.PATH_THIN, A, batch)[1] == "dd2dia_rows_kernel"
    assert ran(_lib.PATH_THIN, A, batch)[0] == "spmm_thin_kernel"
large = matrix(256 * 512, 256 * 512, D.filter_factory_float(256, 512, 9, 1, 1).offsets())      # matrix cores, by size
assert ran(_lib.PATH_AUTO, large, 256) == ["spmm_plane_kernel", "dd2dia_plane_kernel"]
assert ran(_lib.PATH_TILED, large, 256) == ["spmm_tiled_kernel", "dd2dia_window_long_kernel"]
assert ran(_lib.PATH_TILED, huge, 8) == [_lib.EUNSUPPORTED] * 2
assert ran(_lib.PATH_AUTO, huge, 8) == ["spmm_thin_kernel", "dd2dia_rows_kernel"]
rf2 = matrix(100, 50, [-1, 0, 1], 2)
assert ran(_lib.PATH_TILED, rf2, 8) == [_lib.EUNSUPPORTED] * 2 and ran(_lib.PATH_THIN, rf2, 8)[0] == _lib.EUNSUPPORTED
""")


MEMORY = """
ip = ctypes.POINTER(ctypes.c_int)
def table(offsets): return (ctypes.c_int * len(offsets))(*offsets)
win = [dy * 40 + dx + 1600 * m for m in range(-1, 2) for dy in range(-2, 3) for dx in range(-2, 3)]
offs, nd, n = table(win), len(win), 3200
x, y, v = 1 << 41, 1 << 42, 1 << 43
A = matrix(n, n, win)
f = ctypes.c_float
"""


def test_compute_calls_allocate_nothing(tmp_path):
    _fake_hip.run(tmp_path, MEMORY + """
calls = [lambda b: L.cuvdia_spmm_f32(A.desc, v, x, n, y, n, b, b"n", 1.0, 0.5, None),
         lambda b: L.cuvdia_spmm_layer_f32(A.desc, v, x, n, y, n, b, b"t", 1.0, 0.0, v, 2, 7, None),
         lambda b: L.cuvdia_dd2dia_f32(A.desc, v, x, n, y, n, b, 1.0, 0.0, None),
         lambda b: L.cuvdia_avg_diagonals_f32(A.desc, v, x, None),
         lambda b: L.cuvdia_learn_step_weight_decay_momentum_f32(x, y, v, 1000, 0.1, 0.9, 0.0, None)]
for path in (0, 1, 2, 4, 6, 8):
    L.cuvdia_set_path(path)
    for b in (1, 30, 200):
        before = flag("fake_news")
        for call in calls:
            assert call(b) == 0, (path, b)
            assert flag("fake_news") == before, (path, b, L.cuvdia_last_kernel())
""")


def test_no_memory_is_an_error_code(tmp_path):
    """Every allocation of every entry point, one after the other, fails: std::bad_alloc must not leave through the C ABI."""
    _fake_hip.run(tmp_path, MEMORY + """
def create():
    d = ctypes.c_void_p()
    rc = L.cuvdia_desc_create(ctypes.byref(d), offs, nd, n, n, n, 1)
    return rc if rc else L.cuvdia_desc_destroy(d)
def offsets_call():
    rc = L.cuvdia_spmm_offsets_f32(v, offs, nd, n, n, n, 1, x, n, y, n, 30, b"n", 1.0, 0.0, None)
    return rc if rc else L.cuvdia_cache_clear()
def waited():
    rc = L.cuvdia_wait_begin()
    return rc if rc else L.cuvdia_wait_end(None)
def failed_launch():
    flag("fake_fail_launch", 1)
    rc = L.cuvdia_spmm_f32(A.desc, v, x, n, y, n, 30, b"n", 1.0, 0.0, None)
    flag("fake_fail_launch", 0)
    assert rc == _lib.EHIP and b"a failure asked for" in L.cuvdia_last_hip_error()
    return 0
L.cuvdia_wait_end.argtypes = [ctypes.c_void_p]
c1, c2 = table([0] * 100), table([0] * 100)
calls = dict(create=create, offsets=offsets_call, waited=waited, failed_launch=failed_launch,
             dd2dia=lambda: L.cuvdia_dd2dia_offsets_f32(v, offs, nd, n, n, n, 1, x, n, y, n, 30, 1.0, 0.0, None) or L.cuvdia_cache_clear(),
             noalloc=lambda: L.cuvdia_spmm_offsets_noalloc_f32(v, offs, nd, n, n, n, 1, x, n, y, n, 30, b"t", 1.0, 0.0, None),
             chunks=lambda: min(0, L.cuvdia_plan_chunks(offs, nd, 0, c1, c2, c1, 0)), units=lambda: min(0, L.cuvdia_plan_units(offs, nd, c1, c2, 100)),
             walk=lambda: min(0, L.cuvdia_plan_walk(offs, nd, n, 0, None, None, None, None)),
             walk_launch=lambda: min(0, L.cuvdia_plan_walk_launch(offs, nd, n, n, n, 0, 64)),
             window_launch=lambda: min(0, L.cuvdia_plan_window_launch(offs, nd, n, n, n, 64)))
for name, call in calls.items():
    for k in range(1, 400):
        print(name, k, flush=True)
        flag("fake_fail_new", k)
        rc = call()
        reached = flag("fake_fail_new") == 0
        flag("fake_fail_new", 0)
        assert rc in (0, _lib.ENOMEM), (name, k, rc)     # (0: an allocation that there is another way without)
        if not reached:
            assert rc == 0
            break
    else:
        raise SystemExit(name)
    assert call() == 0
""")


@pytest.mark.parametrize("first", ["sys.modules['cuv_amd._native'] = None", "torch.__version__ = '2.9.1+rocm6.4'",
                                   "torch.__version__ += '.post1'"])
def test_without_a_module_that_fits_the_calls_go_through_ctypes(tmp_path, first):
    fits = "post1" in first
    out = _fake_hip.run(tmp_path, CALLS + """
print("module" if D._native.__class__.__name__ == "module" else "ctypes")
""", "import ctypes, os, sys\nctypes.CDLL(os.environ['FAKE_HIP'], mode=ctypes.RTLD_GLOBAL)\nimport torch\n" + first)
    assert out.split()[-1] == ("module" if fits else "ctypes")
    assert ("slower way through ctypes" in out) != fits
