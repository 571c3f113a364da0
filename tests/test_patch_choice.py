"""Which products of window tables run patch by patch: both sides of every limit of the choice, without a GPU."""
import _fake_hip


def test_the_products_that_run_patch_by_patch(tmp_path):
    _fake_hip.run(tmp_path, """
def ran(px, py, fs, batch, trans="n", maps=1, path=_lib.PATH_AUTO):
    n = px * py * maps
    A = matrix(n, n, D.filter_factory_float(px, py, fs, maps, maps).offsets())
    L.cuvdia_set_path(path)
    D.prod(tensor(batch, n, bytes_at=1 << 41), A, tensor(batch, n, bytes_at=1 << 42), trans)
    L.cuvdia_set_path(_lib.PATH_AUTO)
    return L.cuvdia_last_kernel().decode()
for call, kernel in [
    ((128, 128, 7, 128), "spmm_tiled_kernel<7, false>"),
    ((128, 128, 7, 128, "t"), "spmm_tiled_kernel<7, false>"),
    ((96, 96, 5, 200), "spmm_tiled_kernel<5, false>"),
    ((100, 100, 3, 500), "spmm_tiled_kernel<3, false>"),
    ((64, 64, 8, 128), "spmm_tiled_kernel<8, 8, 1, false, false>"),           # no patches of 8 x 8 windows
    ((64, 64, 7, 128, "n", 2), "spmm_tiled_kernel<7, 8, 1, false, false>"),   # nor of several maps
    ((64, 64, 7, 32), "spmm_thin_kernel<7, 2, 1>"),                           # few patches
    ((66, 66, 7, 300), "spmm_tiled_kernel<7, false>"),                        # 510 of them
    ((66, 66, 7, 683), "spmm_tiled_kernel<7, 8, 1, false, false>"),           # ... 1122, a third of their positions not there
    ((224, 180, 7, 32), "spmm_thin_kernel<7, 4, 1>"),                         # 315, and 322 of one column tile
    ((224, 184, 7, 32), "spmm_tiled_kernel<7, false>"),
    ((224, 184, 7, 33), "spmm_thin_kernel<7, 4, 1>"),
    ((201, 260, 7, 32), "spmm_thin_kernel<7, 4, 1>"),                         # a tenth of their width not there
]:
    assert ran(*call) == kernel, (call, ran(*call))
assert ran(128, 128, 7, 128, path=_lib.PATH_TILED) == ran(128, 128, 7, 128, path=_lib.PATH_TILED_NOWALK) == "spmm_tiled_kernel<7, 8, 1, false, false>"
""")


def test_patches_only_where_they_are_ahead_of_rows_in_a_line(tmp_path):
    """Rounds of 256 workgroups here and there, widths, ends and exits: a call on either side of every line of the rule."""
    _fake_hip.run(tmp_path, """
def patches(px, py, fs, batch, beta=0.0, act=None):
    n = px * py
    A = matrix(n, n, D.filter_factory_float(px, py, fs, 1, 1).offsets())
    dst, X = tensor(batch, n, bytes_at=1 << 41), tensor(batch, n, bytes_at=1 << 42)
    if act is None:
        D.prod(dst, A, X, "n", "n", 1.0, beta)
    else:
        D.prod_bias_act(dst, A, X, "n", 1.0, beta, bias=tensor(n, bytes_at=1 << 43), act=act)
    name = L.cuvdia_last_kernel().decode()
    assert name.startswith("spmm_tiled_kernel<%d, " % fs)
    return name in ("spmm_tiled_kernel<%d, %s>" % (fs, f) for f in ("true", "false"))
SIGMOID, SAMPLE = _lib.ACT_SIGMOID, _lib.ACT_SIGMOID_SAMPLE
for want, call in [
    # 7 x 7: not more rounds than there
    (False, (104, 104, 7, 156)),                 # 520 patches, 507 tiles
    (False, (224, 146, 7, 61)),                  # 518 and 511
    (True, (224, 144, 7, 64)),                   # 504 and 504
    (True, (224, 147, 7, 64)),                   # 518 and 515
    (False, (100, 154, 7, 64)),                  # 312 and 241
    # one round, two rounds: the widest that are taken, ends of 16-byte pieces, exits
    (True, (71, 72, 7, 64)), (False, (72, 72, 7, 64)), (True, (73, 73, 7, 64)),
    (True, (128, 128, 7, 128)), (True, (128, 128, 7, 128, 0.0, SIGMOID)), (False, (128, 128, 7, 128, 0.0, SAMPLE)),
    (False, (90, 90, 7, 170, 0.0, SIGMOID)), (True, (90, 90, 7, 170)),
    (True, (91, 91, 7, 192, 0.0, SAMPLE)),
    # 5 x 5: a third round that is not there in a line, a sample's second one
    (False, (90, 90, 5, 256)), (True, (62, 65, 5, 512)), (False, (48, 60, 5, 577, 0.0, SAMPLE)), (True, (40, 42, 3, 861)), (True, (96, 96, 5, 256)), (True, (73, 73, 5, 192)), (False, (74, 86, 5, 128, 0.5, SAMPLE)), (True, (47, 64, 5, 942, 0.0, SIGMOID)),
    # 3 x 3: map rows that are no multiples of 16 bytes, only written, from the fourth round on
    (False, (127, 127, 3, 512)), (True, (124, 124, 3, 512)), (True, (127, 127, 3, 512, 0.5)), (True, (127, 127, 3, 512, 0.0, SAMPLE)),
    (False, (186, 272, 3, 640, 0.5)), (True, (303, 303, 3, 80)), (False, (303, 303, 3, 160)), (True, (127, 127, 3, 128)),
]:
    assert patches(*call) == want, (call, L.cuvdia_last_kernel())
""")


def test_which_of_the_two_tile_by_tile_kernels_runs(tmp_path):
    """Both are called spmm_tiled_kernel: rows in a line have five template arguments, patches two.  The calls that other tests expect to
    be served tile by tile."""
    _fake_hip.run(tmp_path, """
def ran(px, py, fs, maps_in, maps_out, batch, trans="n", path=_lib.PATH_AUTO):
    h, w = px * py * maps_in, px * py * maps_out
    A = matrix(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets())
    out, inner = (w, h) if trans == "t" else (h, w)
    L.cuvdia_set_path(path)
    D.prod(tensor(batch, out, bytes_at=1 << 41), A, tensor(batch, inner, bytes_at=1 << 42), trans)
    L.cuvdia_set_path(_lib.PATH_AUTO)
    return L.cuvdia_last_kernel().decode()
for call, kernel in [
    ((40, 40, 7, 1, 1, 150), "spmm_tiled_kernel<7, false>"),
    ((64, 64, 5, 3, 4, 128), "spmm_tiled_kernel<5, 8, 1, false, false>"),
    ((64, 64, 13, 2, 2, 92), "spmm_tiled_kernel<13, 8, 1, false, false>"),
    ((56, 152, 7, 1, 1, 897), "spmm_tiled_kernel<7, 8, 1, false, false>"),
    ((272, 60, 7, 1, 2, 569), "spmm_tiled_kernel<7, 8, 1, false, false>"),
    ((40, 40, 7, 1, 1, 150, "n", _lib.PATH_TILED), "spmm_tiled_kernel<7, 8, 1, false, false>"),
    ((56, 152, 7, 1, 1, 897, "t", _lib.PATH_TILED_NOWALK), "spmm_tiled_kernel<7, 8, 1, false, false>"),
]:
    assert ran(*call) == kernel, (call, ran(*call))
""")
