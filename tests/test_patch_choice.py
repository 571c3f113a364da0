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
