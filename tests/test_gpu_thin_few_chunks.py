"""The product with rows along the lanes where a row block meets few chunks: every number of waves and of columns per lane that
is chosen there, ragged rows and batches, both transposes, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch,trans,columns", [
    (227, 221, 3, 1, 1, 23, "n", 4),      # 3 chunks: 2 waves
    (227, 221, 5, 1, 1, 22, "t", 4),      # 5: 4 waves
    (227, 221, 13, 1, 1, 9, "n", 4),
    (223, 225, 5, 1, 4, 17, "t", 4),      # many workgroups: 2 waves
    (251, 249, 3, 1, 4, 131, "t", 8),     # 16 thousand, 8 columns per lane: 1 wave
    (253, 255, 3, 1, 16, 24, "t", 8),     # 12 thousand: 2 waves
    (227, 223, 9, 4, 2, 9, "n", 8),       # 18 chunks of a table of 45: as before
])
def test_shapes(oracle, px, py, fs, maps_in, maps_out, batch, trans, columns):
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(px + batch)
    h, w = px * py * maps_in, px * py * maps_out
    A = oracle.Dia(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets(), max(h, w), 1)
    A.vals[:] = np.nan                                   # padding must never be read
    valid = oracle.valid_mask(A)
    A.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
    gu.check_prod(oracle, A, B, dst, trans, 0.75, -0.5, _lib.PATH_THIN, "%d x %d" % (px, py))
    assert _lib.lib().cuvdia_last_kernel() == b"spmm_thin_kernel<%d, %d, 1>" % (fs, columns)


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch,trans,thin", [
    (201, 192, 7, 1, 1, 32, "n", True),       # half of the 64 columns, 302 tiles by those that exist
    (201, 190, 7, 1, 1, 32, "t", False),      # 299
    (201, 192, 7, 1, 1, 36, "n", False),
    (201, 100, 7, 1, 1, 67, "n", False),      # the second column tile nearly empty
])
def test_few_columns_of_many_tiles(oracle, px, py, fs, maps_in, maps_out, batch, trans, thin):
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(px + py + batch)
    h, w = px * py * maps_in, px * py * maps_out
    A = oracle.Dia(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets(), max(h, w), 1)
    A.vals[:] = rng.uniform(-1, 1, A.vals.shape).astype(np.float32)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
    gu.check_prod(oracle, A, B, dst, trans, 1.0, 0.5, _lib.PATH_AUTO, "%d x %d" % (px, py))
    assert _lib.lib().cuvdia_last_kernel().decode().startswith("spmm_thin_kernel") == thin
