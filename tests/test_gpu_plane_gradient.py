"""The projection of square windows on the matrix cores, against the oracle where it can go wrong: map widths around its
tiles of 64 positions, map rows around its tiles of 8, batches around its stages of 4 columns, windows that start at each
remainder of 4 rows, several maps, windows that leave the operands at either end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dia(oracle, rng, h, w, offsets):
    C = oracle.Dia(h, w, offsets, max(h, w), 1)
    valid = oracle.valid_mask(C)
    C.vals[:] = rng.uniform(-1, 1, C.vals.size).astype(np.float32)
    return C, valid


def _offsets(px, rows, k, shift, maps_in, maps_out):
    """k x k windows, first diagonal `shift` behind the centred one's, one per map distance."""
    return sorted(m * px * rows + dy * px + dx - shift for m in range(1 - maps_in, maps_out)
                  for dy in range(-(k // 2), k - k // 2) for dx in range(-(k // 2), k - k // 2))


@pytest.mark.parametrize("k", [9, 11])
@pytest.mark.parametrize("px,rows,shift,maps_in,maps_out,batch,beta", [
    (64, 17, 0, 1, 1, 4, 0.0),
    (68, 8, 1, 1, 1, 5, 0.9),
    (36, 20, 2, 1, 1, 1, 0.0),
    (132, 9, 3, 1, 1, 130, 0.9),
    (60, 32, 1, 2, 3, 7, 0.5),
    (192, 24, 2, 3, 1, 9, 0.0),
    (256, 16, 0, 2, 2, 33, -1.0),
])
def test_sizes(oracle, k, px, rows, shift, maps_in, maps_out, batch, beta):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(k * px + batch)
    h, w = px * rows * maps_in, px * rows * maps_out
    C, valid = _dia(oracle, rng, h, w, _offsets(px, rows, k, shift, maps_in, maps_out))
    A = np.asfortranarray(rng.uniform(-1, 1, (h, batch)).astype(np.float32))
    B = np.asfortranarray(rng.uniform(-1, 1, (w, batch)).astype(np.float32))
    if not beta:
        C.vals[valid] = np.nan                           # only written
    gu.check_dd2dia(oracle, C, A, B, 1.0 / batch, beta, _lib.PATH_PLANE, "%d x %d, window %d" % (px, rows, k))
    assert _lib.lib().cuvdia_last_kernel().decode().startswith("dd2dia_plane_kernel<%d, " % k)
    assert _lib.lib().cuvdia_last_path() == _lib.PATH_PLANE


def test_non_finite_operands_reach_their_slots_only(oracle):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(5)
    px, rows, batch = 64, 24, 6
    C, valid = _dia(oracle, rng, px * rows, px * rows, _offsets(px, rows, 9, 0, 1, 1))
    C.vals[valid] = 0.0
    A = np.asfortranarray(rng.uniform(-1, 1, (px * rows, batch)).astype(np.float32))
    B = np.asfortranarray(rng.uniform(-1, 1, (px * rows, batch)).astype(np.float32))
    A[5, 1], A[700, 5], B[3, 0], B[901, 2], B[-1, 5] = np.inf, np.nan, -np.inf, np.nan, np.inf
    with np.errstate(invalid="ignore"):
        ref = oracle.dd2dia(C, A, B, 1.0, 0.0)
    got, ran = gu.gpu_dd2dia(C, A, B, path=_lib.PATH_PLANE)
    assert ran == _lib.PATH_PLANE
    assert np.array_equal(np.isnan(got[valid]), np.isnan(ref[valid])) and np.array_equal(np.isinf(got[valid]), np.isinf(ref[valid]))
    assert np.array_equal(got[~valid], C.vals[~valid])   # the padding is not written


@pytest.mark.parametrize("k,px,rows,maps_out,batch,kernel", [
    (9, 256, 256, 2, 24, "dd2dia_plane_kernel<9, 9>"),       # 256 tiles: one of them per CU
    (11, 256, 128, 4, 26, "dd2dia_plane_kernel<11, 11>"),    # 256, of several maps
    (9, 256, 256, 1, 24, "dd2dia_window_long_kernel"),       # 128: half the chip
])
def test_automatic_choice(oracle, k, px, rows, maps_out, batch, kernel):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(k)
    h, w = px * rows, px * rows * maps_out
    C, valid = _dia(oracle, rng, h, w, _offsets(px, rows, k, 0, 1, maps_out))
    A = np.asfortranarray(rng.uniform(-1, 1, (h, batch)).astype(np.float32))
    B = np.asfortranarray(rng.uniform(-1, 1, (w, batch)).astype(np.float32))
    gu.check_dd2dia(oracle, C, A, B, 0.5, 0.9, _lib.PATH_AUTO, "automatic choice")
    assert _lib.lib().cuvdia_last_kernel().decode().startswith(kernel)
