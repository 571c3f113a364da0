"""The projection of 13 x 13 windows with split operands on the matrix cores, against the oracle where it can go wrong: map
widths and rows around its tiles of 32 x 8 positions, batches around its stages of 16 columns, windows that start at each
remainder of 4 rows, several maps, windows that leave the operands at either end, values that no sum of three bfloat16
numbers holds, and the automatic choice on both sides of its rule."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dia(oracle, rng, h, w, offsets):
    C = oracle.Dia(h, w, offsets, max(h, w), 1)
    valid = oracle.valid_mask(C)
    C.vals[:] = rng.uniform(-1, 1, C.vals.size).astype(np.float32)
    return C, valid


def _offsets(px, rows, shift, maps_in, maps_out):
    """13 x 13 windows, first diagonal `shift` behind the centred one's, one per map distance."""
    return sorted(m * px * rows + dy * px + dx - shift for m in range(1 - maps_in, maps_out) for dy in range(-6, 7) for dx in range(-6, 7))


def _operands(rng, h, w, batch):
    return (np.asfortranarray(rng.uniform(-1, 1, (n, batch)).astype(np.float32)) for n in (h, w))


def _split_ran():
    from cuv_amd import _lib
    return _lib.lib().cuvdia_last_kernel() == b"dd2dia_split_kernel<13, 13>"


@pytest.mark.parametrize("px,rows,shift,maps_in,maps_out,batch,beta", [
    (32, 8, 0, 1, 1, 1, 0.0),        # one tile
    (64, 17, 1, 1, 1, 16, 0.0),
    (68, 9, 2, 1, 1, 17, 0.9),       # a tile of 4 positions, one of a row
    (36, 20, 3, 1, 1, 15, 0.0),
    (132, 31, 0, 1, 1, 130, 0.9),
    (60, 32, 1, 2, 3, 33, 0.5),
    (192, 24, 2, 3, 1, 9, 0.0),
    (256, 16, 3, 2, 2, 48, -1.0),
])
def test_sizes(oracle, px, rows, shift, maps_in, maps_out, batch, beta):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(px + batch)
    h, w = px * rows * maps_in, px * rows * maps_out
    C, valid = _dia(oracle, rng, h, w, _offsets(px, rows, shift, maps_in, maps_out))
    if not beta:
        C.vals[valid] = np.nan                           # only written
    _, ran = gu.check_dd2dia(oracle, C, *_operands(rng, h, w, batch), 1.0 / batch, beta, _lib.PATH_PLANE, "%d x %d" % (px, rows))
    assert _split_ran() and ran == _lib.PATH_PLANE


def test_values_that_no_three_parts_hold(oracle):
    """Infinities and NaN reach their slots only; the smallest numbers keep all their bits, beside ordinary ones too."""
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(5)
    px, rows, batch = 64, 24, 40
    n = px * rows
    C, valid = _dia(oracle, rng, n, n, _offsets(px, rows, 0, 1, 1))
    C.vals[valid] = 0.0
    A, B = _operands(rng, n, n, batch)
    A[5, 1], A[700, 5], B[3, 0], B[901, 33], B[-1, 39] = np.inf, np.nan, -np.inf, np.nan, np.inf
    with np.errstate(invalid="ignore"):
        ref = oracle.dd2dia(C, A, B, 1.0, 0.0)
    got, ran = gu.gpu_dd2dia(C, A, B, path=_lib.PATH_PLANE)
    assert _split_ran() and ran == _lib.PATH_PLANE
    fin = valid & np.isfinite(ref)
    assert np.array_equal(np.isnan(got[valid]), np.isnan(ref[valid])) and np.array_equal(np.isinf(got[valid]), np.isinf(ref[valid]))
    np.testing.assert_allclose(got[fin], ref[fin], rtol=0, atol=1e-5 * batch)          # 1e-5 of the terms' magnitudes, which are below 1
    assert np.array_equal(got[~valid], C.vals[~valid])   # the padding is not written
    # a row of A around 2^-120, the largest numbers elsewhere: sums of either, each against its own terms
    A, B = _operands(rng, n, n, batch)
    A[100] *= np.float32(2.0 ** -120)
    A[900] *= np.float32(2.0 ** 120)
    _, ran = gu.check_dd2dia(oracle, C, A, B, 1.0, 0.0, _lib.PATH_PLANE, "tiny rows")
    assert _split_ran()


@pytest.mark.parametrize("columns", [(3,), (1023,), (1024,), (1045, 1056), (0, 500, 1023, 1024, 1059), (1008, 1039)])
def test_such_values_in_batches_of_several_blocks(oracle, columns):
    """Stages of 16 columns that the split does not hold are multiplied behind their block of 64: the first and the last of a block,
    those of the second, of either operand, and the block that follows."""
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(columns[0])
    px, rows, batch = 32, 16, 1060
    n = px * rows
    C, valid = _dia(oracle, rng, n, n, _offsets(px, rows, 0, 1, 1))
    A, B = _operands(rng, n, n, batch)
    for i, c in enumerate(columns):
        (A if i % 2 == 0 else B)[::7, c] = np.float32(1e-39)
    gu.check_dd2dia(oracle, C, A, B, 1.0 / batch, 0.5, _lib.PATH_PLANE, "tiny numbers in columns %r" % (columns,))
    assert _split_ran()
    C.vals[valid] = 0.0
    for i, c in enumerate(columns):
        (B if i % 2 == 0 else A)[100 + 77 * i, c] = (np.inf, np.nan, -np.inf)[i % 3]
    with np.errstate(invalid="ignore"):
        ref = oracle.dd2dia(C, A, B, 1.0, 0.0)
    got, ran = gu.gpu_dd2dia(C, A, B, path=_lib.PATH_PLANE)
    assert _split_ran() and ran == _lib.PATH_PLANE
    assert np.array_equal(np.isnan(got[valid]), np.isnan(ref[valid])) and np.array_equal(got[valid] == np.inf, ref[valid] == np.inf)
    assert np.array_equal(got[valid] == -np.inf, ref[valid] == -np.inf)
    fin = valid & np.isfinite(ref)
    assert 0 < fin.sum() < valid.sum()
    np.testing.assert_allclose(got[fin], ref[fin], rtol=0, atol=1e-5 * batch)          # 1e-5 of the terms' magnitudes, which are below 1


@pytest.mark.parametrize("px,rows,batch,split", [(256, 256, 128, True), (256, 256, 127, False), (256, 264, 128, False)])
def test_automatic_choice(oracle, px, rows, batch, split):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(batch)
    h = px * rows
    C, valid = _dia(oracle, rng, h, h, _offsets(px, rows, 0, 1, 1))
    gu.check_dd2dia(oracle, C, *_operands(rng, h, h, batch), 0.5, 0.9, _lib.PATH_AUTO, "automatic choice")
    assert _split_ran() == split                         # 256 tiles, one per CU; 264 are two rounds
