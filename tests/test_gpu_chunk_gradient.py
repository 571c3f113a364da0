"""The gradient chunk by chunk, added to old values: quads of rows of which a part exists, in the middle of the buffer, at its very end and
in a buffer shorter than a quad; pairs of rows that share B, whose chunks' sums meet at once or one after the other; against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _window(px, rows, length, shifts=(0,)):
    """Window rows of `length` diagonals on maps px wide, a window for every shift; an odd number of rows leaves one to pair with the
    next window's first."""
    return sorted(s + dy * px + dx for s in shifts for dy in range(-(rows // 2), rows - rows // 2) for dx in range(-(length // 2), length - length // 2))


@pytest.mark.parametrize("h,w,offsets,batch,kernel", [
    (101, 99, range(-3, 4), 40, "7, false, false, 0"),       # the last quad ends past the buffer
    (103, 110, range(0, 5), 33, "5, false, false, 0"),
    (3, 5, [1], 24, "1, false, false, 0"),                   # 12 bytes of values
    (5, 4, [0], 24, "1, false, false, 0"),
    (100, 97, range(-6, 7), 40, "13, true, false, 0"),       # long chunks
    (100, 140, range(30, 43), 25, "13, true, false, 0"),
    (512, 509, range(-2, 3), 64, "5, true, false, 0"),
    (1024, 1024, _window(32, 7, 7), 48, "7, true, true, 0"),
    (1024, 1021, _window(160, 3, 3), 36, "3, true, true, 1"),
    (2048, 2048, _window(32, 3, 4, (-1024, 0, 1024)), 40, "4, true, true, 2"),
    (2048, 2048, _window(32, 5, 5, (-1024, 0, 1024)), 40, "5, true, true, 2"),
    (2048, 2045, _window(32, 5, 6, (-1024, 0, 1024)), 29, "6, true, true, 2"),
    (2048, 2048, _window(32, 7, 7, (-1024, 0, 1024)), 40, "7, true, true, 2"),
    (2048, 2048, _window(32, 7, 8, (-1024, 0, 1024)), 40, "8, true, true, 2"),
])
def test_added_to_old_values(oracle, h, w, offsets, batch, kernel):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(h + batch)
    C = oracle.Dia(h, w, np.asarray(list(offsets), np.int32), h, 1)
    C.vals[:] = np.nan                                   # padding is neither used nor written
    valid = oracle.valid_mask(C)
    C.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    A, B = (np.asfortranarray(rng.uniform(-1, 1, (n, batch)).astype(np.float32)) for n in (h, w))
    for alpha, beta in ((1.0 / batch, 0.9), (0.5, 0.0), (-1.0, 1.0)):
        _, ran = gu.check_dd2dia(oracle, C, A, B, alpha, beta, _lib.PATH_TILED, "%d x %d, beta %g" % (h, w, beta))
        assert ran == _lib.PATH_TILED and _lib.lib().cuvdia_last_kernel().decode() == "dd2dia_tiled_kernel<%s>" % kernel
