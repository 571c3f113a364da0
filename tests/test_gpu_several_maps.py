"""Products of layers with several maps, whose tiles meet a few of the table's window rows: the walking kernel's blocks without
dense rows, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(oracle, offsets, h, w, batch, trans, path, what):
    import _gpu_util as gu
    rng = np.random.default_rng(h + w + batch)
    A = oracle.Dia(h, w, np.asarray(offsets, np.int32), max(h, w), 1)
    A.vals[:] = np.nan                                   # padding must never be read
    valid = oracle.valid_mask(A)
    A.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
    for alpha, beta, old in ((1.0, 0.0, None), (0.75, -0.5, dst)):
        _, ran = gu.check_prod(oracle, A, B, old, trans, alpha, beta, path, what)
        assert ran == path or path != 3                  # (3: the walking kernel)


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch", [
    (64, 20, 7, 1, 8, 33),       # one map to 8, transposed: seven of eight groups without rows
    (64, 9, 5, 8, 1, 64),        # walks of few tiles: ...
    (64, 8, 7, 4, 3, 70),        # ... one of as many tiles as the window has rows
    (128, 16, 3, 3, 4, 65),
    (64, 16, 5, 1, 16, 24),
])
@pytest.mark.parametrize("trans", ["n", "t"])
def test_walk_over_maps(oracle, px, py, fs, maps_in, maps_out, batch, trans):
    from cuv_amd import _lib, dia as D
    off = D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets()
    _check(oracle, off, px * py * maps_in, px * py * maps_out, batch, trans, _lib.PATH_WALK, "walk")


@pytest.mark.parametrize("shift", [64 * 40, -64 * 40, 64 * 200])
def test_walk_with_rows_that_meet_nothing(oracle, shift):
    """Rows before or behind every window row of the operand, up to all of them: their steps have no block."""
    from cuv_amd import _lib, workloads as W
    off = W.window_offsets(64, 7) + shift
    for trans in "nt":
        _check(oracle, off, 64 * 64, 64 * 64, 40, trans, _lib.PATH_WALK, "far window")
