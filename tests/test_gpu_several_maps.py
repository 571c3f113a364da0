"""Products of layers with several maps, whose tiles meet a few of the table's window rows: the walking kernel's blocks without
dense rows, and the tile-by-tile kernel's range of chunks at the operand's ends, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(oracle, offsets, h, w, batch, trans, path, what):
    import _gpu_util as gu
    from cuv_amd import _lib
    kernel, ran_path = (b"spmm_walk_kernel", _lib.PATH_WALK) if path == _lib.PATH_WALK else (b"spmm_tiled_kernel", _lib.PATH_TILED)
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
        assert ran == ran_path and _lib.lib().cuvdia_last_kernel().startswith(kernel)


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


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch", [
    (29, 27, 7, 1, 8, 33),       # odd rows; one group of eight, or two, per tile: odd and even numbers of chunks
    (28, 20, 5, 1, 4, 64),       # rows that are multiples of 4, chunks of up to 8: few tiles come here
    (33, 15, 11, 4, 4, 65),      # chunks longer than 8
    (32, 12, 13, 2, 3, 24),
    (31, 9, 9, 8, 1, 70),        # 72 chunks: the larger table
    (7, 7, 3, 16, 16, 30),       # every chunk of a tile crosses an end
])
@pytest.mark.parametrize("trans", ["n", "t"])
def test_tiles_at_the_ends(oracle, px, py, fs, maps_in, maps_out, batch, trans):
    from cuv_amd import _lib, dia as D
    off = D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets()
    _check(oracle, off, px * py * maps_in, px * py * maps_out, batch, trans, _lib.PATH_TILED_NOWALK, "ends")


def test_mixed_chunks_at_the_ends(oracle):
    """Chunks of 3, 7 and 10 diagonals, two of them outside for most rows; and rows that meet none."""
    from cuv_amd import _lib
    off = np.concatenate([np.arange(-900, -893), np.arange(-4, -1), np.arange(5, 15), np.arange(800, 807)])
    for trans in "nt":
        _check(oracle, off, 1001, 777, 48, trans, _lib.PATH_TILED_NOWALK, "mixed")
        _check(oracle, off + 1500, 2001, 777, 48, trans, _lib.PATH_TILED_NOWALK, "mixed, far")
