"""The projection with rows along the lanes, against the oracle where it can go wrong: row counts around its blocks of 256
rows, both operands' ends inside a 16-byte load, every chunk length, batches around its steps and ranges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(oracle, seed, h, w, offsets, batch, beta, kernel="dd2dia_rows_kernel"):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(seed)
    C = oracle.Dia(h, w, offsets, max(h, w) + 1, 1)
    C.vals[:] = np.nan                                   # padding: neither read nor written
    valid = oracle.valid_mask(C)
    C.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32) if beta else np.nan
    A = np.asfortranarray(rng.uniform(-1, 1, (h, batch)).astype(np.float32))
    B = np.asfortranarray(rng.uniform(-1, 1, (w, batch)).astype(np.float32))
    if not beta:
        C.vals[valid] = 0.0
    gu.check_dd2dia(oracle, C, A, B, 1.0 / batch, beta, _lib.PATH_AUTO, "%dx%d batch %d" % (h, w, batch))
    assert _lib.lib().cuvdia_last_kernel().decode().startswith(kernel)


@pytest.mark.parametrize("run", range(1, 14))
@pytest.mark.parametrize("rows", [5, 255, 257, 1022])        # (no multiples of 4: the automatic choice at every batch)
def test_rows_runs_and_batches(oracle, run, rows):
    offsets = [d - run // 2 for d in range(run)] + [20 + d for d in range(max(run - 1, 1))] + [-rows + 2, rows - 2]
    for batch in (1, 2, 3, 16, 37):
        _check(oracle, run + rows + batch, rows, rows + 6, sorted(set(offsets)), batch, 0.9 if batch % 2 else 0.0)


@pytest.mark.parametrize("h,w,runs,batch", [
    (301, 2000, 5, 300),                     # eight ranges of the batch
    (303, 2000, 5, 1100),                    # ... each summed in blocks of columns
    (30001, 30003, 20, 70),                  # several rounds of waves, four ranges
    (70001, 69999, 60, 9),                   # one range
])
def test_ranges_of_the_batch(oracle, h, w, runs, batch):
    _check(oracle, h, h, w, [41 * (r - runs // 2) + d for r in range(runs) for d in range(3)], batch, 0.5)


def test_several_maps_on_aligned_operands_and_short_batches(oracle):
    # 14 chunks or more at a batch up to 64; a band of 160 rows; the plane's tiles of 64 positions not full
    win = [[m * 1024 + dy * 32 + dx for dy in range(-2, 3) for dx in range(-2, 3)] for m in range(3)]
    _check(oracle, 1, 1024, 3072, sum(win, []), 20, 0.9)
    _check(oracle, 2, 160 * 40, 160 * 40, [dy * 160 + dx for dy in range(-2, 3) for dx in range(-2, 3)], 40, 0.0)
    _check(oracle, 3, 1024, 3072, sum(win, []), 80, 0.9, "dd2dia_tiled_kernel")
