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


@pytest.mark.parametrize("run", [1, 5, 6, 7, 8, 9, 13])
@pytest.mark.parametrize("batch", [63, 64, 67, 255, 256, 259, 2048, 2049])     # (16 ranges from 256 to 2048, windows up to 8)
def test_four_columns_in_flight_and_sixteen_ranges(oracle, run, batch):
    offsets = sorted([d - run // 2 for d in range(run)] + [40 + d for d in range(max(run - 2, 1))])
    waves = 16 if run <= 8 and 256 <= batch <= 2048 else 8           # (a range each)
    columns = 2 if batch < 64 or (waves == 16 and run > 6) else 4    # (two steps of 4 in every range)
    _check(oracle, run + batch, 301, 299, offsets, batch, 0.9 if batch % 2 else 0.0, "dd2dia_rows_kernel<%d, %d, %d>" % (run, columns, waves))


def test_several_maps_on_aligned_operands_and_short_batches(oracle):
    # 14 chunks or more at a batch up to 64; a band of 160 rows; the plane's tiles of 64 positions not full
    win = [[m * 1024 + dy * 32 + dx for dy in range(-2, 3) for dx in range(-2, 3)] for m in range(3)]
    _check(oracle, 1, 1024, 3072, sum(win, []), 20, 0.9)
    _check(oracle, 2, 160 * 40, 160 * 40, [dy * 160 + dx for dy in range(-2, 3) for dx in range(-2, 3)], 40, 0.0)
    _check(oracle, 3, 1024, 3072, sum(win, []), 80, 0.9, "dd2dia_tiled_kernel")


OFFSETS = [d - 6 for d in range(13)] + [20 + d for d in range(12)] + [-250, 250]


@pytest.mark.parametrize("rows,lead,batch", [(257, 0, 1), (257, 3, 5), (1022, 1, 37), (1022, 6, 300), (255, 2, 1100)])
def test_padded_operands_with_nan_between_the_columns(oracle, rows, lead, batch):
    """Columns apart by more than their length, a base on no 16-byte boundary, and NaN in all that lies around the operands
    in the same allocations: the kernel's 16-byte loads reach into it."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(rows + batch)
    h, w = rows, rows + 6
    C = oracle.Dia(h, w, OFFSETS, w + 1, 1)
    valid = oracle.valid_mask(C)
    C.vals[:] = np.nan                                   # padding: neither read nor written
    C.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    host = [np.asfortranarray(rng.uniform(-1, 1, (r, batch)).astype(np.float32)) for r in (h, w)]
    views = []
    for m, pad in zip(host, (lead, 2 * lead + 1)):
        flat = torch.full(((batch + 2) * (m.shape[0] + pad) + 3,), float("nan"), device="cuda:0")
        view = flat[m.shape[0] + 1:][:batch * (m.shape[0] + pad)].view(batch, m.shape[0] + pad)[:, :m.shape[0]]
        view.copy_(D.to_device_colmajor(m))
        views.append(view)
    dev = gu.make_dev_dia(C)
    D.densedense_to_dia(dev, None, *views, 1.0 / batch, 0.9)
    assert _lib.lib().cuvdia_last_kernel().decode().startswith("dd2dia_rows_kernel")
    got, ref = dev.pull(), oracle.dd2dia_f64(C, *host, 1.0 / batch, 0.9)
    mag = oracle.dd2dia_f64(type(C)(h, w, C.offsets, C.stride, 1, np.abs(C.vals)), np.abs(host[0]), np.abs(host[1]), 1.0 / batch, 0.9)
    gu.assert_close_mag(got[valid], ref[valid], mag[valid], "padded")
    assert np.array_equal(got[~valid].view(np.uint32), C.vals[~valid].view(np.uint32))


@pytest.mark.parametrize("rows,batch", [(257, 3), (1022, 37), (255, 300)])
def test_non_finite_operands_reach_their_slots_only(oracle, rows, batch):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(rows)
    C = oracle.Dia(rows, rows + 6, OFFSETS, rows + 7, 1)
    valid = oracle.valid_mask(C)
    C.vals[:] = 0.0
    A = np.asfortranarray(rng.uniform(-1, 1, (rows, batch)).astype(np.float32))
    B = np.asfortranarray(rng.uniform(-1, 1, (rows + 6, batch)).astype(np.float32))
    A[0, 0], A[rows - 1, batch - 1], A[131, 1], B[0, 1], B[200, 2], B[rows + 5, 0] = np.inf, np.nan, -np.inf, np.nan, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        ref = oracle.dd2dia(C, A, B, 1.0, 0.0)
    got, _ = gu.gpu_dd2dia(C, A, B)
    assert _lib.lib().cuvdia_last_kernel().decode().startswith("dd2dia_rows_kernel")
    assert np.array_equal(np.isnan(got[valid]), np.isnan(ref[valid])) and np.array_equal(np.isinf(got[valid]), np.isinf(ref[valid]))
    assert np.array_equal(got[~valid], C.vals[~valid])


@pytest.mark.parametrize("n,offsets,ld,batch", [
    (4099, [-70, -3, -2, -1, 0, 1, 2, 64, 65], ((1 << 26) + 4) * 8, 5),      # columns 2 GiB apart
    (4099, [-70, -3, -2, -1, 0, 1, 2, 64, 65], (1 << 26) + 4, 40),           # operands of 10 GiB
    ((1 << 21) + 3, [300 * r + d for r in range(-22, 22) for d in range(6)], (1 << 21) + 3, 4),      # values of 2.2 GiB
])
def test_values_and_operands_above_2_gib(n, offsets, ld, batch):
    import torch
    from cuv_amd import _lib, dia as D
    C = D.dev_dia_matrix_f(n, n, len(offsets), n, device="cuda:0")
    C.set_offsets(offsets)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(n + batch)
    old = C.vec.uniform_(-1, 1, generator=g).clone().view(len(offsets), n)
    A, B = (torch.empty(batch, ld, device="cuda:0")[:, :n] for _ in range(2))
    A.uniform_(-1, 1, generator=g)
    B.uniform_(-1, 1, generator=g)
    D.densedense_to_dia(C, None, A, B, 1.0, 0.9)
    assert _lib.lib().cuvdia_last_kernel().decode().startswith("dd2dia_rows_kernel")
    got = C.vec.view(len(offsets), n)
    for d, k in enumerate(offsets):
        lo, hi = max(0, -k), min(n, n - k)
        term = A[:, lo:hi].double() * B[:, lo + k:hi + k].double()
        ref, mag = term.sum(0) + 0.9 * old[d, lo:hi], term.abs().sum(0) + 0.9 * old[d, lo:hi].abs()
        assert torch.all((got[d, lo:hi].double() - ref).abs() <= 1e-5 * mag), (d, k)
        assert torch.equal(got[d, :lo], old[d, :lo]) and torch.equal(got[d, hi:], old[d, hi:])
