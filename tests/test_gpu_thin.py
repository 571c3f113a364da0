"""The product kernel for few batch columns (rows along the lanes), against the oracle where it can go wrong: row counts
around its blocks of 64 and 256 rows, every chunk length, column counts that its column blocks do not divide, tables
that reach past both ends of the dense operand, and each of its launch shapes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dia(oracle, rng, h, w, offsets):
    A = oracle.Dia(h, w, offsets, max(h, w), 1)
    A.vals[:] = np.nan                                   # padding must never be read
    valid = oracle.valid_mask(A)
    A.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    return A


def _check(oracle, seed, h, w, offsets, batch, alpha, beta, kernel):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(seed)
    A = _dia(oracle, rng, h, w, offsets)
    for trans in ("n", "t"):
        n_in, n_out = (h, w) if trans == "t" else (w, h)
        B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
        dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32)) if beta else None
        gu.check_prod(oracle, A, B, dst, trans, alpha, beta, _lib.PATH_AUTO, "%dx%d %s batch %d" % (h, w, trans, batch))
        assert _lib.lib().cuvdia_last_kernel().decode().startswith(kernel)


@pytest.mark.parametrize("run", range(1, 14))
@pytest.mark.parametrize("rows", [3, 63, 64, 257, 1021])
def test_rows_runs_and_columns(oracle, run, rows):
    # a band of `run` diagonals, one of run - 1 (mixed lengths), and two that leave the matrix early at either end
    offsets = [d - run // 2 for d in range(run)] + [40 + d for d in range(max(run - 1, 1))] + [-rows + 2, rows - 2]
    offsets = sorted(set(offsets))
    for batch in (1, 2, 3, 7, 23):
        _check(oracle, 100 * run + rows + batch, rows, rows + 5, offsets, batch, 0.75, -1.5 if batch % 2 else 0.0, "spmm_thin_kernel")


@pytest.mark.parametrize("h,w,runs,batch,shape", [
    (300, 290, 20, 9, "2, 4>"),              # few rows, many chunks: 64 rows per workgroup
    (300, 290, 20, 1, "1, 4>"),
    (98307, 98301, 17, 5, "8, 1>"),          # eight columns per lane, four waves
    (33029, 33030, 65, 4, "4, 1>"),          # four columns per lane, sixteen waves
    (5000, 5003, 3, 14, "2, 1>"),
])
def test_launch_shapes(oracle, h, w, runs, batch, shape):
    offsets = [37 * (r - runs // 2) + d for r in range(runs) for d in range(3)]
    from cuv_amd import _lib
    _check(oracle, h + batch, h, w, offsets, batch, 1.0, 0.5, "spmm_thin_kernel<3, ")
    assert _lib.lib().cuvdia_last_kernel().decode().endswith(shape)


@pytest.mark.parametrize("trans", ["n", "t"])
def test_non_finite_values_and_sampling(oracle, trans):
    """An Inf or NaN of the dense operand reaches the rows that reference it and no other, chunks of mixed length
    included; the fused sample draws what the oracle draws."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(3)
    n, batch = 700, 13
    A = _dia(oracle, rng, n, n, list(range(-3, 4)) + [100, 101])
    B = np.asfortranarray(rng.uniform(-1, 1, (n, batch)).astype(np.float32))
    B[2, 5], B[300, 3], B[697, 12] = -np.inf, np.inf, np.nan
    with np.errstate(invalid="ignore"):
        ref = oracle.prod(A, B, None, trans)
    got, _ = gu.gpu_prod(A, B, None, trans)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    B = np.asfortranarray(rng.uniform(-1, 1, (n, batch)).astype(np.float32))
    bias = rng.uniform(-1, 1, n).astype(np.float32)
    p = oracle.prod_bias_act(A, B, None, trans, 1.0, 0.0, bias, True)
    u = oracle.sample_uniform(n, batch, 77)
    out = torch.empty(batch, n, device="cuda:0")
    D.prod_bias_act(out, gu.make_dev_dia(A), D.to_device_colmajor(B), trans, bias=torch.from_numpy(bias).cuda(),
                    act=_lib.ACT_SIGMOID_SAMPLE, seed=77)
    decided = np.abs(p.astype(np.float64) - u) > 1e-5
    assert np.array_equal(D.to_host_colmajor(out)[decided], oracle.rnd_binarize(p, u)[decided])


@pytest.mark.parametrize("px,k,maps_in,maps_out,batch,kernel", [
    (40, 7, 1, 1, 24, "spmm_thin_kernel<7"),             # 25 row tiles: few of them, whatever the batch up to ...
    (40, 7, 1, 1, 140, "spmm_thin_kernel<7"),            # 55 tiles' worth of columns
    (40, 7, 1, 1, 150, "spmm_tiled_kernel<7"),           # 59
    (64, 5, 3, 4, 70, "spmm_thin_kernel<5"),             # many tiles, 58 of 128 columns not there
    (64, 5, 3, 4, 128, "spmm_tiled_kernel<5"),           # all there
    (64, 13, 2, 2, 88, "spmm_thin_kernel<13"),           # runs longer than 5: up to 70 % there
    (64, 13, 2, 2, 92, "spmm_tiled_kernel<13"),
])
def test_automatic_choice_by_tiles_and_columns(oracle, px, k, maps_in, maps_out, batch, kernel):
    n = px * px
    offsets = sorted(m * n + dy * px + dx for m in range(1 - maps_in, maps_out)
                     for dy in range(-(k // 2), k - k // 2) for dx in range(-(k // 2), k - k // 2))
    _check(oracle, px + batch, n * maps_in, n * maps_out, offsets, batch, 0.75, 0.5 if batch % 4 else 0.0, kernel)


def _band_reference(vals, offsets, X, trans):
    """The product of an n x n matrix with few diagonals in float64, a diagonal at a time, and the sums of its |terms|."""
    import torch
    n = X.shape[1]
    out, mag = torch.zeros(X.shape, dtype=torch.float64, device=X.device), torch.zeros(X.shape, dtype=torch.float64, device=X.device)
    for d, k in enumerate(offsets):
        lo, hi = max(0, -k), min(n, n - k)               # rows of the matrix
        src, dst = (slice(lo, hi), slice(lo + k, hi + k)) if trans == "t" else (slice(lo + k, hi + k), slice(lo, hi))
        term = vals[d, lo:hi].double() * X[:, src].double()
        out[:, dst] += term
        mag[:, dst] += term.abs()
    return out, mag


@pytest.mark.parametrize("batch", [5, 40])
def test_operands_above_2_gib(batch):
    """Columns 2^26 and more floats apart: byte offsets pass 2^31 and 2^32 inside the batch."""
    import torch
    from cuv_amd import _lib, dia as D
    n, offsets = 4099, [-70, -3, -2, -1, 0, 1, 2, 64, 65]
    ld = ((1 << 26) + 4) * (8 if batch < 8 else 1)
    A = D.dev_dia_matrix_f(n, n, len(offsets), n, device="cuda:0")
    A.set_offsets(offsets)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(batch)
    A.vec.uniform_(-1, 1, generator=g)
    X, Y = (torch.empty(batch, ld, device="cuda:0")[:, :n] for _ in range(2))
    X.uniform_(-1, 1, generator=g)
    for trans in ("n", "t"):
        old = Y.uniform_(-1, 1, generator=g).clone()
        D.prod(Y, A, X, trans, "n", 1.0, 0.5)
        assert _lib.lib().cuvdia_last_kernel().decode().startswith("spmm_thin_kernel")
        ref, mag = _band_reference(A.vec.view(len(offsets), n), offsets, X, trans)
        assert torch.all((Y.double() - (ref + 0.5 * old)).abs() <= 1e-5 * (mag + 0.5 * old.abs()))


def test_values_above_2_gib():
    """2.2 GiB of values: diagonals 8 MiB apart, the last ones beyond 2^31 bytes."""
    import torch
    from cuv_amd import _lib, dia as D
    n, offsets = (1 << 21) + 3, [300 * r + d for r in range(-22, 22) for d in range(6)]
    A = D.dev_dia_matrix_f(n, n, len(offsets), n, device="cuda:0")
    assert A.vec.numel() * 4 > 1 << 31
    A.set_offsets(offsets)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(1)
    A.vec.uniform_(-1, 1, generator=g)
    X = torch.rand(4, n, generator=g, device="cuda:0")
    Y = torch.empty_like(X)
    for trans in ("n", "t"):
        D.prod(Y, A, X, trans, "n", 1.0, 0.0)
        assert _lib.lib().cuvdia_last_kernel().decode().startswith("spmm_thin_kernel")
        ref, mag = _band_reference(A.vec.view(len(offsets), n), offsets, X, trans)
        assert torch.all((Y.double() - ref).abs() <= 1e-5 * mag)


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch,trans,shape", [
    (40, 41, 5, 1, 1, 1, "n", "<5, 1, 1>"),          # a block of the generator for one column, ...
    (40, 41, 5, 1, 1, 7, "t", "<5, 2, 1>"),          # ... for one of two neighbours
    (31, 33, 7, 3, 4, 6, "n", "<7, 2, 4>"),
    (40, 41, 3, 1, 1, 6, "n", "<3, 2, 1>"),          # three waves: two columns of a row, the first or the third of a block
    (200, 163, 9, 1, 1, 7, "n", "<9, 4, 1>"),        # eight waves: two of a lane's four
    (231, 233, 9, 1, 1, 22, "t", "<9, 4, 1>"),       # four waves: a block whole; two columns at the end
    (117, 117, 5, 3, 4, 27, "n", "<5, 8, 1>"),       # three at the end
    (48, 48, 5, 1, 16, 4, "t", "<5, 4, 1>"),         # sixteen waves: one column
])
def test_sampled_exit_of_every_shape(oracle, px, py, fs, maps_in, maps_out, batch, trans, shape):
    """The sample of an element is the one its row, column and seed name, however many columns a thread takes."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(px + batch)
    h, w = px * py * maps_in, px * py * maps_out
    A = _dia(oracle, rng, h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets())
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
    bias = rng.uniform(-1, 1, n_out).astype(np.float32)
    u = oracle.sample_uniform(n_out, batch, 321)
    dev, Bd = gu.make_dev_dia(A), D.to_device_colmajor(B)
    L = _lib.lib()
    _lib.check(L.cuvdia_set_path(_lib.PATH_THIN), "set_path")
    try:
        for beta, b in ((0.0, bias), (0.5, None)):
            old = dst if beta else None
            p = oracle.prod_bias_act(A, B, old, trans, 0.25, beta, b, True)
            # a quarter (the sigmoid's steepest slope) of 1e-5 of the sum's terms, and the sigmoid's own rounding
            tol = 0.25 * gu.REL_TOL * (oracle.prod_mag(A, B, old, trans, 0.25, beta) + 1.0) + 3e-7
            out = torch.full((batch + 1, n_out + 3), -7.0, device="cuda:0")
            view = out[:batch, :n_out]
            view.copy_(D.to_device_colmajor(dst))
            D.prod_bias_act(view, dev, Bd, trans, 0.25, beta, bias=None if b is None else torch.from_numpy(b).cuda(),
                            act=_lib.ACT_SIGMOID_SAMPLE, seed=321)
            assert L.cuvdia_last_kernel().decode() == "spmm_thin_kernel" + shape
            decided = np.abs(p.astype(np.float64) - u) > tol
            assert decided.mean() > 0.99
            assert np.array_equal(D.to_host_colmajor(view)[decided], oracle.rnd_binarize(p, u)[decided])
            assert torch.all(out[:, n_out:] == -7.0) and torch.all(out[batch] == -7.0)
    finally:
        L.cuvdia_set_path(_lib.PATH_AUTO)
