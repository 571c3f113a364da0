"""The tile-by-tile product whose tiles are patches of the window's plane: widths, map rows and batches that do not divide, tables in
either order, operands that end inside a patch's window, both transposes, the fused exits, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # map width, output and input map rows, window, shift of its first row, batch
    (64, 64, 64, 7, 0, 64),
    (33, 37, 37, 7, 0, 190),         # the last patch of a row moved up by 31, one map row of four, 30 columns of 32
    (28, 30, 30, 5, 0, 250),         # maps narrower than a patch
    (9, 9, 9, 3, 0, 1500),           # a patch's window rows overlap
    (100, 32, 36, 5, 100 * 2 + 1, 129),
    (70, 48, 40, 7, -70 * 9, 129),   # patches that meet no dense row
    (34, 40, 40, 3, 3, 130),
    (224, 184, 184, 7, 0, 32),       # one column tile, where rows along the lanes would be taken otherwise
]


def _layer(oracle, rng, px, rows, rows_in, k, shift, trans, reverse):
    off = np.array([dy * px + dx for dy in range(-(k // 2), k // 2 + 1) for dx in range(-(k // 2), k // 2 + 1)], np.int32)
    off = off + shift if trans == "n" else off - shift
    if reverse:
        off = off[::-1].copy()
    h, w = (px * rows, px * rows_in) if trans == "n" else (px * rows_in, px * rows)
    A = oracle.Dia(h, w, off, max(h, w) + 5, 1)
    A.vals[:] = np.nan                                   # padding must never be read
    valid = oracle.valid_mask(A)
    A.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    return A


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("px,rows,rows_in,k,shift,batch", CASES)
def test_product(oracle, px, rows, rows_in, k, shift, batch, trans):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(px + batch)
    A = _layer(oracle, rng, px, rows, rows_in, k, shift, trans, batch % 2 == 1)
    B = np.asfortranarray(rng.uniform(-1, 1, (px * rows_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (px * rows, batch)).astype(np.float32))
    for alpha, beta, old in ((1.0, 0.0, None), (0.75, -0.5, dst)):
        _, ran = gu.check_prod(oracle, A, B, old, trans, alpha, beta, _lib.PATH_AUTO, "%d x %d" % (px, rows))
        assert ran == _lib.PATH_TILED and _lib.lib().cuvdia_last_kernel() == b"spmm_tiled_kernel<%d, false>" % k


@pytest.mark.parametrize("px,rows,rows_in,k,shift,batch", CASES[1:5])
def test_fused_exits_and_padded_destinations(oracle, px, rows, rows_in, k, shift, batch):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(px)
    n_out = px * rows
    A = _layer(oracle, rng, px, rows, rows_in, k, shift, "n", False)
    B = np.asfortranarray(rng.uniform(-1, 1, (px * rows_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
    bias = rng.uniform(-1, 1, n_out).astype(np.float32)
    u = oracle.sample_uniform(n_out, batch, 99)
    dev, Bd, bias_d = gu.make_dev_dia(A), D.to_device_colmajor(B), torch.from_numpy(bias).cuda()
    for beta, b in ((0.0, bias), (0.5, None), (0.5, bias)):
        old = dst if beta else None
        p = oracle.prod_bias_act(A, B, old, "n", 0.25, beta, b, True)
        # a quarter (the sigmoid's steepest slope) of 1e-5 of the sum's terms, and the sigmoid's own rounding
        tol = 0.25 * gu.REL_TOL * (oracle.prod_mag(A, B, old, "n", 0.25, beta) + 1.0) + 3e-7
        for act in (_lib.ACT_SIGMOID, _lib.ACT_SIGMOID_SAMPLE):
            out = torch.full((batch + 1, n_out + 3), -7.0, device="cuda:0")
            view = out[:batch, :n_out]
            view.copy_(D.to_device_colmajor(dst))
            D.prod_bias_act(view, dev, Bd, "n", 0.25, beta, bias=None if b is None else bias_d, act=act, seed=99)
            assert _lib.lib().cuvdia_last_kernel() == b"spmm_tiled_kernel<%d, true>" % k
            got = D.to_host_colmajor(view)
            if act == _lib.ACT_SIGMOID:
                assert np.all(np.abs(got.astype(np.float64) - p) <= tol)
            else:
                decided = np.abs(p.astype(np.float64) - u) > tol
                assert decided.mean() > 0.99 and np.array_equal(got[decided], oracle.rnd_binarize(p, u)[decided])
            assert torch.all(out[:, n_out:] == -7.0) and torch.all(out[batch] == -7.0)


@pytest.mark.parametrize("px,rows,rows_in,k,shift,batch", CASES[1:4])
def test_non_finite_values(oracle, px, rows, rows_in, k, shift, batch):
    """An infinity or a NaN reaches the results that use it and no other, in the interior and at both ends."""
    import _gpu_util as gu
    rng = np.random.default_rng(batch)
    n_in = px * rows_in
    for trans in "nt":
        A = _layer(oracle, rng, px, rows, rows_in, k, shift, trans, False)
        B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
        B[0, 5], B[n_in // 2, 3], B[n_in - 1, 12], B[n_in - 2, batch - 1] = -np.inf, np.inf, np.nan, np.inf
        with np.errstate(invalid="ignore"):
            ref = oracle.prod(A, B, None, trans)
        got, _ = gu.gpu_prod(A, B, None, trans)
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(got == np.inf, ref == np.inf)
        assert np.array_equal(got == -np.inf, ref == -np.inf)


@pytest.mark.parametrize("px,rows,rows_in,k,shift,batch", CASES[:7])
def test_operands_off_every_alignment(oracle, px, rows, rows_in, k, shift, batch):
    """Bases of the values, the dense rows, the destination and the bias off 16 bytes by 1 to 3 floats, columns of odd pitch with NaN
    between them, transposed and not, plain and with a sigmoid and a sample: each result, and nothing beside them."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(3 * px + batch)
    n_in, n_out = px * rows_in, px * rows
    u = oracle.sample_uniform(n_out, batch, 31)
    for trans in "nt":
        A = _layer(oracle, rng, px, rows, rows_in, k, shift, trans, trans == "t")
        B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
        dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
        bias = rng.uniform(-1, 1, n_out).astype(np.float32)
        dev = gu.make_dev_dia(A)
        vals = torch.full((dev.vec.numel() + 1,), float("nan"), device="cuda:0")
        vals[1:] = dev.vec
        dev.vec = vals[1:]
        X = torch.full((batch, n_in + 5), float("nan"), device="cuda:0")
        X[:, 3:3 + n_in] = D.to_device_colmajor(B)
        X, bias_d = X[:, 3:3 + n_in], torch.cat([torch.zeros(2), torch.from_numpy(bias)]).cuda()[2:]
        mag = oracle.prod_mag(A, B, dst, trans, 0.25, -0.5)
        for act in (_lib.ACT_NONE, _lib.ACT_SIGMOID, _lib.ACT_SIGMOID_SAMPLE):
            out = torch.full((batch, n_out + 7), -7.0, device="cuda:0")
            view = out[:, 1:1 + n_out]
            view.copy_(D.to_device_colmajor(dst))
            if act == _lib.ACT_NONE:
                D.prod(view, dev, X, trans, "n", 0.25, -0.5)
            else:
                D.prod_bias_act(view, dev, X, trans, 0.25, -0.5, bias=bias_d, act=act, seed=31)
            ran = _lib.lib().cuvdia_last_kernel()
            got = D.to_host_colmajor(view.contiguous()).astype(np.float64)
            if act == _lib.ACT_NONE:
                assert ran == b"spmm_tiled_kernel<%d, false>" % k
                assert np.all(np.abs(got - oracle.prod(A, B, dst, trans, 0.25, -0.5)) <= gu.REL_TOL * mag)
            else:
                p = oracle.prod_bias_act(A, B, dst, trans, 0.25, -0.5, bias, True).astype(np.float64)
                tol = 0.25 * gu.REL_TOL * (mag + 1.0) + 3e-7     # a quarter (the sigmoid's steepest slope) of the sum's, and its own rounding
                assert ran == b"spmm_tiled_kernel<%d, true>" % k
                if act == _lib.ACT_SIGMOID:
                    assert np.all(np.abs(got - p) <= tol)
                else:
                    decided = np.abs(p - u) > tol
                    assert decided.mean() > 0.99 and np.array_equal(got[decided], oracle.rnd_binarize(p.astype(np.float32), u)[decided])
            assert torch.all(out[:, 0] == -7.0) and torch.all(out[:, 1 + n_out:] == -7.0)


@pytest.mark.parametrize("px,rows,rows_in,k,shift,batch", [CASES[1], CASES[4]])
def test_capture_and_replay(oracle, px, rows, rows_in, k, shift, batch):
    """Added to old values, with a sample, transposed: a graph's replays against the eager calls, operands changed in between."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(px)
    dev = gu.make_dev_dia(_layer(oracle, rng, px, rows, rows_in, k, shift, "t", False))
    X, bias = torch.empty(batch, px * rows_in, device="cuda:0"), torch.randn(px * rows, device="cuda:0")
    plain, layer = torch.empty(batch, px * rows, device="cuda:0"), torch.empty(batch, px * rows, device="cuda:0")

    def calls():
        D.prod(plain, dev, X, "t", "n", 0.5, 0.25, sync=False)
        assert _lib.lib().cuvdia_last_kernel() == b"spmm_tiled_kernel<%d, false>" % k
        D.prod_bias_act(layer, dev, X, "t", bias=bias, act=_lib.ACT_SIGMOID_SAMPLE, seed=5, sync=False)
        assert _lib.lib().cuvdia_last_kernel() == b"spmm_tiled_kernel<%d, true>" % k

    def refill(i):
        X.copy_(torch.from_numpy(np.random.default_rng(i).uniform(-1, 1, tuple(X.shape)).astype(np.float32)))
        plain.fill_(0.5 + i)
        layer.fill_(-1.0)
    refill(0)
    calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls()
    for i in range(1, 5):
        refill(i)
        calls()
        eager = plain.clone(), layer.clone()
        refill(i)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(plain, eager[0]) and torch.equal(layer, eager[1])
