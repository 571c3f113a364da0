"""The product that walks the window's plane on the matrix cores, against the oracle: every window it is built for, both
transposes, maps whose width its tiles of 32 positions do not divide, several groups, ragged batches, a destination that is
read, bias / sigmoid / sample at the tiles' exit, non-finite operands, padded leading dimensions, graph replay."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [                    # (px, py, window, maps in, maps out, batch)
    (37, 40, 5, 1, 1, 70),
    (75, 23, 5, 3, 4, 33),    # several groups; 3 tiles of 32 positions, the last moved up
    (32, 50, 7, 1, 1, 64),
    (150, 20, 8, 2, 1, 40),
    (41, 33, 9, 2, 2, 129),
    (100, 37, 11, 1, 2, 30),
    (33, 60, 13, 1, 1, 24),
    (64, 31, 13, 2, 1, 64),
]


def _case(oracle, seed, px, py, fs, maps_in, maps_out, batch, trans):
    from cuv_amd import dia as D
    rng = np.random.default_rng(seed)
    h, w = px * py * maps_in, px * py * maps_out
    A = oracle.Dia(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets(), max(h, w), 1)
    A.vals[:] = np.nan                                   # padding must never be read
    valid = oracle.valid_mask(A)
    A.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    B = np.asfortranarray(rng.uniform(-1, 1, (n_in, batch)).astype(np.float32))
    dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))
    return rng, A, B, dst


@pytest.fixture
def plane():
    from cuv_amd import _lib
    L = _lib.lib()
    _lib.check(L.cuvdia_set_path(_lib.PATH_PLANE), "set_path")
    yield L
    L.cuvdia_set_path(_lib.PATH_AUTO)


def _ran():
    from cuv_amd import _lib
    return _lib.lib().cuvdia_last_path() == _lib.PATH_PLANE


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_windows_maps_and_batches(oracle, shape, trans):
    import _gpu_util as gu
    from cuv_amd import _lib
    _, A, B, dst = _case(oracle, sum(shape), *shape, trans)
    for beta in (0.0, -1.5):
        _, ran = gu.check_prod(oracle, A, B, dst if beta else None, trans, 0.75, beta, _lib.PATH_PLANE, str(shape))
        assert ran == _lib.PATH_PLANE


@pytest.mark.parametrize("trans", ["n", "t"])
def test_bias_sigmoid_sample_and_non_finite_values(oracle, plane, trans):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng, A, B, dst = _case(oracle, 5, 35, 40, 9, 1, 1, 70, trans)
    n, batch = dst.shape
    bias = rng.uniform(-1, 1, n).astype(np.float32)
    dev, Bd, bd = gu.make_dev_dia(A), D.to_device_colmajor(B), torch.from_numpy(bias).cuda()
    for beta in (0.0, 0.5):
        p = oracle.prod_bias_act(A, B, dst if beta else None, trans, 1.0, beta, bias, True)
        out = D.to_device_colmajor(dst)
        D.prod_bias_act(out, dev, Bd, trans, 1.0, beta, bias=bd, act=_lib.ACT_SIGMOID)
        assert _ran()
        np.testing.assert_allclose(D.to_host_colmajor(out), p, rtol=0, atol=2e-5)
        out = D.to_device_colmajor(dst)
        D.prod_bias_act(out, dev, Bd, trans, 1.0, beta, bias=bd, act=_lib.ACT_SIGMOID_SAMPLE, seed=99)
        u = oracle.sample_uniform(n, batch, 99)
        decided = np.abs(p.astype(np.float64) - u) > 5e-5
        assert _ran() and np.array_equal(D.to_host_colmajor(out)[decided], oracle.rnd_binarize(p, u)[decided])
    for r, c, v in ((3, 5, -np.inf), (n // 2, 0, np.inf), (n - 2, 69, np.nan), (777, 33, np.nan)):
        B[r, c] = v
    with np.errstate(invalid="ignore"):
        ref = oracle.prod(A, B, None, trans)
    got, ran = gu.gpu_prod(A, B, None, trans, path=_lib.PATH_PLANE)
    assert ran == _lib.PATH_PLANE and np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))


def test_padded_operands_and_graph_replay(oracle, plane):
    import torch
    import _gpu_util as gu
    from cuv_amd import dia as D
    _, A, B, _ = _case(oracle, 6, 45, 40, 8, 1, 1, 66, "n")
    n, batch = B.shape
    dev = gu.make_dev_dia(A)
    X = torch.full((batch + 1, n + 7), float("nan"), device="cuda:0")
    X[:batch, :n] = D.to_device_colmajor(B)
    out = torch.full((batch + 2, n + 3), -7.0, device="cuda:0")
    view = out[1:batch + 1, :n]
    D.prod(view, dev, X[:batch, :n], "n")
    assert _ran()
    gu.assert_close_mag(D.to_host_colmajor(view), oracle.prod(A, B), oracle.prod_mag(A, B), "padded")
    assert torch.all(out[:, n:] == -7.0) and torch.all(out[0] == -7.0) and torch.all(out[batch + 1] == -7.0)
    eager = view.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        D.prod(view, dev, X[:batch, :n], "n", sync=False)
    for _ in range(3):
        view.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(view, eager)


def test_the_automatic_choice_takes_it_for_large_products(oracle):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    A = oracle.Dia(75 * 1500, 75 * 1500, D.filter_factory_float(75, 1500, 8, 1, 1).offsets(), 75 * 1500, 1)
    A.vals[:] = np.random.default_rng(7).uniform(-1, 1, A.vals.shape)
    dev, B = gu.make_dev_dia(A), torch.rand((130, A.w), device="cuda:0")
    out, ref = torch.empty_like(B), torch.empty_like(B)
    L = _lib.lib()
    D.prod(out, dev, B, "n")
    assert L.cuvdia_last_path() == _lib.PATH_PLANE
    _lib.check(L.cuvdia_set_path(_lib.PATH_TILED_NOWALK), "set_path")
    try:
        D.prod(ref, dev, B, "n")
    finally:
        L.cuvdia_set_path(_lib.PATH_AUTO)
    torch.testing.assert_close(out, ref, rtol=1e-5, atol=2e-5)


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_fused_exit_of_every_window(oracle, plane, shape, trans):
    """Bias, sigmoid and sample of every window the kernel is built for, into a destination that is read or only written."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng, A, B, dst = _case(oracle, 17 + sum(shape), *shape, trans)
    n, batch = dst.shape
    bias = rng.uniform(-1, 1, n).astype(np.float32)
    dev, Bd, bd = gu.make_dev_dia(A), D.to_device_colmajor(B), torch.from_numpy(bias).cuda()
    for beta in (0.0, 0.5):
        old = dst if beta else None
        p = oracle.prod_bias_act(A, B, old, trans, 0.25, beta, bias, True)
        # a quarter (the sigmoid's steepest slope) of 1e-5 of the sum's terms, and the sigmoid's own rounding
        tol = 0.25 * gu.REL_TOL * (oracle.prod_mag(A, B, old, trans, 0.25, beta) + np.abs(bias)[:, None]) + 3e-7
        out = D.to_device_colmajor(dst if beta else np.full_like(dst, np.nan))
        D.prod_bias_act(out, dev, Bd, trans, 0.25, beta, bias=bd, act=_lib.ACT_SIGMOID)
        assert _ran() and _lib.lib().cuvdia_last_kernel().decode().endswith("true>")
        assert np.all(np.abs(D.to_host_colmajor(out).astype(np.float64) - p) <= tol)
        out = D.to_device_colmajor(dst if beta else np.full_like(dst, np.nan))
        D.prod_bias_act(out, dev, Bd, trans, 0.25, beta, bias=bd, act=_lib.ACT_SIGMOID_SAMPLE, seed=5)
        u = oracle.sample_uniform(n, batch, 5)
        decided = np.abs(p.astype(np.float64) - u) > tol
        assert _ran() and np.array_equal(D.to_host_colmajor(out)[decided], oracle.rnd_binarize(p, u)[decided])
    out = D.to_device_colmajor(dst)
    D.prod_bias_act(out, dev, Bd, trans, 0.25, 0.5, bias=bd)                   # a bias alone
    ref = oracle.prod(A, B, dst, trans, 0.25, 0.5) + bias[:, None]
    gu.assert_close_mag(D.to_host_colmajor(out), ref, oracle.prod_mag(A, B, dst, trans, 0.25, 0.5) + np.abs(bias)[:, None], str(shape))


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch", [
    (150, 61, 7, 1, 2, 70),   # 5 walks of 32 positions: one unit of 4, and 1
    (262, 40, 7, 2, 1, 76),   # 9 walks: two units of 4, and 1
    (190, 50, 8, 1, 1, 130),  # 6: 4 and 2, three column tiles
    (200, 45, 5, 2, 2, 65),   # 7: 4 and 3
])
def test_walks_that_units_of_four_do_not_divide(oracle, px, py, fs, maps_in, maps_out, batch):
    import _gpu_util as gu
    from cuv_amd import _lib
    _, A, B, dst = _case(oracle, px + py, px, py, fs, maps_in, maps_out, batch, "t")
    _, ran = gu.check_prod(oracle, A, B, dst, "t", 1.0, 0.5, _lib.PATH_PLANE, "%d x %d" % (px, py))
    assert ran == _lib.PATH_PLANE


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch", [
    (40, 33, 7, 1, 9, 66),    # a map row of 9 groups' tables meets one or two of them
    (64, 20, 5, 9, 1, 40),
    (36, 10, 9, 5, 4, 33),    # maps hardly taller than the window
    (34, 8, 7, 3, 3, 65),
])
def test_groups_that_a_segment_does_not_meet(oracle, px, py, fs, maps_in, maps_out, batch, trans):
    import _gpu_util as gu
    from cuv_amd import _lib
    _, A, B, dst = _case(oracle, px + py, px, py, fs, maps_in, maps_out, batch, trans)
    _, ran = gu.check_prod(oracle, A, B, dst, trans, 1.0, 0.5, _lib.PATH_PLANE, "%d x %d" % (px, py))
    assert ran == _lib.PATH_PLANE


@pytest.mark.parametrize("h,w,offsets", [
    (40 * 200, 40 * 20, [0]),                  # a map that ends long before the rows do
    (40 * 150, 40 * 150, [-40 * 90, 40 * 90]), # two maps with nothing between them
])
def test_rows_that_no_group_reaches(oracle, h, w, offsets):
    import _gpu_util as gu
    from cuv_amd import _lib
    rng = np.random.default_rng(h + w)
    window = [o + 40 * dy + dx for o in offsets for dy in range(-3, 4) for dx in range(-3, 4)]
    A = oracle.Dia(h, w, window, h, 1)
    A.vals[:] = rng.uniform(-1, 1, A.vals.shape).astype(np.float32)
    for trans in ("n", "t"):
        n_in, n_out = (h, w) if trans == "t" else (w, h)
        B = np.asfortranarray(rng.uniform(-1, 1, (n_in, 66)).astype(np.float32))
        dst = np.asfortranarray(rng.uniform(-1, 1, (n_out, 66)).astype(np.float32))
        gu.check_prod(oracle, A, B, dst, trans, 1.0, 0.5, _lib.PATH_PLANE, str((h, w, trans)))


@pytest.mark.parametrize("trans", ["n", "t"])
def test_as_many_groups_as_a_table_has(oracle, plane, trans):
    """51 groups of 5 window rows: the last of the chunks' starts."""
    import _gpu_util as gu
    from cuv_amd import _lib
    _, A, B, dst = _case(oracle, 5, 32, 6, 5, 26, 26, 25, trans)
    for alpha, beta, old in ((1.0, 0.0, None), (0.75, -0.5, dst)):
        _, ran = gu.check_prod(oracle, A, B, old, trans, alpha, beta, _lib.PATH_PLANE, "51 groups")
        assert ran == _lib.PATH_PLANE


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("act", ["plain", "bias", "sigmoid", "sample"])
@pytest.mark.parametrize("shape", [SHAPES[i] for i in (0, 1, 2, 3, 4, 5)], ids=lambda s: "x".join(map(str, s)))
def test_padded_destination_that_is_read(oracle, plane, shape, act, trans):
    """Old values and results go by 32-bit offsets from the destination's columns, apart by more than their length and on no 16-byte
    boundary: what lies between and around them stays, and none of it is read."""
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng, A, B, dst = _case(oracle, 29 + sum(shape), *shape, trans)
    n, batch = dst.shape
    bias = rng.uniform(-1, 1, n).astype(np.float32) if act != "plain" else None
    code = {"sigmoid": _lib.ACT_SIGMOID, "sample": _lib.ACT_SIGMOID_SAMPLE}.get(act, _lib.ACT_NONE)
    dev = gu.make_dev_dia(A)
    X = torch.full((batch + 1, B.shape[0] + 5), float("nan"), device="cuda:0")
    X[:batch, 1:B.shape[0] + 1] = D.to_device_colmajor(B)
    out = torch.full((batch + 2, n + 7), float("nan"), device="cuda:0")
    view = out[1:batch + 1, 3:n + 3]
    view.copy_(D.to_device_colmajor(dst))
    D.prod_bias_act(view, dev, X[:batch, 1:B.shape[0] + 1], trans, 0.25, 0.5, bias=None if bias is None else torch.from_numpy(bias).cuda(),
                    act=code, seed=11)
    assert _ran()
    got = D.to_host_colmajor(view)
    mag = oracle.prod_mag(A, B, dst, trans, 0.25, 0.5) + (0 if bias is None else np.abs(bias)[:, None])
    if code == _lib.ACT_NONE:
        gu.assert_close_mag(got, oracle.prod(A, B, dst, trans, 0.25, 0.5) + (0 if bias is None else bias[:, None]), mag, "padded")
    else:
        p = oracle.prod_bias_act(A, B, dst, trans, 0.25, 0.5, bias, True)
        tol = 0.25 * gu.REL_TOL * mag + 3e-7         # (the sigmoid's steepest slope, and its own rounding)
        if act == "sample":
            u = oracle.sample_uniform(n, batch, 11)
            decided = np.abs(p.astype(np.float64) - u) > tol
            assert decided.mean() > 0.99 and np.array_equal(got[decided], oracle.rnd_binarize(p, u)[decided])
        else:
            assert np.all(np.abs(got.astype(np.float64) - p) <= tol)
    assert torch.isnan(out[0]).all() and torch.isnan(out[batch + 1]).all() and torch.isnan(out[1:-1, :3]).all() and torch.isnan(out[1:-1, n + 3:]).all()
