"""The product of 13 x 13 windows with split operands on the matrix cores, against the oracle where it can go wrong: maps around
its strips of 16 positions and patches of 4 x 4, batches around its 64 columns, several maps, rows of bfloat16 numbers and not,
values that no sum of three bfloat16 numbers holds, graph replay, and the automatic choice on both sides of its rule."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(oracle, px, py, maps_in, maps_out, batch, trans, binary=False):
    from cuv_amd import dia as D
    rng = np.random.default_rng(px * py + batch)
    h, w = px * py * maps_in, px * py * maps_out
    A = oracle.Dia(h, w, D.filter_factory_float(px, py, 13, maps_in, maps_out).offsets(), max(h, w), 1)
    A.vals[:] = np.nan                                   # padding must never be read
    valid = oracle.valid_mask(A)
    A.vals[valid] = rng.uniform(-1, 1, int(valid.sum())).astype(np.float32)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    B = rng.uniform(-1, 1, (n_in, batch))
    B = np.asfortranarray((B > 0 if binary else B).astype(np.float32))
    return rng, A, B, np.asfortranarray(rng.uniform(-1, 1, (n_out, batch)).astype(np.float32))


def _split_ran():
    from cuv_amd import _lib
    return _lib.lib().cuvdia_last_kernel().startswith(b"spmm_split_kernel<13, 13")


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("px,py,maps_in,maps_out,batch,binary", [
    (32, 13, 1, 1, 1, False),     # one row of two strips; a last patch of one map row
    (33, 16, 1, 2, 63, True),     # the last strip moved up by 15 positions
    (47, 18, 2, 1, 64, False),
    (128, 9, 1, 1, 65, True),     # maps lower than the window; one unit of 8 strips
    (145, 31, 1, 1, 34, False),   # 10 strips: a unit of 8, and 2
    (36, 40, 3, 3, 130, False),
])
def test_sizes(oracle, px, py, maps_in, maps_out, batch, binary, trans):
    import _gpu_util as gu
    from cuv_amd import _lib
    _, A, B, dst = _case(oracle, px, py, maps_in, maps_out, batch, trans, binary)
    for beta in (0.0, -1.5):
        _, ran = gu.check_prod(oracle, A, B, dst if beta else None, trans, 0.75, beta, _lib.PATH_PLANE, "%d x %d" % (px, py))
        assert _split_ran() and ran == _lib.PATH_PLANE


@pytest.mark.parametrize("trans,maps_in,maps_out", [("n", 1, 1), ("t", 3, 2)])
@pytest.mark.parametrize("every,columns", [(5, slice(0, 1)), (7, slice(40, 70)), (40, slice(3, 70, 16))])
def test_bfloat16_rows_among_others(oracle, trans, maps_in, maps_out, every, columns):
    """Second and third parts are read and multiplied only in steps where some dense row has them: some map rows of some columns
    do, from step to step, from wave to wave, from map to map."""
    import _gpu_util as gu
    from cuv_amd import _lib
    rng, A, B, _ = _case(oracle, 36, 40, maps_in, maps_out, 70, trans, binary=True)
    other = np.flatnonzero(np.arange(B.shape[0]) // 36 % every == 1)
    B[other, columns] = rng.uniform(-1, 1, B[other, columns].shape).astype(np.float32)
    gu.check_prod(oracle, A, B, None, trans, 1.0, 0.0, _lib.PATH_PLANE, "every %d" % every)
    assert _split_ran()


@pytest.mark.parametrize("where", ["rows", "values", "both"])
def test_values_that_no_three_parts_hold(oracle, where):
    """Infinities and NaN reach the elements that have them in their sums and no others; small numbers keep all their bits."""
    import _gpu_util as gu
    from cuv_amd import _lib
    rng, A, B, _ = _case(oracle, 50, 30, 1, 2, 70, "n")
    valid = np.flatnonzero(oracle.valid_mask(A))
    if where != "values":
        B[rng.integers(0, B.shape[0], 40), rng.integers(0, 70, 40)] *= np.float32(2.0 ** -125)
    if where != "rows":
        A.vals[rng.choice(valid, 40)] *= np.float32(2.0 ** -125)
    gu.check_prod(oracle, A, B, None, "n", 1.0, 0.0, _lib.PATH_PLANE, where)
    assert _split_ran()
    if where != "values":
        B[rng.integers(0, B.shape[0], 3), rng.integers(0, 70, 3)] = [np.inf, -np.inf, np.nan]
    if where != "rows":
        A.vals[rng.choice(valid, 3)] = [np.inf, -np.inf, np.nan]
    with np.errstate(invalid="ignore"):
        ref = oracle.prod(A, B, None, "n")
    got, _ = gu.gpu_prod(A, B, None, "n", path=_lib.PATH_PLANE)
    fin = np.isfinite(ref)
    assert _split_ran() and 0 < fin.sum() < fin.size
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    A.vals[~np.isfinite(A.vals)] = 0
    B[~np.isfinite(B)] = 0
    assert np.all(np.abs(got[fin] - ref[fin]) <= gu.REL_TOL * oracle.prod_mag(A, B)[fin] + 1e-37)


def test_tiny_operands_on_both_sides(oracle):
    """Products of which one factor or the other is below 2^-110, beside none that are larger."""
    import _gpu_util as gu
    from cuv_amd import _lib
    _, A, B, _ = _case(oracle, 40, 20, 1, 1, 20, "t")
    for sa, sb in ((2.0 ** -115, 2.0 ** 100), (2.0 ** 100, 2.0 ** -115), (2.0 ** 60, 2.0 ** 60)):
        a, b = oracle.Dia(A.h, A.w, A.offsets, A.stride, 1), np.asfortranarray(B * np.float32(sb))
        a.vals[:] = A.vals * np.float32(sa)
        gu.check_prod(oracle, a, b, None, "t", 1.0, 0.0, _lib.PATH_PLANE, str(sa))
        assert _split_ran()


def test_graph_replay(oracle):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    _, A, B, _ = _case(oracle, 60, 40, 1, 1, 66, "n")
    dev, X = gu.make_dev_dia(A), D.to_device_colmajor(B)
    out = torch.empty_like(X)
    L = _lib.lib()
    _lib.check(L.cuvdia_set_path(_lib.PATH_PLANE), "set_path")
    try:
        D.prod(out, dev, X, "n")
        eager, g = out.clone(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            D.prod(out, dev, X, "n", sync=False)
    finally:
        L.cuvdia_set_path(_lib.PATH_AUTO)
    assert _split_ran()
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("px,py,maps_out,batch,act,taken", [
    (256, 256, 1, 256, "", True),
    (256, 256, 1, 256, "sigmoid", True),
    (512, 512, 1, 64, "", True),          # one column tile
    (96, 96, 1, 64, "", False),           # few workgroups
    (256, 256, 1, 24, "", False),         # most columns of a tile empty
    (256, 256, 1, 256, "sample", True),
])
def test_the_automatic_choice(px, py, maps_out, batch, act, taken):
    import torch
    from cuv_amd import _lib, dia as D
    m = D.filter_factory_float(px, py, 13, 1, maps_out).get_dia("cuda:0")
    m.vec.normal_()
    X = torch.rand((batch, m.w), device="cuda:0")
    out = torch.empty((batch, m.h), device="cuda:0")
    if act:
        D.prod_bias_act(out, m, X, "n", 1.0, 0.0, bias=torch.zeros(m.h, device="cuda:0"),
                        act=_lib.ACT_SIGMOID if act == "sigmoid" else _lib.ACT_SIGMOID_SAMPLE, seed=1)
    else:
        D.prod(out, m, X, "n")
    assert _split_ran() == taken
