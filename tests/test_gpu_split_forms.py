"""The kernels that multiply parts of fp32 numbers (13 x 13 windows) on the forms their operands can take."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _offsets(px, rows, maps_in=1, maps_out=1, shift=0):
    return sorted(m * px * rows + dy * px + dx - shift for m in range(1 - maps_in, maps_out) for dy in range(-6, 7) for dx in range(-6, 7))


def _dia(h, w, offsets, stride=0):
    from cuv_amd import dia as D
    m = D.dev_dia_matrix_f(h, w, len(offsets), stride or max(h, w), 1)
    m.set_offsets(np.asarray(offsets, np.int32))
    m.vec.zero_()
    return m


def _forced(run, kernel):
    from cuv_amd import _lib
    L = _lib.lib()
    _lib.check(L.cuvdia_set_path(_lib.PATH_PLANE), "set_path")
    try:
        out = run()
    finally:
        L.cuvdia_set_path(_lib.PATH_AUTO)
    assert L.cuvdia_last_kernel().startswith(kernel)
    return out


def _in_columns(x, ld, lead, fill):
    """x, (batch, rows), with columns ld apart, `lead` numbers behind an allocation's start, `fill` wherever x is not."""
    import torch
    flat = torch.full((lead + x.shape[0] * ld + 8,), fill, device="cuda:0")
    view = flat[lead:lead + x.shape[0] * ld].view(x.shape[0], ld)[:, :x.shape[1]]
    view.copy_(x)
    return view


def _rand(seed, *shape):
    import torch
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return torch.rand(shape, generator=g, device="cuda:0") * 2 - 1


@pytest.mark.parametrize("fill", [float("nan"), 1e-40])
@pytest.mark.parametrize("px,rows,maps_in,maps_out,shift", [(68, 9, 1, 1, 2), (36, 20, 2, 1, 0), (60, 15, 1, 2, 3)])
def test_gradient_bits_do_not_depend_on_what_lies_between_the_columns(px, rows, maps_in, maps_out, shift, fill):
    """Tiles that reach over an end of the operands, whatever memory holds there."""
    import torch
    from cuv_amd import dia as D
    batch, out = 33, []
    h, w = px * rows * maps_in, px * rows * maps_out
    m = _dia(h, w, _offsets(px, rows, maps_in, maps_out, shift))
    bd, A, B = D.dev_block_descriptor_f(m), _rand(1, batch, h), _rand(2, batch, w)
    for between in (0.0, fill):
        a, b = _in_columns(A, h + 8, 0, between), _in_columns(B, w + 4, 4, between)
        m.vec.zero_()
        _forced(lambda: D.densedense_to_dia(m, bd, a, b, 0.5, 0.0), b"dd2dia_split_kernel")
        out.append(m.vec.clone())
    assert torch.equal(*out)


def test_price_of_numbers_that_no_three_parts_hold():
    """A product whose every step has them: 6 times an ordinary one's time as measured, and 66 times where each dense row of a column was
    fetched by itself."""
    import torch
    from cuv_amd import dia as D
    n_in, n_out, batch = 40000 * 2, 40000, 128
    m = _dia(n_out, n_in, _offsets(200, 200, 1, 2))
    m.vec.normal_()
    X, out, best = _rand(1, batch, n_in), torch.empty((batch, n_out), device="cuda:0"), []
    for tiny in (False, True):
        if tiny:
            X[::8] *= 2.0 ** -126
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        times = []
        for _ in range(4):
            e[0].record()
            _forced(lambda: D.prod(out, m, X, "n", sync=False), b"spmm_split_kernel")
            e[1].record()
            torch.cuda.synchronize()
            times.append(e[0].elapsed_time(e[1]))
        best.append(min(times))
    assert best[1] < 16 * best[0], best


def _spans(h, w, offsets):
    for d, k in enumerate(offsets):
        rows = slice(max(0, -k), min(h, w - k))
        if rows.stop > rows.start:
            yield d, rows, slice(rows.start + k, rows.stop + k)


def _exact_product(vals, X, h, w, offsets, trans):
    """(sums, sums of magnitudes) in 64 bits"""
    import torch
    out = [torch.zeros((X.shape[0], w if trans == "t" else h), dtype=torch.float64, device="cuda:0") for _ in range(2)]
    for d, rows, cols in _spans(h, w, offsets):
        to, of = (cols, rows) if trans == "t" else (rows, cols)
        term = vals[d, rows].double() * X[:, of].double()
        out[0][:, to] += term
        out[1][:, to] += term.abs()
    return out


@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("more,lead,pad_x,pad_y,descending", [
    (1, 0, 1, 5, False),         # value rows, columns at every remainder of 4 numbers
    (2, 1, 2, 0, True),
    (3, 2, 0, 3, False),
    (0, 3, 7, 2, True),
])
def test_product(more, lead, pad_x, pad_y, descending, trans):
    import torch
    import _gpu_util as gu
    from cuv_amd import dia as D
    px, rows, batch, beta = 50, 23, 37, -0.5
    h, w = px * rows, px * rows * 2
    offsets = _offsets(px, rows, 1, 2)[::-1 if descending else 1]
    m = _dia(h, w, offsets, max(h, w) + more)
    vals = m.vec.view(len(offsets), -1)
    m.vec.fill_(float("nan"))
    for i, (d, span, _) in enumerate(_spans(h, w, offsets)):
        vals[d, span] = _rand(100 + i, span.stop - span.start)
    n_in, n_out = (h, w) if trans == "t" else (w, h)
    X, Y = _rand(1, batch, n_in), _rand(2, batch, n_out)
    x, y = _in_columns(X, n_in + pad_x, lead, float("nan")), _in_columns(Y, n_out + pad_y, lead + 1, -7.0)
    whole = torch.as_strided(y, (batch * (n_out + pad_y) + lead + 9,), (1,), 0)
    _forced(lambda: D.prod(y, m, x, trans, "n", 0.75, beta), b"spmm_split_kernel")
    ref, mag = _exact_product(vals, X, h, w, offsets, trans)
    gu.assert_close_mag(y.cpu(), (0.75 * ref + beta * Y.double()).cpu(), (0.75 * mag + 0.5 * Y.double().abs()).cpu(), "product")
    y.fill_(-7.0)
    assert torch.all(whole == -7.0)                      # nothing was written beside the columns


@pytest.mark.parametrize("lead,descending", [(1, False), (2, True), (3, False), (0, True)])
def test_gradient(lead, descending):
    """A at every remainder of 16 bytes, columns apart, tables in either order; the padding keeps what it held."""
    import torch
    import _gpu_util as gu
    from cuv_amd import dia as D
    px, rows, batch = 44, 19, 37
    h, w = px * rows * 2, px * rows
    offsets = _offsets(px, rows, 2, 1)[::-1 if descending else 1]
    m = _dia(h, w, offsets)
    m.vec.fill_(float("nan"))
    vals, old = m.vec.view(len(offsets), -1), {}
    for d, span, _ in _spans(h, w, offsets):
        vals[d, span] = old[d] = _rand(200 + d, span.stop - span.start)
    A, B = _rand(3, batch, h), _rand(4, batch, w)
    a, b = _in_columns(A, h + 4, lead, float("nan")), _in_columns(B, w + 8, 4, float("nan"))
    _forced(lambda: D.densedense_to_dia(m, D.dev_block_descriptor_f(m), a, b, 0.5, 0.9), b"dd2dia_split_kernel")
    written = torch.zeros_like(vals, dtype=torch.bool)
    for d, span, cols in _spans(h, w, offsets):
        term = A[:, span].double() * B[:, cols].double()
        ref, mag = 0.5 * term.sum(0) + 0.9 * old[d].double(), 0.5 * term.abs().sum(0) + 0.9 * old[d].double().abs()
        assert ((vals[d, span].double() - ref).abs() <= gu.REL_TOL * mag).all()
        written[d, span] = True
    assert torch.all(vals[~written].isnan())


def test_gradient_graph_replay():
    import torch
    from cuv_amd import dia as D
    px, rows, batch = 64, 24, 50
    m = _dia(px * rows, px * rows, _offsets(px, rows))
    bd, A, B = D.dev_block_descriptor_f(m), _rand(5, batch, px * rows), _rand(6, batch, px * rows)
    _forced(lambda: D.densedense_to_dia(m, bd, A, B, 0.5, 0.0), b"dd2dia_split_kernel")
    eager, g = m.vec.clone(), torch.cuda.CUDAGraph()

    def capture():
        with torch.cuda.graph(g):
            D.densedense_to_dia(m, bd, A, B, 0.5, 0.0, sync=False)
    _forced(capture, b"dd2dia_split_kernel")
    for _ in range(3):
        m.vec.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(m.vec, eager)


@pytest.mark.parametrize("where", ["first", "second"])
@pytest.mark.parametrize("op", ["product", "gradient"])
def test_numbers_whose_nearest_bfloat16_number_is_infinite(op, where):
    """The largest fp32 numbers and the last one below them that bfloat16 rounds down, against small ones."""
    import torch
    import _gpu_util as gu
    from cuv_amd import dia as D
    px, rows, batch = 40, 24, 40
    n, offsets = px * rows, _offsets(px, rows)
    m = _dia(n, n, offsets)
    bd, vals, X, Y = D.dev_block_descriptor_f(m), _rand(7, len(offsets), n), _rand(8, batch, n), _rand(9, batch, n)
    first, second = (vals, X) if op == "product" else (X, Y)
    large, small = (first, second) if where == "first" else (second, first)
    small *= 2.0 ** -20
    bits = torch.tensor([0x7f7fffff, 0x7f7f8000, 0x7f7f7fff], dtype=torch.int32, device="cuda:0").view(torch.float32)
    large.view(-1)[::997] = bits[torch.arange(large.view(-1)[::997].numel(), device="cuda:0") % 3]
    if op == "product":
        m.vec.copy_(vals.view(-1))
        got = _forced(lambda: D.prod(torch.empty((batch, n), device="cuda:0"), m, X, "n"), b"spmm_split_kernel").double()
        ref, mag = _exact_product(vals, X, n, n, offsets, "n")
    else:
        _forced(lambda: D.densedense_to_dia(m, bd, X, Y, 1.0, 0.0), b"dd2dia_split_kernel")
        got = m.vec.view(len(offsets), n).double()
        ref, mag = torch.zeros_like(got), torch.zeros_like(got)
        for d, span, cols in _spans(n, n, offsets):
            term = X[:, span].double() * Y[:, cols].double()
            ref[d, span], mag[d, span] = term.sum(0), term.abs().sum(0)
    assert ((got - ref).abs() <= gu.REL_TOL * mag).all()
