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
