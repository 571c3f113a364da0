"""The automatic choice of the plane's walk on either side of its lines, its result and the tile-by-tile
kernel's against 64 bits."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,py,fs,maps_in,maps_out,batch,trans,fused,taken", [
    (282, 282, 7, 2, 5, 128, "n", False, True),
    (282, 282, 7, 2, 5, 128, "n", True, False),       # with a bias and a sigmoid 7 x 7 have the lower line
    (282, 282, 7, 2, 5, 70, "n", False, False),       # most of the second column tile is empty
    (517, 517, 5, 3, 5, 64, "n", False, True),        # one column tile
    (300, 620, 11, 2, 1, 192, "t", True, True),
])
def test_well_filled_tiles(px, py, fs, maps_in, maps_out, batch, trans, fused, taken):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    m = D.filter_factory_float(px, py, fs, maps_in, maps_out).get_dia("cuda:0")
    g = torch.Generator(device="cuda:0")
    g.manual_seed(1)
    m.vec.normal_(0.0, 0.1, generator=g)
    n_in, n_out = (m.h, m.w) if trans == "t" else (m.w, m.h)
    X = torch.rand((batch, n_in), device="cuda:0", generator=g)
    bias = torch.rand(n_out, device="cuda:0", generator=g)
    L, out = _lib.lib(), []
    for path in (_lib.PATH_AUTO, _lib.PATH_TILED_NOWALK):
        _lib.check(L.cuvdia_set_path(path), "set_path")
        try:
            y = torch.full((batch, n_out), float("nan"), device="cuda:0")
            if fused:
                D.prod_bias_act(y, m, X, trans, 1.0, 0.0, bias=bias, act=_lib.ACT_SIGMOID)
            else:
                D.prod(y, m, X, trans)
        finally:
            L.cuvdia_set_path(_lib.PATH_AUTO)
        if path == _lib.PATH_AUTO:
            assert (L.cuvdia_last_path() == _lib.PATH_PLANE) == taken
        out.append(y)
    ref, mag = (torch.zeros((batch, n_out), dtype=torch.float64, device="cuda:0") for _ in range(2))
    offsets = D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets().tolist()
    vals = m.vec.view(len(offsets), -1)
    for d, k in enumerate(offsets):
        rows = slice(max(0, -k), min(m.h, m.w - k))
        cols = slice(rows.start + k, rows.stop + k)
        to, of = (cols, rows) if trans == "t" else (rows, cols)
        term = vals[d, rows].double() * X[:, of].double()
        ref[:, to] += term
        mag[:, to] += term.abs()
    tol = gu.REL_TOL * mag
    if fused:                                            # a sigmoid's slope is 1/4 at most; itself within 8 units of the last place
        ref, tol = torch.sigmoid(ref + bias.double()), tol / 4 + 2.0 ** -21
    for y in out:
        assert ((y.double() - ref).abs() <= tol).all()
