"""The plane's walk on 13 x 13 windows, which only the automatic choice takes (a forced one takes the kernel with split operands): the
smallest products it is chosen for, against 64 bits, with NaN wherever nothing may be read, and with infinities and NaN."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,py,maps_in,maps_out,batch,trans,beta", [
    (311, 320, 1, 1, 137, "t", 0.0),      # the last strip of 32 positions moved up by 9; a third column tile of 9
    (249, 278, 1, 1, 210, "n", -1.5),
    (302, 257, 4, 1, 70, "n", 0.0),       # four groups
    (259, 187, 2, 4, 65, "t", 0.5),       # ... and walks that change from map to map
])
def test_automatic_choice(px, py, maps_in, maps_out, batch, trans, beta):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    g = torch.Generator(device="cuda:0")
    g.manual_seed(px)
    m = D.filter_factory_float(px, py, 13, maps_in, maps_out).get_dia("cuda:0")
    offsets = D.filter_factory_float(px, py, 13, maps_in, maps_out).offsets().tolist()
    n_in, n_out = (m.h, m.w) if trans == "t" else (m.w, m.h)
    vals, X = m.vec.view(len(offsets), -1), torch.rand((batch, n_in + 4), device="cuda:0", generator=g)[:, :n_in]
    m.vec.fill_(float("nan"))
    spans = []
    for d, k in enumerate(offsets):
        rows = slice(max(0, -k), min(m.h, m.w - k))
        cols = slice(rows.start + k, rows.stop + k)
        vals[d, rows].normal_(0.0, 1.0, generator=g)
        spans.append((d, rows, cols) if trans == "n" else (d, cols, rows))

    def run(dst):
        out = dst.clone()
        D.prod(out, m, X, trans, "n", 0.75, beta)
        assert _lib.lib().cuvdia_last_kernel() == b"spmm_plane_kernel<13, 13, false>"
        return out

    def exact(dst, magnitude=False):
        out = torch.zeros((batch, n_out), dtype=torch.float64, device="cuda:0")
        for d, to, of in spans:
            v, x = vals[d, to if trans == "n" else of].double(), X[:, of].double()
            out[:, to] += v.abs() * x.abs() if magnitude else v * x
        return 0.75 * out + (abs(beta) * dst.double().abs() if magnitude else beta * dst.double()) if beta else 0.75 * out
    dst = torch.rand((batch, n_out), device="cuda:0", generator=g) if beta else torch.full((batch, n_out), float("nan"), device="cuda:0")
    assert ((run(dst).double() - exact(dst)).abs() <= gu.REL_TOL * exact(dst, True)).all()
    for at, value in zip((7, n_in // 2, n_in - 1), (float("inf"), -float("inf"), float("nan"))):
        X[at % batch, at] = value
    got, ref = run(dst), exact(dst)
    fin = ref.isfinite()
    assert not fin.all() and torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[ref.isinf()], ref[ref.isinf()].float())
    assert ((got.double() - ref).abs()[fin] <= gu.REL_TOL * exact(dst, True)[fin]).all()
