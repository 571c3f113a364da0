"""Powers of two on an operand of the kernels that multiply parts of fp32 numbers (13 x 13 windows): the parts, their products and sums
take the same power, so the result is the same but for it, bit for bit, at every size whose smallest parts are bfloat16 numbers."""
import pytest

pytestmark = pytest.mark.gpu

PX, BATCH = 64, 70


def _operands(seed, *shapes):
    import torch
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return [torch.rand(s, generator=g, device="cuda:0") * 2 - 1 for s in shapes]


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


@pytest.mark.parametrize("which", ["first", "second"])
@pytest.mark.parametrize("power", [-60, 17, 18, 20, 22, 24, 60])
@pytest.mark.parametrize("op", ["product", "gradient"])
def test_powers_of_two(op, power, which):
    import torch
    from cuv_amd import dia as D
    n, scale = PX * PX, 2.0 ** power
    m = D.filter_factory_float(PX, PX, 13, 1, 1).get_dia("cuda:0")
    bd = D.dev_block_descriptor_f(m)
    vals, X, Y = _operands(3, m.vec.shape, (BATCH, n), (BATCH, n))

    def run(a, b):
        if op == "product":
            m.vec.copy_(vals * a)
            return _forced(lambda: D.prod(torch.empty((BATCH, n), device="cuda:0"), m, X * b, "n"), b"spmm_split_kernel")
        m.vec.zero_()
        _forced(lambda: D.densedense_to_dia(m, bd, X * a, Y * b, 1.0, 0.0), b"dd2dia_split_kernel")
        return m.vec.clone()
    one = run(1.0, 1.0)
    assert torch.equal(run(scale, 1.0) if which == "first" else run(1.0, scale), one * scale)


@pytest.mark.parametrize("power", [-30, -55])
@pytest.mark.parametrize("op", ["product", "gradient"])
def test_products_next_to_the_smallest_numbers(op, power):
    """Both operands around 2^-30 and 2^-55: the products around 2^-110 and their parts' down to 2^-126 and below, where they are no
    normal numbers.  Against 64 bits: 2^-24 of each of at most 169 (70) terms for the roundings, and 2^-149 for each of their parts' six."""
    import torch
    from cuv_amd import dia as D
    n = PX * PX
    m = D.filter_factory_float(PX, PX, 13, 1, 1).get_dia("cuda:0")
    bd = D.dev_block_descriptor_f(m)
    vals, X, Y = (t * 2.0 ** power for t in _operands(4, m.vec.shape, (BATCH, n), (BATCH, n)))
    offsets = D.filter_factory_float(PX, PX, 13, 1, 1).offsets().tolist()
    table = lambda v: v.view(len(offsets), -1).double()
    spans = [(d, slice(max(0, -k), n - max(0, k)), slice(max(0, k), n + min(0, k))) for d, k in enumerate(offsets)]
    if op == "product":
        m.vec.copy_(vals)
        got = _forced(lambda: D.prod(torch.empty((BATCH, n), device="cuda:0"), m, X, "n"), b"spmm_split_kernel").double()
        ref, mag = torch.zeros_like(got), torch.zeros_like(got)
        for d, rows, cols in spans:
            term = table(vals)[d, rows] * X[:, cols].double()
            ref[:, rows] += term
            mag[:, rows] += term.abs()
    else:
        m.vec.zero_()
        _forced(lambda: D.densedense_to_dia(m, bd, X, Y, 1.0, 0.0), b"dd2dia_split_kernel")
        got = table(m.vec).clone()
        ref, mag = torch.zeros_like(got), torch.zeros_like(got)
        for d, rows, cols in spans:
            term = X[:, rows].double() * Y[:, cols].double()
            ref[d, rows], mag[d, rows] = term.sum(0), term.abs().sum(0)
    assert ((got - ref).abs() <= 169 * 2.0 ** -24 * mag + 169 * 6 * 2.0 ** -149).all()
