"""The error against 64 bits of the kernels that multiply parts of fp32 numbers (13 x 13 windows), in sums of one product to many: each
product within its bound, none of the six products of parts missing, no bias, and the 2-norm beside the fp32 FMA chains' own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PX, BATCH = 64, 128
N = PX * PX
OFFSETS = [dy * PX + dx for dy in range(-6, 7) for dx in range(-6, 7)]


def _uniform(g, low, *shape):
    import torch
    return torch.rand(shape, generator=g, device="cuda:0") * (1 - low) + low


def _worst(x):
    """A third of the numbers each: 1 + 2^-7 - 2^-23, the largest rest behind 8 bits cut off; 0x3f807fc0, behind 8 rounded; as they are."""
    import torch
    i = torch.arange(x.numel(), device=x.device).view(x.shape) * 2654435761 % 2147483647 % 3
    x[i == 0] = 1 + 2.0 ** -7 - 2.0 ** -23
    x[i == 1] = float(np.uint32(0x3f807fc0).view(np.float32))
    return x


def _table():
    from cuv_amd import dia as D
    m = D.dev_dia_matrix_f(N, N, len(OFFSETS), N, 1)
    m.set_offsets(np.asarray(OFFSETS, np.int32))
    return m


def _product(vals, X, path):
    import torch
    from cuv_amd import _lib, dia as D
    L, m, out = _lib.lib(), _table(), torch.empty((X.shape[0], N), device="cuda:0")
    m.vec.copy_(vals.reshape(-1))
    _lib.check(L.cuvdia_set_path(path), "set_path")
    try:
        D.prod(out, m, X, "n")
    finally:
        L.cuvdia_set_path(_lib.PATH_AUTO)
    assert (path == _lib.PATH_PLANE) == L.cuvdia_last_kernel().startswith(b"spmm_split_kernel")
    return out.double()


def _gradient(A, B, path):
    from cuv_amd import _lib, dia as D
    L, m = _lib.lib(), _table()
    m.vec.zero_()
    _lib.check(L.cuvdia_set_path(path), "set_path")
    try:
        D.densedense_to_dia(m, D.dev_block_descriptor_f(m), A, B, 1.0, 0.0)
    finally:
        L.cuvdia_set_path(_lib.PATH_AUTO)
    assert (path == _lib.PATH_PLANE) == L.cuvdia_last_kernel().startswith(b"dd2dia_split_kernel")
    return m.vec.view(len(OFFSETS), N).double()


def _spans():
    for d, k in enumerate(OFFSETS):
        lo, hi = max(0, -k), N - max(0, k)
        yield d, k, slice(lo, hi), slice(lo + k, hi + k)


def _results(op, every, low, worst=False):
    """(exact result, the split kernel's, the fp32 chains'): product with rows that are 0 but for one in `every` x `every`
    positions, or gradient with `every` columns of a position that are not 0."""
    import torch
    from cuv_amd import _lib
    g = torch.Generator(device="cuda:0")
    g.manual_seed(every)
    if op == "product":
        vals, X = _uniform(g, low, len(OFFSETS), N), _uniform(g, low, BATCH, N)
        if worst:
            _worst(vals), _worst(X)
        i = torch.arange(N, device="cuda:0")
        X *= (i % PX % every == 0) & (i // PX % every == 0)
        ref = torch.zeros((BATCH, N), dtype=torch.float64, device="cuda:0")
        for d, k, rows, cols in _spans():
            ref[:, rows] += vals[d, rows].double() * X[:, cols].double()
        return ref, _product(vals, X, _lib.PATH_PLANE), _product(vals, X, _lib.PATH_TILED_NOWALK)
    A, B = _uniform(g, low, BATCH, N), _uniform(g, low, BATCH, N)
    if worst:
        _worst(A), _worst(B)
    A *= torch.rand((BATCH, N), generator=g, device="cuda:0").argsort(0) < every
    ref = torch.zeros((len(OFFSETS), N), dtype=torch.float64, device="cuda:0")
    for d, k, rows, cols in _spans():
        ref[d, rows] = (A[:, rows].double() * B[:, cols].double()).sum(0)
    return ref, _gradient(A, B, _lib.PATH_PLANE), _gradient(A, B, _lib.PATH_WINDOW)


@pytest.mark.parametrize("op,every", [("product", 16), ("gradient", 1)])
def test_one_product(op, every):
    """2^-24 of the product are left out; 2^-24 are cut off beside the first parts' product; the result is rounded (2^-24); the
    small parts' own roundings are 2^-8 of that.  A product of parts that is missing would be 2^-18 and more."""
    ref, got, _ = _results(op, every, -1.0, worst=True)
    assert ((got - ref).abs() <= 3.25 * 2.0 ** -24 * ref.abs()).all()


@pytest.mark.parametrize("op,every", [("product", 1), ("gradient", BATCH)])
def test_no_bias(op, every):
    """Sums of positive numbers: of a block's 16 products, 4 on average, the core cuts 2^-25 on average off where the small parts' sum
    meets the first ones'; what it rounds and what is left out has no sign."""
    ref, got, _ = _results(op, every, 0.0)
    assert abs((got - ref).sum().item()) <= 1.5e-8 * ref.sum().item()


@pytest.mark.parametrize("low", [-1.0, 0.0])
@pytest.mark.parametrize("op,every", [("product", e) for e in (16, 9, 7, 5, 3, 1)] + [("gradient", e) for e in (1, 2, 4, 8, 16, BATCH)])
def test_beside_the_fp32_chains(op, every, low):
    """A product is rounded once by a chain, and here where its parts meet (0.9 - 1.2 of that rounding's quadratic mean, with what is cut
    off) and, unless it is alone, where the blocks of a sum meet: 1.4 of one rounding.  A long sum has as many of either as
    it has blocks of 16 or 32, the chain as it has products: from 16 on it is the chain that is further off."""
    ref, got, chain = _results(op, every, low)
    assert (got - ref).norm() <= (1.0 if every in (3, 1) and op == "product" or every >= 16 and op == "gradient" else 1.4) * (chain - ref).norm()
