"""The projection of a batch without columns: only the factor of the old values is left of the update."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,offsets", [(301, [-7, 0, 5]), (4096, [64 * dy + dx for dy in range(-2, 3) for dx in range(-2, 3)])])
@pytest.mark.parametrize("beta", [0.0, -1.5])
def test_scales_the_valid_slots_only(oracle, n, offsets, beta):
    import torch
    import _gpu_util as gu
    from cuv_amd import _lib, dia as D
    rng = np.random.default_rng(n)
    C = oracle.Dia(n, n, offsets, n + 3, 1)
    valid = oracle.valid_mask(C)
    C.vals[:] = rng.uniform(-1, 1, C.vals.size).astype(np.float32)
    if beta == 0.0:
        C.vals[valid] = np.nan                           # only written
    empty = torch.empty(0, n, device="cuda:0")
    for path in (_lib.PATH_AUTO, _lib.PATH_TILED):
        dev = gu.make_dev_dia(C)
        _lib.check(_lib.lib().cuvdia_set_path(path), "set_path")
        try:
            D.densedense_to_dia(dev, None, empty, empty, float("inf"), beta)
        finally:
            _lib.lib().cuvdia_set_path(_lib.PATH_AUTO)
        want = np.where(valid, np.float32(beta) * np.nan_to_num(C.vals), C.vals)
        np.testing.assert_array_equal(dev.pull(), want)
