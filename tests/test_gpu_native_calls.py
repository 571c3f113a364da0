"""The direct calls into the library (cuv_amd/_native) and the wait they end with: same results as the general way through
ctypes, on the default and on other streams, from several threads at once; unusual operands take the general way."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layer(seed, px=40, batch=30):
    import torch
    from cuv_amd import dia as D
    A = D.filter_factory_float(px, px, 5, 1, 1).get_dia(device="cuda:0")
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    A.vec.normal_(generator=g)
    A.desc
    X = torch.rand(batch, px * px, generator=g, device="cuda:0")
    return A, X, torch.zeros(batch, px * px, device="cuda:0")


@pytest.mark.parametrize("sync", [True, False])
@pytest.mark.parametrize("trans", ["n", "t"])
def test_same_as_through_ctypes(monkeypatch, trans, sync):
    import torch
    from cuv_amd import dia as D
    A, X, Y = _layer(1)
    G = D.filter_factory_float(40, 40, 5, 1, 1).get_dia(device="cuda:0")
    W, M = torch.rand(1000, device="cuda:0"), torch.rand(1000, device="cuda:0")
    bias = torch.rand(1600, device="cuda:0")
    results = []
    for direct in (True, False):
        taken = []
        if not direct:
            for name in ("product", "projection", "weight_step"):
                monkeypatch.setattr(D._native, name, lambda *a: taken.append(1) or False)
        G.desc
        G.vec.zero_()
        w, m = W.clone(), M.clone()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            D.prod(Y, A, X, trans, "n", 0.5, 0.0, sync=sync)
            Z = D.prod_bias_act(torch.empty_like(Y), A, Y, trans, bias=bias, act=1, sync=sync)
            D.densedense_to_dia(G, None, Y, Z, 0.1, 0.0, sync=sync)
            D.learn_step_weight_decay_momentum(w, m, M, 0.1, 0.9, 0.01, sync=sync)
            D.learn_step_weight_decay(w, M, 0.1, 0.01, sync=sync)
            results.append([t.clone() for t in (Y, Z, G.vec, w, m)])
        torch.cuda.current_stream().wait_stream(s)
        assert len(taken) == (0 if direct else 5)
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_unusual_operands_are_left_to_the_general_way():
    import torch
    from cuv_amd import dia as D
    A, X, Y = _layer(2)
    call = D._native.product
    assert call(Y, A, X, "n", 1.0, 0.0, None, 0, 0, True) is True
    for args in ((Y, A, X[:, :-1], "n"), (Y[:-1], A, X, "n"), (Y, A, X.double(), "n"), (Y, A, X.cpu(), "n"), (Y, A, X, "x"),
                 (Y, A, X[:1].expand(30, -1), "n"), (Y, None, X, "n"), (None, A, X, "n")):
        assert call(*args, 1.0, 0.0, None, 0, 0, True) is False
    with pytest.raises(RuntimeError):
        D.prod(Y[:-1], A, X)


def test_waiting_in_several_threads():
    import torch
    from cuv_amd import dia as D
    bad = []

    def work(seed):
        A, X, Y = _layer(seed)
        want = D.prod(Y, A, X).clone()
        host = torch.empty(Y.shape, pin_memory=True)
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            for _ in range(50):
                Y.zero_()
                D.prod(Y, A, X)
                host.copy_(Y, non_blocking=True)
                s.synchronize()
                if not np.array_equal(host.numpy(), want.cpu().numpy()):
                    bad.append(seed)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
