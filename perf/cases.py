"""The work whose time matters to a user of this library, as cases a timing program can run.

A locally connected layer is a DIA matrix whose offset table is a window on a map (`filter_factory_float`).  Programs
call three operations on it -- the product with a batch of dense columns in both transposes (`prod`, or with bias,
sigmoid and Bernoulli sample fused: `prod_bias_act`), and the weight gradient (`densedense_to_dia`) -- one at a time,
as an inference server or a script does (the default, which waits for the result), or queued one behind the other
without waiting, as a training loop does (`sync=False`).  All data is fp32; there is no other type.

A case is a dict of plain values:
  op        "prod", "layer" (prod_bias_act), "grad" (densedense_to_dia) or "step" (one training step, six calls)
  table     "factory" (filter_factory_float), "channels" (one window per channel shift on a square map, offsets
            c*px*px + dy*px + dx) or "band" (offsets -fs//2 ... fs//2 on px*py rows)
  px, py, fs, maps_in, maps_out      the map, the window and the numbers of maps
  batch     dense columns
  trans     "n" or "t" (prod and layer)
  beta      factor of the destination's old value; 0: it is only written
  act       layer: "sigmoid" or "sample"
  sync      whether the call waits for its result
"""
import functools
import math

import numpy as np
import torch

from cuv_amd import _lib
from cuv_amd import dia as D
from cuv_amd import workloads as W

DEVICE = "cuda:0"
ACTS = {"sigmoid": _lib.ACT_SIGMOID, "sample": _lib.ACT_SIGMOID_SAMPLE}


def _case(name, op, table, px, py, fs, maps_in, maps_out, batch, trans="n", beta=0.0, act="", sync=False):
    return dict(name=name, op=op, table=table, px=px, py=py, fs=fs, maps_in=maps_in, maps_out=maps_out, batch=batch,
                trans=trans, beta=beta, act=act, sync=sync)


def listed():
    return [
        # one matrix-vector product of a banded matrix, waited for: the smallest call there is (configuration 0)
        _case("vector", "prod", "band", 64, 64, 33, 1, 1, 1, sync=True),
        # a handful of columns through a layer that widens 1 map to 16 (65536 x 1048576, 1024 diagonals, batch 14: the
        # shape of CUV's own product speed test): the values are nearly all of the traffic
        _case("few_columns", "prod", "factory", 256, 256, 8, 1, 16, 14, beta=0.5, sync=True),
        # the gradient of CUV's own gradient speed test (784 x 1568, 128 diagonals, batch 96), waited for
        _case("small_gradient", "grad", "factory", 28, 28, 8, 1, 2, 96, sync=True),
        # the up-pass of the 16384-unit layer at batch 128, waited for (configuration 1)
        _case("up_pass", "prod", "factory", 128, 128, 7, 1, 1, 128, sync=True),
        # one contrastive-divergence step on that layer: up, down, up, two gradients, the momentum update; queued
        _case("train_step", "step", "factory", 128, 128, 7, 1, 1, 128),
        # inference with a layer of odd sizes: 3 maps of 75 x 53 to 4, a batch of 100, down the layer
        _case("odd_layer", "layer", "factory", 75, 53, 5, 3, 4, 100, trans="t", act="sigmoid"),
        # several maps of odd width: 4 maps of 150 x 150 to 6, batch 200, in a training loop
        _case("odd_maps", "prod", "factory", 150, 150, 7, 4, 6, 200),
        # sampled hidden units of a 512 x 512 map
        _case("sampled_layer", "layer", "factory", 512, 512, 7, 1, 1, 128, act="sample"),
        # the down-pass into a prefilled destination on a large map with a large batch: the most traffic
        _case("down_pass_wide", "prod", "factory", 512, 512, 7, 1, 1, 512, trans="t", beta=0.5),
        # the gradient of the 16384-unit layer over a large batch, added to 0.9 times the last one
        _case("gradient_deep", "grad", "factory", 128, 128, 7, 1, 1, 2048, beta=0.9),
        # the large layer (262144 rows, 676 diagonals, batch 256; configuration 4): product and gradient
        _case("large_forward", "prod", "channels", 256, 256, 13, 4, 4, 256),
        _case("large_gradient", "grad", "channels", 256, 256, 13, 4, 4, 256),
    ]


# Drawn cases stay well below the largest listed case's arithmetic and traffic.
MOST_FLOPS, MOST_BYTES = 1.5e10, 1.2e9


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A layer of any size between a small map with one window and the large ones listed: widths and batches over
    their logarithm, half of each rounded to the usual multiples of 32 and half left odd; one or several maps.  One in
    ten is a banded matrix instead."""
    while True:
        op = rng.choice(["prod", "prod", "layer", "grad", "grad", "step"])
        px = _log_int(rng, 28, 512)
        if rng.random() < 0.5:
            px = max(32, (px + 16) // 32 * 32)
        py = px if rng.random() < 0.7 else max(16, int(px * rng.uniform(0.5, 1.5)))
        fs = rng.choice([3, 5, 5, 7, 7, 7, 8, 9, 11, 13])
        maps_in, maps_out = rng.choice([(1, 1), (1, 1), (1, 1), (1, 2), (2, 2), (3, 4), (1, 8), (1, 16), (4, 4), (4, 6)])
        table = "factory"
        if rng.random() < 0.1:
            table, fs, maps_in, maps_out = "band", 2 * _log_int(rng, 2, 40) + 1, 1, 1
        batch = _log_int(rng, 12, 1024) if rng.random() < 0.9 else rng.randint(1, 12)
        if batch > 24 and rng.random() < 0.5:
            batch = max(32, (batch + 16) // 32 * 32)
        c = _case("", op, table, px, py, fs, maps_in, maps_out, batch)
        del c["name"]
        if op in ("prod", "layer"):
            c["trans"] = rng.choice(["n", "t"])
            c["beta"] = rng.choice([0.0, 0.0, 0.5])
            c["sync"] = rng.random() < 0.3
        if op == "layer":
            c["act"] = rng.choice(["sigmoid", "sample"])
            c["beta"] = 0.0
        if op == "grad":
            c["beta"] = rng.choice([0.0, 0.9])
            c["sync"] = rng.random() < 0.3
        w = work(c)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return c


def _pattern(c):
    return _pattern_of(c["table"], c["px"], c["py"], c["fs"], c["maps_in"], c["maps_out"])


@functools.lru_cache(maxsize=64)
def _pattern_of(table, px, py, fs, maps_in, maps_out):
    if table == "band":
        return W.Pattern(px * py, px * py, np.arange(-(fs // 2), fs // 2 + 1, dtype=np.int32), px * py)
    if table == "channels":
        return W.pattern_large(px, maps_in, fs)
    h, w = px * py * maps_in, px * py * maps_out
    return W.Pattern(h, w, D.filter_factory_float(px, py, fs, maps_in, maps_out).offsets(), max(h, w))


def _dia(p):
    m = D.dev_dia_matrix_f(p.h, p.w, p.nd, p.stride, p.rf, device=DEVICE)
    m.set_offsets(p.offsets)
    m.desc                                   # the tables a program keeps with its matrix
    return m


def prepare(case, seed):
    """The layer and its operands: weights N(0, 0.01), units in [0, 1], binary inputs where the layer is binary."""
    c, p, b = case, _pattern(case), case["batch"]
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)

    def uniform(rows):
        return torch.rand(b, rows, generator=g, device=DEVICE)

    def binary(rows):
        return uniform(rows).lt_(0.5)

    def weights():
        m = _dia(p)
        m.vec.normal_(0.0, 0.01, generator=g)
        return m

    s = dict(case=c, A=weights(), seed=int(seed) * 7919 + 1)
    if c["op"] in ("prod", "layer"):
        n_out, n_in = (p.w, p.h) if c["trans"] == "t" else (p.h, p.w)
        s["X"] = uniform(n_in) if c["trans"] == "t" else binary(n_in)
        s["dst"] = uniform(n_out)
        if c["op"] == "layer":
            s["bias"] = torch.randn(n_out, generator=g, device=DEVICE) * 0.1
    elif c["op"] == "grad":
        s["H"], s["V"] = uniform(p.h), binary(p.w)
        s["bd"] = D.dev_block_descriptor_f(s["A"])
    else:
        s["V0"] = binary(p.w)
        s["H0"], s["V1"], s["H1"] = (torch.empty(b, r, device=DEVICE) for r in (p.h, p.w, p.h))
        s["bias_h"] = torch.randn(p.h, generator=g, device=DEVICE) * 0.1
        s["bias_v"] = torch.randn(p.w, generator=g, device=DEVICE) * 0.1
        s["dW"], s["M"] = _dia(p), _dia(p)
        s["bd"] = D.dev_block_descriptor_f(s["dW"])
    return s


def run(s):
    c, A = s["case"], s["A"]
    if c["op"] == "prod":
        return D.prod(s["dst"], A, s["X"], c["trans"], "n", 1.0, c["beta"], sync=c["sync"])
    if c["op"] == "layer":
        out = D.prod_bias_act(s["dst"], A, s["X"], c["trans"], 1.0, c["beta"], bias=s["bias"], act=ACTS[c["act"]],
                              seed=s["seed"], sync=c["sync"])
        # samples are 0 or 1: handed out as the whole numbers their bits are, to be compared as such
        return out.view(torch.int32) if c["act"] == "sample" else out
    if c["op"] == "grad":
        return D.densedense_to_dia(A, s["bd"], s["H"], s["V"], 1.0 / c["batch"], c["beta"], sync=c["sync"]).vec
    b = c["batch"]
    D.prod_bias_act(s["H0"], A, s["V0"], "n", bias=s["bias_h"], act=_lib.ACT_SIGMOID, sync=False)
    D.prod_bias_act(s["V1"], A, s["H0"], "t", bias=s["bias_v"], act=_lib.ACT_SIGMOID, sync=False)
    D.prod_bias_act(s["H1"], A, s["V1"], "n", bias=s["bias_h"], act=_lib.ACT_SIGMOID, sync=False)
    D.densedense_to_dia(s["dW"], s["bd"], s["H1"], s["V1"], 1.0 / b, 0.0, sync=False)
    D.densedense_to_dia(s["dW"], s["bd"], s["H0"], s["V0"], -1.0 / b, 1.0, sync=False)
    D.learn_step_weight_decay_momentum(A, s["M"], s["dW"], 0.05, 0.9, 2e-4, sync=False)
    return dict(H0=s["H0"], V1=s["V1"], H1=s["H1"], dW=s["dW"].vec, M=s["M"].vec, W=A.vec)


def work(case):
    """Every operand in and every result out once (4 bytes each, stored diagonals without their padding), and a
    multiplication and an addition per stored element and column."""
    c, p, b = case, _pattern(case), case["batch"]
    nnz, flops = p.nnz, W.flops(p, b)
    if c["op"] in ("prod", "layer"):
        extra = 4 * (p.w if c["trans"] == "t" else p.h) if c["op"] == "layer" else 0
        return dict(bytes=W.spmm_bytes(p, b, c["trans"], c["beta"]) + extra, flops=flops)
    if c["op"] == "grad":
        return dict(bytes=W.dd2dia_bytes(p, b, c["beta"]), flops=flops)
    # V0 in; H0, V1, H1 out; W and the momentum in and out, the gradient out; both biases in
    return dict(bytes=4 * (2 * p.h * b + 2 * p.w * b + 5 * nnz + p.h + p.w), flops=5 * flops)


def tolerance(case):
    if case["act"] == "sample":
        return dict(rel=0.0, differ=1e-5)    # a sample turns over where its probability meets the draw within rounding
    return dict(rel=1e-5)                    # fp32 sums in another order
