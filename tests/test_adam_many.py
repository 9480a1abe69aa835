"""Adam on several tensors in one launch against the formula in 64 bits: sizes
about a block and beyond the grid's stride, with and without a BF16 copy, and
a network of more tensors than one launch takes.

Bound: a step's update is a dozen float32 operations on values up to 1.5 times
the learning rate, the parameter's own rounding half a unit (2^-24) more."""

import ctypes

import numpy as np
import pytest

import galax_amd.surrogate as S
from galax_amd import _abi, _lib

pytestmark = pytest.mark.gpu
LR, B1, B2, EPS = 1e-2, 0.9, 0.999, 1e-8


class _Reference:
    def __init__(self, p):
        self.p, self.m, self.v = p.double().cpu().numpy(), 0.0, 0.0

    def step(self, g, k):
        g = g.double().cpu().numpy()
        self.m = B1 * self.m + (1 - B1) * g
        self.v = B2 * self.v + (1 - B2) * g * g
        self.p = self.p - LR * (self.m / (1 - B1 ** k)) / (np.sqrt(self.v / (1 - B2 ** k)) + EPS)

    def check(self, p, pb, steps):
        got = p.double().cpu().numpy()
        assert np.all(np.abs(got - self.p) <= steps * (2.0 ** -24 * np.abs(self.p) + 1.5 * LR * 2.0 ** -19))
        if pb is not None:
            assert bool((pb == p.bfloat16()).all())


def _tensors(torch, sizes):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes))
    new = lambda n: torch.randn(n, generator=g, device="cuda")
    return [(new(n), new(n)) for n in sizes]


@pytest.mark.parametrize("sizes", [[1], [255, 256, 257], [4096 * 256 + 5, 3, 0, 70_001], list(range(1, 21))])
def test_many_tensors_in_one_launch(sizes):
    import torch

    pairs = _tensors(torch, sizes)
    zeros = [[torch.zeros(n, device="cuda") for n in sizes] for _ in range(2)]
    copies = [torch.zeros(n, dtype=torch.bfloat16, device="cuda") if k % 2 == 0 else None for k, n in enumerate(sizes)]
    refs = [_Reference(p) for p, _ in pairs]
    table = lambda xs: (ctypes.c_void_p * len(xs))(*[None if x is None or not x.numel() else int(x.data_ptr()) for x in xs])
    for k in (1, 2, 3):
        rc = _lib.lib().gx_mlp_adam_many(len(sizes), table([p for p, _ in pairs]), table([g for _, g in pairs]),
                                         table(zeros[0]), table(zeros[1]), table(copies),
                                         (ctypes.c_int64 * len(sizes))(*sizes), LR, B1, B2, EPS, k, _lib.stream_ptr())
        _lib.check(rc, "gx_mlp_adam_many")
        for r, (_, g) in zip(refs, pairs):
            r.step(g, k)
    for r, (p, _), pb in zip(refs, pairs, copies):
        r.check(p, pb, 3)


def test_a_network_of_more_tensors_than_one_launch_takes():
    import torch

    mlp = S.MLP(hidden=64, depth=11, seed=3)
    assert len(mlp.params) > _abi.GX_ADAM_TENSORS
    refs = [_Reference(p) for p in mlp.params]
    for k in (1, 2):
        for g, (_, new) in zip(mlp.g, _tensors(torch, [p.numel() + k for p in mlp.params])):
            g.copy_(new[:g.numel()].view_as(g))
        for r, g in zip(refs, mlp.g):
            r.step(g, k)
        mlp.adam(LR, B1, B2, EPS)
    for r, p, pb in zip(refs, mlp.params, mlp.Wb + [None] * len(mlp.b)):
        r.check(p, pb, 2)


def test_what_is_refused():
    lib, none = _lib.lib(), (ctypes.c_void_p * 1)(None)
    size = (ctypes.c_int64 * 1)(4)
    call = lambda count, step, n=size: lib.gx_mlp_adam_many(count, none, none, none, none, none, n, LR, B1, B2, EPS, step,
                                                            _lib.stream_ptr())
    assert call(-1, 1) == call(_abi.GX_ADAM_TENSORS + 1, 1) == call(1, 0) == call(1, 1) == _abi.GX_EINVAL
    assert call(0, 1) == call(1, 1, (ctypes.c_int64 * 1)(0)) == _abi.GX_OK
