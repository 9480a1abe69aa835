"""The large products of a network's layers at shapes that take the 128 x 128
tiles, for each reading of the weights (along k, as columns), each result and
each edge: ragged rows and columns, k beside the slabs of 32, row lengths that
keep the results from 16-byte stores.

Bounds: a product accumulates K terms in float32, in another order than the
reference: 2 K units in the last place (2^-24) of the sum of |a b|; BF16
results half a unit (2^-8) of themselves more; SiLU's slope is below 1.1, its
hardware exponential and reciprocal within 2^-20."""

import numpy as np
import pytest

import galax_amd.surrogate as S
from galax_amd import _abi

pytestmark = pytest.mark.gpu
EPS32, EPS16 = 2.0 ** -24, 2.0 ** -8


def _rand(torch, *shape):
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)


class _Product:
    """A (M, K) with rows of sam elements; B read along k or as columns."""

    def __init__(self, M, N, K, columns, extra):
        import torch

        self.torch, self.size, self.extra = torch, (M, N, K), extra
        sam = K + (8 if extra else 0)
        A = _rand(torch, M, sam)
        # k beyond the row is not part of it: NaN there must not reach a result
        A[:, K:] = float("nan")
        W = _rand(torch, N, K)
        B = W.T.contiguous() if columns else W
        self.ops = (A, sam, 1, B, *((N, 1) if columns else (1, K)), M, N, K)
        self.keep = (A, B)
        self.bias = _rand(torch, N).float()
        self.ref = A[:, :K].float() @ W.float().T
        self.scale = A[:, :K].float().abs() @ W.float().abs().T
        self.tol = 2 * K * EPS32 * (self.scale + self.bias.abs())

    def new(self, dtype, pad):
        M, N, _ = self.size
        t = self.torch.full((M, N + pad), 7.0, dtype=dtype, device="cuda")
        return t, N + pad

    def check(self, got, pad, want, tol):
        N = self.size[1]
        err = (got[:, :N].float() - want).abs()
        assert bool((err <= tol).all()), float((err - tol).max())
        assert pad == 0 or bool((got[:, N:] == 7.0).all())


# 1,024 blocks (65,531 x 250 and the like) for what is read along k with the
# pre-activations kept, three quarters of 512 for the derivative, 640 else
SILU = [(131_065, 128, 40, False), (131_069, 100, 24, False), (65_531, 256, 256, False), (65_530, 250, 72, False),
        (131_065, 128, 40, True), (65_531, 256, 256, True)]


@pytest.mark.parametrize("M, N, K, columns", SILU)
@pytest.mark.parametrize("extra", [0, 1])
def test_layers_forward(M, N, K, columns, extra):
    p = _Product(M, N, K, columns, extra)
    (Z, ldz), (H, ldh) = p.new(p.torch.float32, extra), p.new(p.torch.bfloat16, extra)
    S.gemm(*p.ops, _abi.GX_EPI_BIAS_SILU, bias=p.bias, C=Z, ldc=ldz, H=H, ldh=ldh)
    ref = p.ref + p.bias
    p.check(Z, extra, ref, p.tol)
    act = ref / (1.0 + (-ref).exp())
    p.check(H, extra, act, 1.1 * p.tol + (EPS16 + 2.0 ** -20) * act.abs() + 1e-30)


@pytest.mark.parametrize("extra", [0, 1])
def test_first_layer_without_its_pre_activations(extra):
    p = _Product(131_065, 128, 8, False, extra)
    H, ldh = p.new(p.torch.bfloat16, extra)
    S.gemm(*p.ops, _abi.GX_EPI_BIAS_SILU, bias=p.bias, H=H, ldh=ldh)
    ref = p.ref + p.bias
    act = ref / (1.0 + (-ref).exp())
    p.check(H, extra, act, 1.1 * p.tol + (EPS16 + 2.0 ** -20) * act.abs() + 1e-30)


# three quarters of a round of blocks, one, and several with an odd half tile
DSILU = [(49_157, 128, 40), (65_003, 100, 72), (24_600, 256, 256), (40_001, 192, 72), (98_290, 192, 40),
         (12_350, 512, 512)]


@pytest.mark.parametrize("M, N, K", DSILU)
@pytest.mark.parametrize("columns", [False, True])
@pytest.mark.parametrize("extra", [0, 1])
def test_gradients_of_activations(M, N, K, columns, extra):
    p = _Product(M, N, K, columns, extra)
    Z, ldz = p.new(p.torch.float32, 3 * extra)
    Z[:, :N] = 2.0 * _rand(p.torch, M, N).float()
    D, ldd = p.new(p.torch.bfloat16, extra)
    S.gemm(*p.ops, _abi.GX_EPI_DSILU, H=D, ldh=ldd, Z=Z, ldz=ldz)
    z = Z[:, :N]
    s = 1.0 / (1.0 + (-z).exp())
    slope = s * (1.0 + z * (1.0 - s))
    want = p.ref * slope
    p.check(D, extra, want, 1.1 * p.tol + EPS16 * want.abs() + 2.0 ** -19 * p.ref.abs() + 1e-30)


@pytest.mark.parametrize("M, N, K, columns", [(131_065, 128, 40, False), (65_531, 256, 72, False),
                                              (40_970, 256, 64, True), (81_925, 100, 72, True)])
@pytest.mark.parametrize("extra", [0, 1])
def test_plain_products(M, N, K, columns, extra):
    p = _Product(M, N, K, columns, extra)
    C, ldc = p.new(p.torch.float32, extra)
    S.gemm(*p.ops, _abi.GX_EPI_STORE, C=C, ldc=ldc)
    p.check(C, extra, p.ref, p.tol)
    S.gemm(*p.ops, _abi.GX_EPI_STORE, C=C, ldc=ldc, accumulate=1)
    p.check(C, extra, 2 * p.ref, 3 * p.tol)
    S.gemm(*p.ops, _abi.GX_EPI_BIAS, bias=p.bias, C=C, ldc=ldc)
    p.check(C, extra, p.ref + p.bias, p.tol)


def test_a_training_step_of_large_products_against_autograd():
    """65,536 rows of hidden width 256, where forward, activations' and
    weights' gradients all take the larger tiles.  Activations and cotangents
    are BF16, so the match is to BF16 level."""
    import torch

    from galax_amd import _lib

    n = 65_536
    mlp = S.MLP(hidden=256, depth=3, seed=1)
    X = torch.zeros((n, S.K_IN), dtype=torch.bfloat16, device="cuda")
    X[:, :5] = _rand(torch, n, 5)
    T = 0.5 * _rand(torch, n, 3).float()
    Y = torch.empty((n, 3), device="cuda")
    dY = torch.empty((n, S.K_IN), dtype=torch.bfloat16, device="cuda")
    loss = torch.zeros(1, dtype=torch.float64, device="cuda")
    mlp.forward(X, n, Y, train=True)
    _lib.check(_lib.lib().gx_mlp_huber(S._p(Y), 3, S._p(T), n, 1.0, 1.0 / n, S._p(dY), S.K_IN, S._p(loss), S._s()),
               "gx_mlp_huber")
    mlp.backward(X, n, dY)
    Ws = [w.float().clone().requires_grad_(True) for w in mlp.Wb]
    bs = [b.clone().requires_grad_(True) for b in mlp.b]
    h = X.float()
    for W, b in zip(Ws[:-1], bs[:-1]):
        h = torch.nn.functional.silu(h @ W.t() + b)
    y = h @ Ws[-1].t() + bs[-1]
    np.testing.assert_allclose(Y.cpu().numpy(), y.detach().cpu().numpy(), rtol=3e-2, atol=3e-2 * float(y.abs().max()))
    ((torch.sqrt(1 + (y - T) ** 2) - 1).sum() / n).backward()
    for got, p in zip(mlp.g, Ws + bs):
        assert float((got - p.grad).norm() / p.grad.norm().clamp_min(1e-30)) < 3e-2
