"""The surrogate's larger tiles at their edges: the products read along k and
along columns, the column sums and the fused inference, against float32
references of the same operations on the same BF16 operands.

Bounds: a product accumulates K terms in float32, in another order than the
reference: 2 K units in the last place (2^-24) of the sum of |a b|, below
sqrt(K) times it in practice; BF16 results half a unit (2^-8) of themselves
more, SiLU's hardware exponential and reciprocal 2^-20."""

import pytest

import galax_amd.surrogate as S
from galax_amd import _abi

pytestmark = pytest.mark.gpu
EPS32, EPS16 = 2.0 ** -24, 2.0 ** -8


def _rand(torch, *shape):
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)


def _silu(z):
    return z / (1.0 + (-z).exp())


@pytest.mark.parametrize("n", [1, 127, 128, 129, 300])
@pytest.mark.parametrize("depth", [1, 2, 4])
def test_fused_inference_follows_the_layers(n, depth):

    import torch

    mlp = S.MLP(hidden=256, depth=depth, seed=n)
    for b in mlp.b:
        b.copy_(0.1 * _rand(torch, b.numel() + 1)[1:].float())
    X = torch.zeros((n, S.K_IN), dtype=torch.bfloat16, device="cuda")
    X[:, :5] = _rand(torch, n, 5)
    Y, F = torch.empty((n, 3), device="cuda"), torch.full((n, 3), float("nan"), device="cuda")
    mlp.forward(X, n, Y)
    mlp.forward_fused(X, n, F)
    # the first layer sums its eight inputs one by one instead of in one
    # matrix instruction, which may move a BF16 activation by a unit
    assert bool(torch.isfinite(F).all())
    assert float((F - Y).abs().max()) <= 2e-2 * float(Y.abs().max())
