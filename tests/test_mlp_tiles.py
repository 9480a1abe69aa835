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


# rows that give the larger tiles 640 blocks with one or two column tiles, and edges around them
@pytest.mark.parametrize("M, N, K", [(81920, 64, 8), (81793, 128, 40), (40961, 256, 256), (41000, 131, 33),
                                     (128, 256, 64)])
@pytest.mark.parametrize("odd", [False, True])
def test_products_along_k(M, N, K, odd):
    import torch

    pad = 1 if odd else 0  # operands and results of odd row length
    A, W, b = _rand(torch, M, K + pad)[:, :K], _rand(torch, N, K + pad)[:, :K], _rand(torch, N).float()
    ref = A.float() @ W.float().T + b
    scale = A.float().abs() @ W.float().abs().T + b.abs()
    Z = torch.empty((M, N + pad), device="cuda")
    H = torch.empty((M, N + pad), dtype=torch.bfloat16, device="cuda")
    S.gemm(A, K + pad, 1, W, 1, K + pad, M, N, K, _abi.GX_EPI_BIAS_SILU, bias=b, C=Z, ldc=N + pad, H=H, ldh=N + pad)
    tol = 2 * K * EPS32 * scale
    assert bool(((Z[:, :N] - ref).abs() <= tol).all())
    act = _silu(ref)
    # SiLU's slope is below 1.1
    assert bool(((H[:, :N].float() - act).abs() <= 1.1 * tol + (EPS16 + 2.0 ** -20) * act.abs() + 1e-30).all())
    # the derivative's epilogue on the same product without the bias
    D = torch.empty((M, N + pad), dtype=torch.bfloat16, device="cuda")
    S.gemm(A, K + pad, 1, W, 1, K + pad, M, N, K, _abi.GX_EPI_DSILU, H=D, ldh=N + pad, Z=Z, ldz=N + pad)
    s = 1.0 / (1.0 + (-Z[:, :N]).exp())
    d = s * (1.0 + Z[:, :N] * (1.0 - s))
    want = (ref - b) * d
    assert bool(((D[:, :N].float() - want).abs() <= 1.1 * tol + 2 * EPS16 * want.abs() + 2.0 ** -19 * scale).all())


@pytest.mark.parametrize("M, N, K, ksplit", [(64, 64, 3072, 1), (128, 256, 3105, 1), (256, 256, 4000, 3),
                                             (132, 68, 4099, 16), (256, 256, 3080, 256), (64, 64, 70, 2)])
def test_products_along_columns(M, N, K, ksplit):
    import torch

    A, B = _rand(torch, K, M), _rand(torch, K, N)
    ref = A.float().T @ B.float()
    scale = A.float().abs().T @ B.float().abs()
    C = torch.zeros((M, N), device="cuda")
    S.gemm(A, 1, M, B, N, 1, M, N, K, _abi.GX_EPI_STORE, C=C, ldc=N, ksplit=ksplit)
    assert bool(((C - ref).abs() <= 2 * K * EPS32 * scale + 1e-30).all())
    if ksplit == 1:
        S.gemm(A, 1, M, B, N, 1, M, N, K, _abi.GX_EPI_STORE, C=C, ldc=N, accumulate=1)
        assert bool(((C - 2 * ref).abs() <= 6 * K * EPS32 * scale + 1e-30).all())


@pytest.mark.parametrize("M, N", [(1, 8), (7, 256), (129, 264), (4099, 256), (1000, 12)])
def test_column_sums(M, N):
    import torch

    from galax_amd import _lib

    X = _rand(torch, M, N)
    out = torch.zeros(N, device="cuda")
    _lib.check(_lib.lib().gx_mlp_colsum(_lib.ptr(X), N, M, N, _lib.ptr(out), _lib.stream_ptr()), "gx_mlp_colsum")
    assert bool(((out - X.float().sum(0)).abs() <= 2 * M * EPS32 * X.float().abs().sum(0)).all())


@pytest.mark.parametrize("n", [1, 127, 128, 129, 300, 16385, 16513])
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
