"""The products of few rows that are not the waves-split-K tiles: the one that splits K over workgroups (slices that meet through a
workspace and a ticket; wide outputs whose workgroups start their walk over K at different places), and the one of up to sixteen
rows over a short K. Shapes end inside tiles, slices, chunks and quads of features; weights row-major and in operand tiles; each
epilogue against float64."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    return module


def draw(*shape, seed=0, scale=1.0):
    generator = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=generator) * scale).to(torch.bfloat16)


def bound(a, w):
    """Products of bfloat16 are exact in float32: K + 16 rounded sums, at most that many 2^-24 of the sum of the products' sizes."""
    return (a.shape[1] + 16) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


def close(found, exact, limit, rounding):
    assert ((found.cpu().double() - exact).abs() <= limit + rounding * exact.abs()).all()


# K in slices of several workgroups (three to sixteen); tiles of 32 features in a round and in two; tiles of 64 features over all
# of K, K x N beyond 2^24 (the walk starts elsewhere in each workgroup) and below; K of half a chunk more
SHAPES = [(1, 512, 12288), (12, 512, 6144), (9, 1000, 8224), (16, 2048, 8192), (17, 2048, 10272), (32, 2552, 6176),
          (40, 2560, 12320), (64, 2046, 12288), (17, 5000, 1024), (20, 16400, 296), (33, 20470, 520), (1, 25000, 1056),
          (9, 25000, 1056), (16, 25000, 1056), (17, 25000, 1056), (40, 25000, 1056), (64, 25000, 1056), (64, 24580, 72)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product_that_splits_k_over_workgroups(ops, M, N, K):
    assert ops.medium_splits_k(0, M, N, K)
    a, w = draw(M, K), draw(N, K, seed=1, scale=K ** -0.5)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2))
    limit, exact = bound(a, w), a.double() @ w.double().T
    A, W, B = a.to(DEV), w.to(DEV), bias.to(DEV)
    T = ops.tile_weights(W)
    product = lambda **how: ops.gemm_medium(A, W, ops.EPILOGUE_STORE, **how)        # noqa: E731
    found = product(out_dtype=torch.float32)
    close(found, exact, limit, 2.0 ** -24)
    for _ in range(3):          # the tickets are left at zero, and whoever comes last adds the slices in their order
        assert torch.equal(product(out_dtype=torch.float32), found)
    if T is not None:
        assert torch.equal(product(out_dtype=torch.float32, w_tiled=T), found)
    close(product(bias=B, out_dtype=torch.float32), exact + bias.double(), limit, 2.0 ** -23)
    close(product(w_tiled=T), exact, limit, 2.0 ** -8)
    # (gelu's slope is below 1.13; its short error function is within 1.5e-7, times half of z)
    close(product(bias=B, w_tiled=T, gelu=True), F.gelu(exact + bias.double()), 1.13 * limit + 1e-6, 2.0 ** -8)
    residual = torch.randn(M, N, generator=torch.Generator().manual_seed(3))
    into = residual.to(DEV)
    ops.gemm_medium(A, W, ops.EPILOGUE_ACCUMULATE, accumulate_into=into, w_tiled=T)
    close(into, exact + residual.double(), limit, 2.0 ** -23)


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("M,N,K,squares_rows", [(1, 25000, 1056, 3), (9, 25000, 1056, 700), (16, 2048, 8192, 128), (17, 25000, 1056, 64),
                                                (40, 2560, 12320, 33), (64, 25000, 1056, 300)])
def test_prepared_activations_in_the_product_that_splits_k(ops, M, N, K, squares_rows, tiled):
    """The rows' 1 / rms is formed from the sums of squares that the product before left (more and fewer of them than are asked for
    ahead) and applied to the sums."""
    assert ops.medium_splits_k(0, M, N, K)
    a, w = draw(M, K), draw(N, K, seed=1, scale=K ** -0.5)
    generator = torch.Generator().manual_seed(4)
    squares = torch.rand(squares_rows, 16 if M <= 16 else 64, generator=generator) * (0.5 + torch.arange(16 if M <= 16 else 64)) * K / squares_rows
    inv = (squares.double().sum(0)[:M] / K + 1e-5).rsqrt()[:, None]
    limit, exact = bound(a, w) * inv, (a.double() @ w.double().T) * inv
    A, W = a.to(DEV), w.to(DEV)
    T = ops.tile_weights(W) if tiled else None
    how = dict(squares=squares.to(DEV), eps=1e-5, w_tiled=T)
    # (the sums of squares are float32: squares_rows roundings at most, half of that in the root; two more in applying it)
    rounding = (squares_rows / 2 + 4) * 2.0 ** -24
    close(ops.gemm_medium(A, W, ops.EPILOGUE_STORE, out_dtype=torch.float32, **how), exact, limit, rounding)
    close(ops.gemm_medium(A, W, ops.EPILOGUE_STORE, **how), exact, limit, rounding + 2.0 ** -8)


@pytest.mark.parametrize("M,N,K", [(9, 1000, 8224), (16, 2048, 8192), (17, 2048, 10272), (40, 2560, 12320)])
def test_what_the_adding_product_that_splits_k_leaves_for_the_next_norm(ops, M, N, K):
    a, w = draw(M, K), draw(N, K, seed=1, scale=K ** -0.5)
    residual, weight = torch.randn(M, N, generator=torch.Generator().manual_seed(5)), torch.rand(N, generator=torch.Generator().manual_seed(6)) + 0.5
    into = residual.to(DEV)
    A, W = a.to(DEV), w.to(DEV)
    activations, squares = ops.gemm_medium(A, W, ops.EPILOGUE_ACCUMULATE, accumulate_into=into, next_norm_weight=weight.to(DEV),
                                           w_tiled=ops.tile_weights(W))
    x = into.cpu().double()
    close(into, residual.double() + a.double() @ w.double().T, bound(a, w), 2.0 ** -23)
    assert ((activations.cpu().double() - x * weight.double()).abs() <= 2.0 ** -8 * (x * weight.double()).abs() + 1e-30).all()
    total = (x * x).sum(1)
    assert ((squares.cpu().double()[:, :M].sum(0) - total).abs() <= 16 * 2.0 ** -24 * total).all()


@pytest.mark.parametrize("M,N,K", [(17, 8200, 1056), (33, 4700, 1024), (64, 9000, 544), (48, 4104, 1536)])
def test_gated_product_that_splits_k_over_workgroups(ops, M, N, K):
    assert ops.medium_splits_k(2, M, N, K)
    a, w = draw(M, K, scale=K ** -0.5), draw(2 * N, K, seed=1)
    sums, limit = a.double() @ w.double().T, bound(a, w)
    g, u = sums[:, :N], sums[:, N:]
    A, W = a.to(DEV), w.to(DEV)
    T = ops.tile_weights(W)
    for glu, unit in ((None, F.silu(g) * u), (ops.GEGLU, F.gelu(g, approximate="tanh") * u)):
        # both units' slopes are below 1.13
        allowed = 1.13 * limit[:, :N] * u.abs() + limit[:, N:] * g.abs() + 1e-6
        found = ops.gemm_medium(A, W, ops.EPILOGUE_SWIGLU, glu=glu, w_tiled=T)
        close(found, unit, allowed, 2.0 ** -8)
        assert torch.equal(ops.gemm_medium(A, W, ops.EPILOGUE_SWIGLU, glu=glu), found)


@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (1, 33, 136), (7, 4097, 1024), (16, 515, 768), (16, 8192, 264), (8, 12296, 512), (15, 4096, 128)])
def test_product_of_up_to_sixteen_rows_over_a_short_k(ops, M, N, K):
    assert ops.skinny_takes(M, N, K)
    a, w = draw(M, K), draw(N, K, seed=1, scale=K ** -0.5)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2))
    limit, exact = bound(a, w), a.double() @ w.double().T
    A, W, B = a.to(DEV), w.to(DEV), bias.to(DEV)
    found = ops.gemm(A, W, out_dtype=torch.float32)
    close(found, exact, limit, 2.0 ** -24)
    assert torch.equal(ops.gemm(A[M - 1:].contiguous(), W, out_dtype=torch.float32)[0], found[M - 1])
    close(ops.gemm(A, W, B, out_dtype=torch.float32), exact + bias.double(), limit, 2.0 ** -23)
    close(ops.gemm(A, W), exact, limit, 2.0 ** -8)
    close(ops.gemm(A, W, B, gelu=True), F.gelu(exact + bias.double()), 1.13 * limit + 1e-6, 2.0 ** -8)
    residual = torch.randn(M, N, generator=torch.Generator().manual_seed(3))
    into = residual.to(DEV)
    ops.gemm(A, W, accumulate_into=into)
    close(into, exact + residual.double(), limit, 2.0 ** -23)
    if N % 2 == 0:
        g, u = exact[:, :N // 2], exact[:, N // 2:]
        allowed = 1.13 * limit[:, :N // 2] * u.abs() + limit[:, N // 2:] * g.abs() + 1e-6
        close(ops.gemm_swiglu(A, W), F.silu(g) * u, allowed, 2.0 ** -8)
        close(ops.gemm_swiglu(A, W, gelu=True), F.gelu(g, approximate="tanh") * u, allowed, 2.0 ** -8)
