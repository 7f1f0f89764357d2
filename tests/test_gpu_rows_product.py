"""The product whose waves split K over tiles of 16 to 64 rows: edges of its tiles in rows and features, K that leaves a rest of a
group or whole waves without work, its epilogues, weights in operand tiles against row-major ones, and what it prepares for the next
norm."""

import pytest
import torch

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


# (rows, features, K): every tile height and its edges; features that end inside a tile or a quad; K of one piece, of a rest, of
# fewer groups than waves, of a half group for operand tiles; one tile and a whole round of them
SHAPES = [(1, 16, 8), (16, 40, 64), (17, 96, 520), (32, 33, 2048), (33, 130, 96), (48, 2048, 1056), (64, 515, 168), (64, 6144, 256),
          (65, 1000, 1024), (130, 1024, 4608), (257, 3072, 224), (512, 2048, 96),
          (1, 40, 1032), (5, 2064, 2048), (16, 515, 1112)]      # up to 16 rows only beyond K 1,024


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product_of_a_few_rows(ops, M, N, K):
    a, w, bias = draw(M, K), draw(N, K, seed=1), torch.randn(N, generator=torch.Generator().manual_seed(2))
    limit, exact = bound(a, w), a.double() @ w.double().T
    A, W, B, T = a.to(DEV), w.to(DEV), bias.to(DEV), ops.tile_weights(w.to(DEV))
    found = ops.gemm(A, W, out_dtype=torch.float32, w_tiled=T)
    assert ((found.cpu().double() - exact).abs() <= limit).all()
    if M <= 64:         # (beyond, row-major weights take other products)
        assert torch.equal(ops.gemm(A, W, out_dtype=torch.float32), found)      # the same sums in the same order
    with_bias = ops.gemm(A, W, B, out_dtype=torch.float32, w_tiled=T).cpu().double()
    assert ((with_bias - exact - bias.double()).abs() <= limit + 2.0 ** -23 * with_bias.abs()).all()
    assert ((ops.gemm(A, W, w_tiled=T).cpu().double() - exact).abs() <= limit + 2.0 ** -8 * exact.abs()).all()
    residual = torch.randn(M, N, generator=torch.Generator().manual_seed(3))
    into = residual.to(DEV)
    ops.gemm(A, W, accumulate_into=into, w_tiled=T)
    total = exact + residual.double()
    assert ((into.cpu().double() - total).abs() <= limit + 2.0 ** -23 * total.abs()).all()
    if N % 4 == 0:      # rows of the output that do not start at 16 bytes
        flat = torch.zeros(M * N + 1, device=DEV)
        flat[1:] = residual.reshape(-1).to(DEV)
        ops.gemm(A, W, accumulate_into=flat[1:].view(M, N), w_tiled=T)
        assert torch.equal(flat[1:].view(M, N), into)


@pytest.mark.parametrize("N,K", [(3072, 1024), (1024, 968), (2048, 96)])
def test_a_row_among_other_rows(ops, N, K):
    """Among as many rows a row's result depends neither on the others nor on its place; the number of rows chooses the tile, and with it
    the number of waves that K is dealt to (at 3,072 features eight up to 32 rows, four beyond), so across numbers of rows it is the
    same up to the order of the sum."""
    a, w = draw(64, K), draw(N, K, seed=1)
    A, W = a.to(DEV), w.to(DEV)
    limit = bound(a, w)
    found = {}
    for M in (12, 17, 32, 33, 64):
        found[M] = ops.gemm(A[:M].contiguous(), W, out_dtype=torch.float32)
        turned = torch.roll(A[:M], 5, 0).contiguous()
        turned[0] = 3.0
        again = ops.gemm(turned, W, out_dtype=torch.float32)
        assert torch.equal(again[6:], found[M].roll(5, 0)[6:]), M
        assert torch.equal(ops.gemm(A[:M].contiguous(), W, out_dtype=torch.float32), found[M])
    for M in found:
        assert ((found[M] - found[64][:M]).abs().cpu().double() <= 2 * limit[:M]).all()


@pytest.mark.parametrize("M,F,K", [(1, 16, 64), (17, 77, 520), (40, 130, 96), (64, 4608, 1024), (190, 1000, 224)])
def test_gated_product_of_a_few_rows(ops, M, F, K):
    a, w = draw(M, K, scale=K ** -0.5), draw(2 * F, K, seed=1)
    limit, sums = bound(a, w), a.double() @ w.double().T
    g, u = sums[:, :F], sums[:, F:]
    exact = torch.nn.functional.silu(g) * u
    # silu's slope is below 1.1; the unit's own roundings are far below the bfloat16 it is rounded to
    allowed = 1.1 * limit[:, :F] * u.abs() + limit[:, F:] * g.abs() + 2.0 ** -7 * exact.abs() + 1e-12
    W = w.to(DEV)
    found = ops.gemm_swiglu(a.to(DEV), W)
    assert ((found.cpu().double() - exact).abs() <= allowed).all()
    if K % 32 == 0:
        tiled = ops.gemm_swiglu(a.to(DEV), W, w_tiled=ops.tile_weights(W))
        assert torch.equal(tiled, found) if M <= 64 else ((tiled.cpu().double() - exact).abs() <= allowed).all()


@pytest.mark.parametrize("M,N,K", [(12, 2048, 4608), (17, 96, 520), (50, 2048, 256), (64, 515, 168)])
def test_a_few_rows_prepare_the_next_norm(ops, M, N, K):
    a, w, weight = draw(M, K), draw(N, K, seed=1, scale=K ** -0.5), 1.0 + 0.1 * torch.randn(N, generator=torch.Generator().manual_seed(4))
    into = torch.randn(M, N, generator=torch.Generator().manual_seed(3)).to(DEV)
    activations, squares = ops.gemm_medium(a.to(DEV), w.to(DEV), ops.EPILOGUE_ACCUMULATE, accumulate_into=into, next_norm_weight=weight.to(DEV))
    assert torch.equal(activations.cpu(), (into.cpu() * weight).to(torch.bfloat16))
    sums = (into.cpu().double() ** 2).sum(1)
    assert ((squares.double().sum(0)[:M].cpu() - sums).abs() <= N * 2.0 ** -24 * sums).all()
    if N % 8 == 0:
        v = draw(96, N, seed=5)
        exact = activations.cpu().double() @ v.double().T / torch.sqrt(sums / N + 1e-5)[:, None]
        found = ops.gemm_medium(activations, v.to(DEV), ops.EPILOGUE_STORE, squares=squares, eps=1e-5, out_dtype=torch.float32).cpu().double()
        scale = 1.0 / torch.sqrt(sums / N + 1e-5)[:, None]
        assert ((found - exact).abs() <= bound(activations.cpu(), v) * scale + (N + 8) * 2.0 ** -24 * exact.abs()).all()
