"""The gated unit with clamped halves behind a product on large tiles, every tile: edges in rows and features, against the unit of the exact sums."""

import pytest
import torch

from test_gpu_large_tiles import DEV, TILES, draw, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("K", [32, 160, 544])
def test_every_tile(ops, tile, K):  # noqa: F811
    rows, columns, _ = tile
    limit, alpha, shift = 0.7, 1.702, 1.0        # sums are about one in size: both clamps are met
    for M, N in ((rows - 1, columns // 2 - 6), (rows + 3, columns + 5), (2 * rows, columns)):
        a, w, exact, off = draw(M, 2 * N, K)
        out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        print(M, N, K, tile, flush=True)
        ops._check(ops.library().fw_gemm_mfma_big_tile_clamped(ops._p(a), ops._p(w), ops._p(out), M, N, K, *tile, limit, alpha, shift, ops._stream()))
        gate, up = exact[:, :N].clamp(max=limit), exact[:, N:].clamp(-limit, limit)
        want = gate * torch.sigmoid(alpha * gate) * (up + shift)
        # g sigmoid(alpha g) slopes below 1.1, its size below |g|; clamping moves nothing further apart; the hardware's exponential and
        # reciprocal 2^-20 of |g| (u + shift); one rounding to bfloat16
        room = (1.1 * off[:, :N] * ((up + shift).abs() + off[:, N:]) + gate.abs() * off[:, N:] + 2.0 ** -20 * (gate * (up + shift)).abs()
                + 2.0 ** -8 * want.abs() + 2.0 ** -133)
        assert ((out.double() - want).abs() <= room).all()


def test_a_models_weights_take_it_and_infinities_are_clamped(ops):  # noqa: F811
    from flyweight_amd.parts.linear import Linear
    g = torch.Generator().manual_seed(5)
    w, a = (torch.randn(n, 512, generator=g).to(torch.bfloat16).to(DEV) for n in (3072, 200))
    a[3, 7] = float("inf")
    product = Linear(w)
    got, want = product.clamped_glu(a, 7.0, 1.702, 1.0), ops.clamped_glu(product.forward(a, out_dtype=torch.float32), 7.0, 1.702, 1.0, torch.bfloat16)
    assert ops.large_tile(2, 200, 1536, 512) is not None
    assert torch.equal(got.isnan(), want.isnan()) and not got[torch.arange(200, device=DEV) != 3].isnan().any()
    rows = torch.arange(200, device=DEV) != 3
    # both are rounded to bfloat16 once, 2^-9 of each element; the sums and sigmoids before that are within some 2^-20
    assert (got - want)[rows].double().norm() <= 2.0 ** -8 * want[rows].double().norm()
    assert torch.equal(got[3].isinf(), want[3].isinf())
    with pytest.raises(ops.KernelError):
        ops._check(ops.library().fw_gemm_mfma_big_tile_clamped(ops._p(a), ops._p(w), ops._p(got), 200, 1536, 512, 128, 256, 1, 0.0, 1.7, 1.0, ops._stream()))


@pytest.mark.parametrize("tile", [(128, 256, 1), (192, 192, 1), (64, 128, 2)])
@pytest.mark.parametrize("limit,alpha,shift", [(7.0, 1.0, 1.0), (30.0, 4.0, 0.0), (1000.0, 16.0, 0.0)])
def test_the_unit_is_as_exact_as_on_float32_sums_in_memory(ops, tile, limit, alpha, shift):  # noqa: F811
    """One number a sum and an alpha that is a power of two, so that the sigmoid's argument is exact; gates of many sizes, to where it leaves float32. What stands before the
    rounding to bfloat16 may be 2^-21.5 of the value away (the sigmoid 2^-22.3, three roundings of 2^-24; the hardware's exponential gives zero below 2^-126): only a value that
    near to the middle between two bfloat16 may be rounded to the other one. (Where the argument is rounded, that alone moves the sigmoid by |alpha g| 2^-24 of it.)"""
    M, N, K = 700, 1000, 32
    g = torch.Generator().manual_seed(3)
    a, w = torch.zeros(M, K), torch.zeros(2 * N, K)
    a[:, 0] = torch.randn(M, generator=g).exp()
    w[:, 0] = torch.randn(2 * N, generator=g)
    a, w = a.to(torch.bfloat16).to(DEV), w.to(torch.bfloat16).to(DEV)
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    ops._check(ops.library().fw_gemm_mfma_big_tile_clamped(ops._p(a), ops._p(w), ops._p(out), M, N, K, *tile, limit, alpha, shift, ops._stream()))
    sums = a[:, :1].double() * w[:, 0].double()
    gate, up = sums[:, :N].clamp(max=limit), sums[:, N:].clamp(-limit, limit)
    want = gate * torch.sigmoid(alpha * gate) * (up + shift)
    slack = 2.0 ** -21.5 * want.abs() + 2.0 ** -125 * (gate * (up + shift)).abs() + 2.0 ** -126
    assert ((out.double() >= (want - slack).to(torch.bfloat16).double()) & (out.double() <= (want + slack).to(torch.bfloat16).double())).all()
