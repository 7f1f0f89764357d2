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
