"""What the products take and refuse at the far ends of their sizes."""

import pytest

F32, BF16 = 0, 1


@pytest.mark.parametrize("gated,K", [(0, 32), (1, 32), (0, 40)])
def test_a_grouped_product_of_too_many_tiles_is_refused(gated, K):
    """Before anything is launched, on either path (K a multiple of 32: straight to LDS; else through registers)."""
    from flyweight_amd.kernels import ops
    lib = ops.library()
    places, experts, N = 1 << 30, 1, 1 << 20        # 2^23 tiles of places times 2^13 of features
    status = lib.fw_grouped_gemm(None, BF16, 1, None, None, BF16, None, None, BF16 if gated else F32, gated, places, experts, N, K,
                                 0.0, 1.0, 0.0, None)
    assert status == -1 and b"too many tiles" in lib.fw_last_error()
