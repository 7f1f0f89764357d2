"""What the products take and refuse at the far ends of their sizes."""

import pytest
import torch

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


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 5, (1 << 22) + 64), (3, (1 << 20) + 2, 64)])
def test_rows_beyond_the_tiles_offsets_are_served(M, N, K):
    """Products called by name with rows that are longer than the 32-bit places of their tiles reach. Products of bfloat16 are exact in float32:
    K + 16 rounded sums, at most that many 2^-24 of the sum of the products' sizes."""
    from flyweight_amd.kernels import ops
    g = torch.Generator().manual_seed(K)
    a, w = torch.randn(M, K, generator=g).to(torch.bfloat16), torch.randn(2 * N, K, generator=g).to(torch.bfloat16)
    A, W = a.cuda(), w.cuda()
    exact = torch.cat([a.double() @ part.double().T for part in w.split(1 << 18)], 1)
    limit = (K + 16) * 2.0 ** -24 * torch.cat([a.double().abs() @ part.double().abs().T for part in w.split(1 << 18)], 1)
    old = torch.randn(M, N, generator=g)

    def big(mode, out):
        ops._check(ops.library().fw_gemm_mfma_big(ops._p(A), ops._p(W), None, ops._p(out), ops._code(out.dtype), mode, M, N, K, ops._stream()))
        return out.cpu().double()

    results = [(big(0, torch.empty(M, N, device="cuda")), 0.0), (big(1, old.cuda()), old.double())]
    for columns in (64, 128):
        results.append((ops.gemm_deep(A, W[:N], out_dtype=torch.float32, columns=columns).cpu().double(), 0.0))
        results.append((ops.gemm_deep(A, W[:N], accumulate_into=old.cuda(), columns=columns).cpu().double(), old.double()))
    for found, before in results:
        assert ((found - exact[:, :N] - before).abs() <= limit[:, :N] + 2.0 ** -23 * found.abs()).all()
    gate, up = exact[:, :N], exact[:, N:]
    want = gate * torch.sigmoid(gate) * up
    # |d silu| <= 1.1 |d gate|, |silu| <= |gate|; the hardware's exponential and reciprocal 2^-20; one rounding to bfloat16
    slack = 1.1 * limit[:, :N] * (up.abs() + limit[:, N:]) + gate.abs() * limit[:, N:] + 2.0 ** -7 * want.abs() + 2.0 ** -133
    assert ((big(2, torch.empty(M, N, device="cuda", dtype=torch.bfloat16)) - want).abs() <= slack).all()
