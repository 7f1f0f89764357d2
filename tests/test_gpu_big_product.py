"""The product on tiles of 256 rows: every number of slabs of K up to where its turns repeat (its four stages half full, full, one
turn, several), every shape of tile, rows and features that end inside one, its three epilogues."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, BF16 = 0, 1
STORE, ADD, GATED = 0, 1, 2


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    return module


def big(ops, a, w, out, mode, N):
    M, K = a.shape
    entry = ops.library().fw_gemm_mfma_big
    ops._check(entry(ops._p(a), ops._p(w), None, ops._p(out), F32 if out.dtype == torch.float32 else BF16, mode, M, N, K, ops._stream()))
    return out


def draw(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def bound(a, w):
    """Products of bfloat16 are exact in float32: K + 16 rounded sums, at most that many 2^-24 of the sum of the products' sizes."""
    return (a.shape[1] + 16) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


# (rows, features) for each tile: 256 x 256, 256 x 192, 128 x 256, 128 x 192 by the count of rounds, and one row of one feature
@pytest.mark.parametrize("M,N", [(256, 512), (300, 185), (129, 257), (77, 190), (1, 1)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192, 288, 1056])
def test_every_number_of_slabs(ops, M, N, K):
    a, w = draw(M, K), draw(2 * N, K, seed=1)
    A, W = a.to(DEV), w.to(DEV)
    exact, limit = a.double() @ w.double().T, bound(a, w)
    plain = big(ops, A, W[:N], torch.empty(M, N, device=DEV), STORE, N).cpu().double()
    assert ((plain - exact[:, :N]).abs() <= limit[:, :N]).all()
    residual = torch.randn(M, N, generator=torch.Generator().manual_seed(3))
    total = big(ops, A, W[:N], residual.to(DEV), ADD, N).cpu().double()
    assert ((total - exact[:, :N] - residual.double()).abs() <= limit[:, :N] + 2.0 ** -23 * total.abs()).all()
    gate, up = exact[:, :N], exact[:, N:]
    want = gate * torch.sigmoid(gate) * up
    got = big(ops, A, W, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), GATED, N).cpu().double()
    # |d silu| <= 1.1 |d gate|, |silu| <= |gate|; the hardware's exponential and reciprocal 2^-20; one rounding to bfloat16
    slack = 1.1 * limit[:, :N] * (up.abs() + limit[:, N:]) + gate.abs() * limit[:, N:] + 2.0 ** -20 * want.abs() + 2.0 ** -8 * want.abs() + 2.0 ** -133
    assert ((got - want).abs() <= slack).all()


def test_a_width_beyond_its_offsets_goes_elsewhere(ops):
    rows, columns = ctypes.c_int(0), ctypes.c_int(0)
    assert ops.library().fw_gemm_mfma_big_tiles(0, 4096, 8192, 1 << 22) > 0
    assert ops.library().fw_gemm_mfma_big_tiles(0, 4096, 8192, (1 << 22) + 32) == 0
    assert ops.library().fw_gemm_mfma_big_plan(0, 4096, 8192, (1 << 22) + 32, ctypes.byref(rows), ctypes.byref(columns)) == 0


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("M,N", [(300, 185), (130, 184), (129, 1), (1, 2), (700, 8193)])
def test_two_byte_outputs_of_any_width_and_place(ops, M, N, shift):
    """Pairs of columns as one word where rows and output lie at multiples of four bytes, else every element by itself; the places around
    the output stay as they are."""
    K = 96
    a, w = draw(M, K), draw(2 * N, K, seed=1)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2))
    A, W, B = a.to(DEV), w.to(DEV), bias.to(DEV)
    exact, limit = a.double() @ w.double().T, bound(a, w)
    gate, up = exact[:, :N], exact[:, N:]

    def run(mode, code, with_bias):
        room = torch.full((M * N + 8,), 7.0, device=DEV, dtype=torch.bfloat16)
        out = room[2 + shift:2 + shift + M * N]
        ops._check(ops.library().fw_gemm_mfma_big(ops._p(A), ops._p(W), ops._p(B) if with_bias else None, ops._p(out), code, mode, M, N, K, ops._stream()))
        assert (room[:2 + shift] == 7.0).all() and (room[2 + shift + M * N:] == 7.0).all()
        return out.view(M, N).cpu().double()

    summed = exact[:, :N] + bias.double()
    assert ((run(STORE, BF16, True) - summed).abs() <= limit[:, :N] + 2.0 ** -8 * summed.abs()).all()
    # (gelu's slope is below 1.13; its short error function is within 1.5e-7, times half of z)
    want = torch.nn.functional.gelu(summed)
    assert ((run(STORE, ops.BF16_GELU, True) - want).abs() <= 1.13 * limit[:, :N] + 1e-6 + 1e-6 * summed.abs() + 2.0 ** -8 * want.abs()).all()
    slack = 1.1 * limit[:, :N] * (up.abs() + limit[:, N:]) + gate.abs() * limit[:, N:] + 2.0 ** -133
    want = gate * torch.sigmoid(gate) * up
    assert ((run(GATED, BF16, False) - want).abs() <= slack + 2.0 ** -7 * want.abs()).all()
    # (the slope of the tanh form is below 1.13 as well)
    want = torch.nn.functional.gelu(gate, approximate="tanh") * up
    assert ((run(GATED, ops.BF16_GEGLU, False) - want).abs() <= 1.03 * slack + 1e-5 * (gate * up).abs() + 2.0 ** -7 * want.abs()).all()
