"""The product on large tiles: every number of slabs of K up to where its turns repeat, every shape of tile, rows and features that end inside one,
its epilogues in both output types."""

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


def draw(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def bound(a, w):
    """Products of bfloat16 are exact in float32: K + 16 rounded sums, at most that many 2^-24 of the sum of the products' sizes."""
    return (a.shape[1] + 16) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


# (rows, features) for each shape of tile, whole and ending inside one, the tile, and the features of the gated product on its 256 rows
TILES = [(2048, 6144, (256, 192)), (1537, 6100, (256, 192)), (1536, 8192, (256, 256)), (1500, 8201, (256, 256)), (1920, 4096, (128, 256)),
         (1900, 4001, (128, 256)), (256, 384, (128, 192)), (129, 257, (128, 192)), (1, 1, (128, 192))]


@pytest.mark.parametrize("M,N,tile", TILES)
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192, 256, 288, 352, 448, 544])
def test_every_number_of_slabs(ops, M, N, tile, K):
    """Every number of slabs of K up to where the turns of the loop repeat: its two to four stages half full, full, one turn, several, the last slab whole and half."""
    rows, columns = ctypes.c_int(0), ctypes.c_int(0)
    for mode in (STORE, ADD):
        assert ops.library().fw_gemm_mfma_big_plan(mode, M, N, K, ctypes.byref(rows), ctypes.byref(columns)) > 0
        assert (rows.value, columns.value) == tile
    half = (N + 1) // 2                         # (of the gated product: the other rows of w)
    a, w = draw(M, K), draw(max(N, 2 * half), K, seed=1)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2))
    residual = torch.randn(M, N, generator=torch.Generator().manual_seed(3))
    A, W, B = a.to(DEV), w.to(DEV), bias.to(DEV)
    # (the products and their bounds on the GPU in float64, by the library: 16 million elements of a large one)
    exact = A.double() @ W.double().T
    limit = (K + 16) * 2.0 ** -24 * (A.double().abs() @ W.double().abs().T)

    def run(mode, out, width, with_bias=False):
        entry = ops.library().fw_gemm_mfma_big
        ops._check(entry(ops._p(A), ops._p(W), ops._p(B) if with_bias else None, ops._p(out), F32 if out.dtype == torch.float32 else BF16, mode, M,
                         width, K, ops._stream()))
        return out.double()

    want, room = exact[:, :N] + B.double(), limit[:, :N] + 2.0 ** -23 * (exact[:, :N].abs() + B.double().abs())
    assert ((run(STORE, torch.empty(M, N, device=DEV), N, True) - want).abs() <= room).all()
    assert ((run(STORE, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), N, True) - want).abs() <= room + 2.0 ** -8 * want.abs()).all()
    total = run(ADD, residual.to(DEV), N)
    assert ((total - exact[:, :N] - residual.to(DEV).double()).abs() <= limit[:, :N] + 2.0 ** -23 * total.abs()).all()
    gate, up, gate_off, up_off = exact[:, :half], exact[:, half:2 * half], limit[:, :half], limit[:, half:2 * half]
    want = gate * torch.sigmoid(gate) * up
    # |d silu| <= 1.1 |d gate|, |silu| <= |gate|; the hardware's exponential and reciprocal 2^-20; one rounding to bfloat16
    slack = 1.1 * gate_off * (up.abs() + up_off) + gate.abs() * up_off + 2.0 ** -20 * want.abs() + 2.0 ** -8 * want.abs() + 2.0 ** -133
    assert ((run(GATED, torch.empty(M, half, device=DEV, dtype=torch.bfloat16), half) - want).abs() <= slack).all()


def test_a_width_beyond_its_offsets_goes_elsewhere(ops):
    plan = lambda M, N, K: ops.library().fw_gemm_mfma_big_plan(0, M, N, K, ctypes.byref(ctypes.c_int(0)), ctypes.byref(ctypes.c_int(0)))    # noqa: E731
    assert plan(4096, 8192, 1 << 22) > 0
    assert plan(4096, 8192, (1 << 22) + 32) == 0
    assert plan(4096, 1 << 20, 64) > 0
    assert plan(4096, (1 << 20) + 1, 64) == 0


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


@pytest.mark.parametrize("rows,experts,top,K,N", [(384, 6, 2, 1536, 200), (383, 6, 2, 1536, 200), (700, 4, 1, 1568, 129), (513, 4, 2, 2048, 128),
                                                  (384, 6, 2, 1504, 200), (300, 3, 1, 1536, 130), (640, 5, 3, 96, 257)])
def test_grouped_product_on_slabs_of_either_depth(ops, rows, experts, top, K, N):
    """Both sides of the rule: a long K and experts of 128 places in the mean, or slabs of half the depth; whole and half last slabs."""
    generator = torch.Generator().manual_seed(rows + K)
    chosen = torch.rand(rows, experts, generator=generator).topk(top, -1).indices.int().to(DEV)
    begin, place_row, pair_place = ops.moe_arrange(chosen, experts)
    a, w = draw(rows, K).to(DEV), draw(experts, 2 * N, K, seed=1).to(DEV)
    gated = ops.grouped_gemm(a, place_row, w, begin, rows * top, gated=True, out_dtype=torch.bfloat16).double()
    plain = ops.grouped_gemm(a, place_row, w, begin, rows * top, gated=False, out_dtype=torch.float32).double()
    first, A = begin.tolist(), a.double()[place_row.long()]
    for e in range(experts):
        here = slice(first[e], first[e + 1])
        exact = A[here] @ w[e].double().T
        limit = (K + 16) * 2.0 ** -24 * (A[here].abs() @ w[e].double().abs().T)
        assert ((plain[here] - exact).abs() <= limit).all()
        gate, up, gate_off, up_off = exact[:, :N], exact[:, N:], limit[:, :N], limit[:, N:]
        want = gate * torch.sigmoid(gate) * up
        slack = 1.1 * gate_off * (up.abs() + up_off) + gate.abs() * up_off + 2.0 ** -20 * want.abs() + 2.0 ** -8 * want.abs() + 2.0 ** -133
        assert ((gated[here] - want).abs() <= slack).all()


# (rows, features, K, slices): whole tiles and ragged ones, slices of equal and of unequal length, the last one with half a slab
@pytest.mark.parametrize("M,N,K,slices", [(256, 512, 1024, 2), (2048, 2048, 2080, 2), (1111, 2048, 8192, 3), (129, 257, 1536, 3), (1, 1, 1568, 3), (1000, 2560, 3104, 3),
                                          (130, 8191, 1056, 2)])
def test_large_tiles_with_k_cut_over_workgroups(ops, M, N, K, slices):
    need_bytes, need_counters, cut = ops._big_split_needs(STORE, M, N, K)
    assert cut == slices and ops._big_split_needs(GATED, M, N, K) == (0, 0, 0)
    a, w = draw(M, K).to(DEV), draw(N, K, seed=1).to(DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2)).to(DEV)
    residual = torch.randn(M, N, generator=torch.Generator().manual_seed(3)).to(DEV)
    exact = a.double() @ w.double().T
    limit = (K + 16) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    workspace = torch.full((need_bytes // 4,), float("nan"), device=DEV)
    counters = torch.zeros(need_counters, dtype=torch.int32, device=DEV)

    def run(mode, out, with_bias=False, code=None):
        ops._check(ops.library().fw_gemm_mfma_big_split(ops._p(a), ops._p(w), ops._p(bias) if with_bias else None, ops._p(out), code or ops._code(out.dtype), mode, M,
                                                        N, K, ops._p(workspace), need_bytes, ops._p(counters), counters.numel(), ops._stream()))
        return out

    want = exact + bias.double()
    room = limit + 2.0 ** -23 * (exact.abs() + bias.double().abs())
    stored = run(STORE, torch.empty(M, N, device=DEV), True)
    assert ((stored.double() - want).abs() <= room).all()
    assert ((run(STORE, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), True).double() - want).abs() <= room + 2.0 ** -8 * want.abs()).all()
    # (gelu's slope is below 1.13; its short error function is within 1.5e-7, times half of z)
    unit = run(STORE, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), True, ops.BF16_GELU).double()
    gelu = torch.nn.functional.gelu(want)
    assert ((unit - gelu).abs() <= 1.13 * room + 1e-6 + 1e-6 * want.abs() + 2.0 ** -8 * gelu.abs()).all()
    total = run(ADD, residual.clone()).double()
    assert ((total - exact - residual.double()).abs() <= limit + 2.0 ** -23 * total.abs()).all()
    # whichever workgroup of a tile ends last, the slices are added in their order, and the counters are left at zero
    for _ in range(3):
        assert torch.equal(run(STORE, torch.empty(M, N, device=DEV), True), stored)
    assert not counters.any()


def test_large_tiles_with_k_cut_refuse_what_they_do_not_take(ops):
    a, w, out = draw(128, 1024).to(DEV), draw(256, 1024, seed=1).to(DEV), torch.empty(128, 256, device=DEV)
    call = lambda K, mode, bytes_, counters: ops._check(ops.library().fw_gemm_mfma_big_split(ops._p(a), ops._p(w), None, ops._p(out), F32, mode, 128, 256, K, ops._p(out),      # noqa: E731,E501
                                                                                             bytes_, ops._p(counters), counters.numel(), ops._stream()))
    one = torch.zeros(1, dtype=torch.int32, device=DEV)
    for K, mode, bytes_, counters, text in [(1000, 0, 1 << 20, one, "is not cut"), (992, 0, 1 << 20, one, "is not cut"), (1024, 2, 1 << 20, one, "is not cut"),
                                            (1024, 0, 1000, one, "bytes of workspace"), (1024, 0, 1 << 20, one[:0], "counters")]:
        with pytest.raises(ops.KernelError, match=text):
            call(K, mode, bytes_, counters)
