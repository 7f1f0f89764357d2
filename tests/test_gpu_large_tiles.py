"""The product on the large tile that the call names: every tile, with edges in rows and features, every number of slabs around its stages, its epilogues and K cut
into slices."""

import ctypes

import pytest
import torch

F32, BF16, BF16_GELU, BF16_GEGLU = 0, 1, 2, 3
STORE, ADD, GATED = 0, 1, 2
DEV = "cuda:0"
TILES = [(64, 128, 1), (64, 128, 2), (128, 128, 1), (128, 128, 2), (192, 128, 1), (64, 192, 1), (128, 192, 1), (192, 192, 1), (256, 192, 1), (128, 256, 1),
         (192, 256, 1), (256, 256, 1), (256, 320, 1)]
CUT = [(64, 128), (128, 128), (128, 256)]


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    return module


def call(ops, a, w, bias, out, code, mode, N, tile, slices=1):
    (M, K), lib = a.shape, ops.library()
    bytes_, counters = ctypes.c_size_t(0), ctypes.c_int(0)
    ops._check(lib.fw_gemm_mfma_big_tile_needs(mode, M, N, K, *tile, slices, ctypes.byref(bytes_), ctypes.byref(counters)))
    workspace = torch.full((max(bytes_.value // 4, 1),), float("nan"), device=DEV)
    tickets = torch.zeros(max(counters.value, 1), dtype=torch.int32, device=DEV)
    print(M, N, K, mode, tile, slices, flush=True)
    ops._check(lib.fw_gemm_mfma_big_tile(ops._p(a), ops._p(w), ops._p(bias), ops._p(out), code, mode, M, N, K, *tile, slices, ops._p(workspace), bytes_.value,
                                         ops._p(tickets), counters.value, ops._stream()))
    assert not tickets.any()        # left at zero
    return out


def draw(M, rows_w, K):
    g = torch.Generator().manual_seed(M * 7 + K)
    a, w = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV), (torch.randn(rows_w, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    exact = a.double() @ w.double().T
    # products of bfloat16 are exact in float32: K + 24 rounded sums (those of up to eight slices among them), at most that many 2^-24 of the sum of their sizes
    return a, w, exact, (K + 24) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("K", [32, 96, 160, 256, 352, 416, 544, 1056])
def test_every_tile(ops, tile, K):
    rows, columns, _ = tile
    for M, N in ((rows - 1, columns - 6), (2 * rows + 3, 2 * columns + 2)):
        a, w, exact, limit = draw(M, N, K)
        bias, old = torch.randn(N, device=DEV), torch.randn(M, N, device=DEV)
        want, room = exact + bias.double(), limit + 2.0 ** -23 * (exact.abs() + bias.double().abs())
        assert ((call(ops, a, w, bias, torch.empty(M, N, device=DEV), F32, STORE, N, tile).double() - want).abs() <= room).all()
        got = call(ops, a, w, bias, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), BF16, STORE, N, tile)
        assert ((got.double() - want).abs() <= room + 2.0 ** -8 * want.abs()).all()
        got = call(ops, a, w, None, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), BF16_GELU, STORE, N, tile).double()
        # |gelu'| < 1.13, the quick form within 1.5e-7 |z|
        assert ((got - torch.nn.functional.gelu(exact)).abs() <= 1.13 * limit + 4e-7 * exact.abs() + 1e-6 + 2.0 ** -8 * got.abs()).all()
        total = call(ops, a, w, None, old.clone(), F32, ADD, N, tile).double()
        assert ((total - exact - old.double()).abs() <= limit + 2.0 ** -23 * total.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("K", [32, 160, 352, 544])
def test_every_gated_tile(ops, tile, K):
    rows, columns, _ = tile
    for M, N in ((rows - 1, columns // 2 - 6), (rows + 3, columns + 5), (rows + 1, 3 * columns // 2)):     # (odd: every element leaves by itself)
        a, w, exact, limit = draw(M, 2 * N, K)
        gate, up, off = exact[:, :N], exact[:, N:], limit
        for code, unit in ((BF16, torch.nn.functional.silu), (BF16_GEGLU, lambda g: torch.nn.functional.gelu(g, approximate="tanh"))):
            got = call(ops, a, w, None, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), code, GATED, N, tile).double()
            want = unit(gate) * up
            # both units' slopes are below 1.13, their sizes below |g|; the hardware's exponential and reciprocal 2^-20 of |g|; one rounding to bfloat16
            slack = 1.13 * off[:, :N] * (up.abs() + off[:, N:]) + gate.abs() * off[:, N:] + 2.0 ** -20 * (gate * up).abs() + 2.0 ** -8 * want.abs() + 2.0 ** -133
            assert ((got - want).abs() <= slack).all()


@pytest.mark.gpu
@pytest.mark.parametrize("edges", CUT)
@pytest.mark.parametrize("slices", [2, 3, 4, 5, 7, 8])
def test_every_number_of_slices(ops, edges, slices):
    tile, M, N = (*edges, 1), edges[0] + 3, edges[1] + 2
    for K in (64 * slices, 64 * (slices - 1) + 32, 192 * slices - 96):       # slices of one slab, a last one of half a slab, of three
        a, w, exact, limit = draw(M, N, K)
        bias, old = torch.randn(N, device=DEV), torch.randn(M, N, device=DEV)
        found = call(ops, a, w, bias, torch.empty(M, N, device=DEV), F32, STORE, N, tile, slices)
        assert ((found.double() - exact - bias.double()).abs() <= limit + 2.0 ** -23 * (exact.abs() + bias.double().abs())).all()
        for _ in range(3):          # whichever workgroup came last
            assert torch.equal(call(ops, a, w, bias, torch.empty(M, N, device=DEV), F32, STORE, N, tile, slices), found)
        got = call(ops, a, w, bias, torch.empty(M, N, device=DEV, dtype=torch.bfloat16), BF16, STORE, N, tile, slices)
        assert torch.equal(got, found.to(torch.bfloat16))
        total = call(ops, a, w, None, old.clone(), F32, ADD, N, tile, slices).double()
        assert ((total - exact - old.double()).abs() <= limit + 2.0 ** -23 * total.abs()).all()


def test_what_is_no_tile_is_refused(ops):
    bytes_, counters = ctypes.c_size_t(0), ctypes.c_int(0)
    needs = lambda *shape: ops.library().fw_gemm_mfma_big_tile_needs(*shape, ctypes.byref(bytes_), ctypes.byref(counters))      # noqa: E731
    for shape in ((0, 64, 128, 64, 96, 128, 1, 1), (0, 64, 128, 64, 128, 320, 1, 1), (0, 64, 128, 64, 192, 128, 2, 1), (0, 64, 128, 64, 64, 128, 3, 1),
                  (2, 64, 128, 4096, 64, 128, 1, 2), (0, 64, 128, 4096, 64, 128, 2, 2), (0, 64, 128, 4096, 192, 128, 1, 2), (0, 64, 128, 4096, 64, 128, 1, 9),
                  (0, 64, 128, 64, 64, 128, 1, 2), (0, 64, 128, 40, 64, 128, 1, 1), (0, 64, 128, (1 << 22) + 32, 64, 128, 1, 1), (0, 64, (1 << 20) + 1, 64, 64, 128, 1, 1),
                  (3, 64, 128, 64, 64, 128, 1, 1), (0, 0, 128, 64, 64, 128, 1, 1)):
        assert needs(*shape) == -1, shape
    assert needs(0, 65, 129, 4096, 64, 128, 1, 4) == 0 and (bytes_.value, counters.value) == (4 * 4 * 64 * 128 * 4, 4)
    # too little workspace, too few counters: refused before anything is launched
    for size, count in ((1 << 20, 0), (0, 4)):
        assert ops.library().fw_gemm_mfma_big_tile(16, 16, None, 16, F32, STORE, 65, 129, 4096, 64, 128, 1, 4, 16, size, 16, count, None) == -1


@pytest.mark.parametrize("mode,M,N,K,tile", [
    (2, 2048, 4608, 1024, (256, 320, 1, 1)), (2, 2048, 8192, 2048, (256, 256, 1, 1)), (2, 2048, 2048, 2048, (128, 256, 1, 1)), (2, 90, 7168, 2048, (64, 128, 1, 1)),
    (1, 2048, 2048, 8192, (128, 128, 1, 1)), (1, 2048, 1024, 1024, (64, 128, 1, 1)), (1, 801, 2048, 7168, (128, 128, 1, 2)), (0, 2048, 6144, 2048, (256, 192, 1, 1)),
    (0, 2048, 3072, 2048, (128, 192, 1, 1)), (0, 120, 2048, 2048, None), (0, 8192, 2048, 520, None), (0, 512, (1 << 20) + 2, 64, None), (0, 512, 64, (1 << 22) + 32, None)])
def test_products_by_a_models_weights_take_the_tile_that_was_the_fastest(ops, mode, M, N, K, tile):
    found = ops.large_tile(mode, M, N, K)
    assert (found[:4] if found else None) == tile
