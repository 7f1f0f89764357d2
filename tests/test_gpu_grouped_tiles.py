"""The experts' grouped product of a prompt on every tile that its rule chooses: the tile is the one named, places that end inside it, features and K that end inside a tile or
a slab, experts without a place, rows by place and by name."""

import ctypes

import numpy as np
import pytest
import torch

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    return module


@pytest.mark.gpu
@pytest.mark.parametrize("gated,rows,experts,top,N,K,tile", [
    (0, 150, 3, 1, 130, 544, (64, 128)), (0, 1600, 16, 2, 1500, 96, (128, 128)), (0, 150, 3, 1, 130, 96, (128, 192)), (0, 2600, 8, 2, 1000, 2080, (128, 256)),
    (0, 700, 8, 2, 200, 96, (192, 192)), (0, 1600, 16, 2, 2050, 544, (192, 256)), (0, 2000, 16, 2, 2050, 544, (256, 256)),
    (1, 150, 3, 1, 130, 96, (64, 128)), (1, 1600, 8, 2, 2050, 96, (128, 128)), (1, 500, 16, 2, 1500, 2080, (128, 192)), (1, 1200, 4, 2, 1000, 544, (128, 256)),
    (1, 700, 8, 2, 2050, 544, (192, 192)), (1, 900, 4, 2, 2050, 2080, (192, 256)), (1, 1600, 16, 2, 1500, 1056, (256, 256))])
@pytest.mark.parametrize("skewed", [False, True])
def test_every_grouped_tile(ops, gated, rows, experts, top, N, K, tile, skewed):
    found = ctypes.c_int(0), ctypes.c_int(0)
    lib, places = ops.library(), rows * top
    tall = lib.fw_grouped_gemm_large_fits(gated, rows, places, experts, N, K)
    ops._check(lib.fw_grouped_gemm_tile(gated, places, experts, N, K, tall, *map(ctypes.byref, found)))
    assert (found[0].value, found[1].value) == tile
    print(gated, rows, experts, top, N, K, tile, skewed, flush=True)
    rng = np.random.default_rng(rows + N)
    weight = 1.0 / (1.0 + np.arange(experts)) if skewed else np.ones(experts)
    if skewed and experts > top + 2:
        weight[experts // 2] = 0.0          # an expert without a place
    chosen = np.stack([rng.choice(experts, top, replace=False, p=weight / weight.sum()) for _ in range(rows)]).astype(np.int32)
    begin, place_row, _ = ops.moe_arrange(torch.from_numpy(chosen).to(DEV), experts)
    g = torch.Generator().manual_seed(K)
    a = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(experts, 2 * N if gated else N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    out_dtype = torch.bfloat16 if gated else torch.float32
    got = ops.grouped_gemm(a, place_row, w, begin, places, gated=bool(gated), out_dtype=out_dtype)
    own = a.index_select(0, place_row[:places].long())
    assert torch.equal(ops.grouped_gemm(own, None, w, begin, places, gated=bool(gated), out_dtype=out_dtype), got)
    b = begin.tolist()
    for e in range(experts):
        x, part = own[b[e]:b[e + 1]].double(), got[b[e]:b[e + 1]].double()
        # products of bfloat16 are exact in float32: K + 16 rounded sums, at most that many 2^-24 of the sum of their sizes
        exact, limit = x @ w[e].double().T, (K + 16) * 2.0 ** -24 * (x.abs() @ w[e].double().abs().T)
        if gated:
            gate, up, lg, lu = exact[:, :N], exact[:, N:], limit[:, :N], limit[:, N:]
            exact = gate * torch.sigmoid(gate) * up
            limit = 1.13 * lg * (up.abs() + lu) + gate.abs() * lu + 2.0 ** -20 * (gate * up).abs() + 2.0 ** -8 * exact.abs() + 2.0 ** -133
        assert ((part - exact).abs() <= limit).all()
