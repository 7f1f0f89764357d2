"""The experts' grouped product of steps with a few places an expert, by weights in operand tiles: edges of places, features and K, both units, experts without a place."""

import numpy as np
import pytest
import torch

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    return module


def step(ops, rows, experts, top, seed=0):
    rng = np.random.default_rng(seed)
    chosen = np.stack([rng.permutation(experts)[:top] for _ in range(rows)]).astype(np.int32)
    return ops.moe_arrange(torch.from_numpy(chosen).to(DEV), experts)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,experts,top,K,N", [
    (1, 4, 1, 32, 16), (1, 4, 4, 96, 33), (3, 5, 2, 160, 31), (9, 4, 2, 512, 129), (31, 4, 2, 544, 40), (33, 2, 1, 1056, 72),       # one, two and three tiles of places an expert
    (30, 70, 3, 64, 24), (64, 8, 2, 2048, 48), (17, 1, 1, 640, 7)])
@pytest.mark.parametrize("place_tiles", [1, 2])
@pytest.mark.parametrize("glu", [None, (1.0, 1.702, 1.0)])
def test_few_places_an_expert(ops, monkeypatch, rows, experts, top, K, N, place_tiles, glu):
    monkeypatch.setattr(ops, "grouped_few_tiles", lambda places, experts: place_tiles)
    g = torch.Generator().manual_seed(rows + N)
    a = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(experts, 2 * N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    begin, place_row, _ = step(ops, rows, experts, top, seed=rows)
    places, tiled = rows * top, ops.tile_weights(w.view(-1, K))
    print(rows, experts, top, K, N, place_tiles, glu, flush=True)
    gated = ops.grouped_gemm(a, place_row, w, begin, places, gated=True, out_dtype=torch.bfloat16, glu=glu, w_tiled=tiled).double()
    plain = ops.grouped_gemm(a, place_row, w, begin, places, gated=False, out_dtype=torch.float32, w_tiled=tiled).double()
    own = a.index_select(0, place_row[:places].long())
    again = ops.grouped_gemm(own, None, w, begin, places, gated=False, out_dtype=torch.float32, w_tiled=tiled).double()      # rows by place
    b = begin.tolist()
    for e in range(experts):
        x = own[b[e]:b[e + 1]].double()
        # products of bfloat16 are exact in float32: K + 16 rounded sums, at most that many 2^-24 of the sum of their sizes
        exact, limit = x @ w[e].double().T, (K + 16) * 2.0 ** -24 * (x.abs() @ w[e].double().abs().T)
        assert ((plain[b[e]:b[e + 1]] - exact).abs() <= limit).all() and torch.equal(plain[b[e]:b[e + 1]], again[b[e]:b[e + 1]])
        gate, up, lg, lu = exact[:, :N], exact[:, N:], limit[:, :N], limit[:, N:]
        if glu is None:
            want, factor = gate * torch.sigmoid(gate) * up, up.abs() + lu
        else:
            gate, up = gate.clamp(max=glu[0]), up.clamp(-glu[0], glu[0])
            want, factor = gate * torch.sigmoid(glu[1] * gate) * (up + glu[2]), (up + glu[2]).abs() + lu
        # both units' slopes in the gate are below 1.13; the hardware's exponential 2^-20; one rounding to bfloat16
        slack = 1.13 * lg * factor + gate.abs() * lu + 2.0 ** -20 * gate.abs() * factor + 2.0 ** -8 * want.abs() + 2.0 ** -133
        assert ((gated[b[e]:b[e + 1]] - want).abs() <= slack).all()


@pytest.mark.gpu
def test_a_places_sums_do_not_depend_on_the_step(ops, monkeypatch):
    experts, top, K, N, rows = 4, 2, 384, 48, 40
    g = torch.Generator().manual_seed(5)
    a, w = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(DEV), torch.randn(experts, N, K, generator=g).to(torch.bfloat16).to(DEV)
    tiled, rng = ops.tile_weights(w.view(-1, K)), np.random.default_rng(1)
    chosen = torch.from_numpy(np.stack([rng.permutation(experts)[:top] for _ in range(rows)]).astype(np.int32)).to(DEV)

    def run(first, count, place_tiles):
        monkeypatch.setattr(ops, "grouped_few_tiles", lambda places, experts: place_tiles)
        begin, place_row, pair_place = ops.moe_arrange(chosen[first:first + count].contiguous(), experts)
        out = ops.grouped_gemm(a[first:first + count], place_row, w, begin, count * top, gated=False, out_dtype=torch.float32, w_tiled=tiled)
        return out[pair_place.long()]

    everything = run(0, rows, 1)
    for first, count, place_tiles in ((0, 40, 2), (0, 3, 1), (7, 1, 2), (20, 20, 1)):
        assert torch.equal(run(first, count, place_tiles), everything[first:first + count])


@pytest.mark.gpu
@pytest.mark.parametrize("experts,top,K,N", [(4, 2, 1536, 96), (5, 1, 2080, 41), (8, 4, 544, 264)])
@pytest.mark.parametrize("glu", [None, (1.0, 1.702, 1.0)])
def test_a_row_has_the_same_bits_alone_and_among_hundreds(ops, experts, top, K, N, glu):
    """Steps of a few places an expert, of the tiles of 32 places beside them (17 to 23 an expert) and of prompts: every place's sums have one order of k."""
    rows, rng = 200 * experts // top, np.random.default_rng(K)
    g = torch.Generator().manual_seed(K)
    a, w = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(DEV), (torch.randn(experts, 2 * N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    tiled, chosen = ops.tile_weights(w.view(-1, K)), torch.from_numpy(np.stack([rng.permutation(experts)[:top] for _ in range(rows)]).astype(np.int32)).to(DEV)

    def run(first, count):
        begin, place_row, pair_place = ops.moe_arrange(chosen[first:first + count].contiguous(), experts)
        own = a[first:first + count].contiguous()
        return [ops.grouped_gemm(own, place_row, w, begin, count * top, gated=gated, out_dtype=dtype, glu=glu if gated else None, w_tiled=tiled)[pair_place.long()]
                for gated, dtype in ((True, torch.bfloat16), (False, torch.float32))]

    everything, taken = run(0, rows), set()
    for first, count in ((0, 1), (rows - 3, 3), (7, 7 * experts // top), (3, 14 * experts // top), (1, 20 * experts // top)):
        taken.add(ops.grouped_few_tiles(count * top, experts))
        for part, whole in zip(run(first, count), everything):
            assert torch.equal(part, whole[first:first + count])
    assert taken == {0, 1, 2}


@pytest.mark.parametrize("places,experts,tiles", [(1, 32, 1), (256, 32, 1), (257, 32, 2), (512, 32, 2), (513, 32, 0), (8192, 32, 0)])
def test_tiles_of_places(ops, places, experts, tiles):
    assert ops.grouped_few_tiles(places, experts) == tiles
