"""The experts' weights, held once: what a mixture keeps of them, and the grouped products by operand tiles alone, bit for bit those by rows."""

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
@pytest.mark.parametrize("hidden,intermediate", [(512, 768), (256, 200), (320, 72), (264, 96)])       # whole tiles of rows, half ones, K no multiple of 32 on either side
def test_a_mixture_holds_its_experts_once(monkeypatch, hidden, intermediate):
    """... whatever memory is free when it is bound, and nothing else: a cache that fits beside the weights still fits."""
    from flyweight_amd.config.spec import PartSpec
    from flyweight_amd.parts.base import build_part
    experts, held = 24, {}
    for free in (1 << 30, 1 << 38):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (free, 288 << 30))
        part = build_part("ffn", PartSpec("moe_swiglu", {"hidden_size": hidden, "intermediate_size": intermediate, "num_experts": experts, "top": 3}, prefix=""))
        g = torch.Generator().manual_seed(1)
        tensors = {name: torch.randn(decl.shape, generator=g).to(torch.float32 if "router.b" in name else torch.bfloat16).to(DEV) for name, decl in part.tensors().items()}
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        part.bind(tensors, torch.bfloat16, torch.device(DEV))
        held[free] = torch.cuda.memory_allocated() - before
    weights = experts * 3 * hidden * intermediate * 2
    router = 2 * experts * hidden * 2 + 16 * hidden * 2
    assert len(set(held.values())) == 1 and weights <= held[free] <= weights + router + 2 * 15 * max(hidden, intermediate) * 2 + (1 << 14)


@pytest.mark.gpu
@pytest.mark.parametrize("gated,rows,experts,top,N,K", [
    (0, 1, 4, 1, 33, 32), (0, 40, 4, 2, 130, 96), (1, 40, 4, 2, 72, 544), (1, 3, 5, 2, 31, 160),                 # tiles of 32 places; few places
    (0, 150, 3, 1, 130, 544), (0, 1600, 16, 2, 1500, 96), (0, 150, 3, 1, 130, 96), (0, 2600, 8, 2, 1000, 2080), (0, 700, 8, 2, 200, 96), (0, 1600, 16, 2, 2050, 544),
    (0, 2000, 16, 2, 2050, 544), (1, 150, 3, 1, 130, 96), (1, 1600, 8, 2, 2050, 96), (1, 500, 16, 2, 1500, 2080), (1, 1200, 4, 2, 1000, 544), (1, 700, 8, 2, 2050, 544),
    (1, 900, 4, 2, 2050, 2080), (1, 1600, 16, 2, 1500, 1056),                                                    # every tile that goes straight to LDS
    (0, 120, 2, 1, 65, 16416), (1, 120, 2, 1, 40, 16416), (1, 300, 4, 2, 129, 160), (1, 130, 3, 1, 7, 64)])      # through registers: the longest K; narrow
def test_by_tiles_alone_as_by_rows(ops, gated, rows, experts, top, N, K):
    print(gated, rows, experts, top, N, K, flush=True)
    begin, place_row, _ = step(ops, rows, experts, top, seed=rows)
    g = torch.Generator().manual_seed(K + N)
    a = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(experts, 2 * N if gated else N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    held, places, dtype = ops.ExpertWeights(experts, lambda e: w[e]), rows * top, torch.bfloat16 if gated else torch.float32
    assert held.rows is None and held.shape == tuple(w.shape) and torch.equal(held.tiled, ops.tile_weights(w.view(-1, K)))
    own = a.index_select(0, place_row[:places].long())
    odd = torch.empty(a.numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view(rows, K).copy_(a)       # at no multiple of 16 bytes
    for glu in (None, (1.0, 1.702, 1.0)) if gated else (None,):
        by_rows = ops.grouped_gemm(a, place_row, w, begin, places, gated=bool(gated), out_dtype=dtype, glu=glu)
        for operand, named in ((a, place_row), (own, None), (odd, place_row)):
            assert torch.equal(ops.grouped_gemm(operand, named, held, begin, places, gated=bool(gated), out_dtype=dtype, glu=glu), by_rows)


@pytest.mark.gpu
def test_what_operand_tiles_do_not_take_is_refused(ops):
    begin, place_row, _ = step(ops, 4, 2, 1)
    w = torch.zeros(2, 32, 64, dtype=torch.bfloat16, device=DEV)
    held = ops.ExpertWeights(2, lambda e: w[e])
    with pytest.raises(ops.KernelError, match="operand tiles"):
        ops.grouped_gemm(torch.zeros(4, 64, device=DEV), place_row, held, begin, 4, gated=False, out_dtype=torch.float32)
    with pytest.raises(ops.KernelError, match="operand tiles"):
        ops.grouped_gemm(torch.zeros(4, 64, dtype=torch.bfloat16, device=DEV), place_row, held, begin, 4, gated=False, out_dtype=torch.bfloat16)
    with pytest.raises(ops.KernelError, match="grouped_gemm: a is"):
        ops.grouped_gemm(torch.zeros(4, 96, dtype=torch.bfloat16, device=DEV), place_row, held, begin, 4, gated=False, out_dtype=torch.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K", [(4, 64), (300, 64), (9, 72)])
def test_gated_float32_outputs_of_bfloat16_rows(ops, rows, K):
    """... hold float32 (K + 16 rounded sums of exact products, the unit's slopes as elsewhere), and the rows behind them are untouched."""
    experts, N = 3, 24
    begin, place_row, _ = step(ops, rows, experts, 2)
    g = torch.Generator().manual_seed(rows)
    a, w = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(DEV), (torch.randn(experts, 2 * N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    got, own, b = ops.grouped_gemm(a, place_row, w, begin, 2 * rows, gated=True, out_dtype=torch.float32), a.index_select(0, place_row.long()), begin.tolist()
    for e in range(experts):
        x, part = own[b[e]:b[e + 1]].double(), got[b[e]:b[e + 1]].double()
        exact, limit = x @ w[e].double().T, (K + 16) * 2.0 ** -24 * (x.abs() @ w[e].double().abs().T)
        gate, up, lg, lu = exact[:, :N], exact[:, N:], limit[:, :N], limit[:, N:]
        want = gate * torch.sigmoid(gate) * up
        assert ((part - want).abs() <= 1.13 * lg * (up.abs() + lu) + gate.abs() * lu + 2.0 ** -20 * (gate * up).abs() + 2.0 ** -133).all()
