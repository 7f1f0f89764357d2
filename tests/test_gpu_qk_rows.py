"""Prompts' rows of 64 and 128 channels through the norm, the rotation and the cache write: four channels to a lane and eight rows to a wave give the
bits of one row to a wave, which the same rows in portions of fewer than 64 take."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
HEADS, KV = 5, 3


def run(ops, rows, dim, v_dim, rotary, portions, in_dtype=torch.float32, dtype=torch.bfloat16, normed=True, interleaved=False, q_only=False, scaled=False,
        start=0, apart=0, shift=0):
    """(queries, key pages, value pages) of `rows` rows of three requests, `portions` of them a call."""
    gen = torch.Generator().manual_seed(3)
    width = HEADS * dim if q_only else (HEADS + KV) * dim + KV * v_dim
    whole = torch.randn(rows * (width + apart) + shift, generator=gen).to(DEV, in_dtype)[shift:].view(rows, width + apart)
    qw, kw = ((1 + 0.1 * torch.randn(dim, generator=gen)).to(DEV) if normed else None for _ in range(2))
    angle = torch.rand(rows, max(rotary // 2, 1), generator=gen) * 6
    cos, sin = (angle.cos().to(DEV), angle.sin().to(DEV)) if rotary else (None, None)
    scale = (1 + torch.rand(rows, generator=gen)).to(DEV) if scaled else None
    lengths = [rows // 3, 1, rows - rows // 3 - 1]
    seg = torch.tensor(np.repeat(np.arange(3), lengths), dtype=torch.int32, device=DEV)
    pos = torch.tensor(np.concatenate([start + np.arange(n) for n in lengths]), dtype=torch.int32, device=DEV)
    stride = (start + rows) // 64 + 1
    table = torch.arange(3 * stride, dtype=torch.int32, device=DEV).flip(0).view(3, stride).contiguous()
    k_pages = torch.full((3 * stride, KV, 64, dim), 7.0, dtype=dtype, device=DEV)
    v_pages = torch.full((3 * stride, KV, v_dim, 64), 7.0, dtype=dtype, device=DEV)
    out = []
    for at in range(0, rows, portions):
        part = slice(at, min(rows, at + portions))
        out.append(ops.qk_norm_rope_kv_write(whole[part, :width], HEADS, KV, dim, qw, kw, 1e-5, None if cos is None else cos[part], None if sin is None else sin[part],
                                             rotary, k_pages, v_pages, table, seg[part], pos[part], write_kv=not q_only, v_dim=v_dim, interleaved=interleaved,
                                             q_only=q_only, q_row_scale=None if scale is None else scale[part]))
    return torch.cat(out), k_pages, v_pages


@pytest.mark.parametrize("rows,dim,v_dim,rotary,more", [
    (64, 64, 64, 64, {}), (71, 64, 64, 64, {"start": 5}), (203, 64, 64, 32, {"start": 61, "apart": 4}), (130, 64, 128, 0, {"scaled": True}),
    (65, 64, 64, 64, {"interleaved": True}), (99, 64, 64, 64, {"shift": 1}), (99, 64, 64, 64, {"apart": 3}), (99, 64, 64, 36, {}),
    (64, 128, 128, 64, {"start": 8}), (149, 128, 128, 128, {"scaled": True}), (149, 128, 192, 32, {"interleaved": True, "normed": False}),
    (80, 128, 64, 8, {"in_dtype": torch.bfloat16}), (80, 128, 128, 64, {"dtype": torch.float32}), (80, 64, 64, 64, {"dtype": torch.float32, "start": 16}),
    (67, 128, 128, 64, {"q_only": True}), (67, 64, 64, 64, {"q_only": True, "in_dtype": torch.bfloat16}), (90, 64, 64, 16, {"normed": False})])
def test_rows_of_a_prompt_have_the_bits_of_single_rows(rows, dim, v_dim, rotary, more):
    from flyweight_amd.kernels import ops
    print(rows, dim, v_dim, rotary, more, flush=True)
    for got, want in zip(run(ops, rows, dim, v_dim, rotary, rows, **more), run(ops, rows, dim, v_dim, rotary, 63, **more)):
        assert torch.equal(got, want)
