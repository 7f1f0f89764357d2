"""Which form of a kernel a call takes, where that is decided on the host: each rule at the sizes where both sides were measured
(no GPU)."""

import numpy as np
import pytest
import torch


def _row0(lengths):
    return [0] + np.cumsum(lengths).tolist()


def _delta_rule(heads, dim, vdim, dtype=torch.bfloat16):
    from flyweight_amd.config.spec import PartSpec
    from flyweight_amd.parts.deltarule import GatedDeltaRule
    part = GatedDeltaRule(PartSpec("gated_delta_rule", {
        "hidden_size": 64, "num_heads": heads, "num_kv_heads": heads, "head_dim": dim, "v_head_dim": vdim, "conv_taps": 4,
        "decay_rank": 8, "gate_rank": 8, "norm_eps": 1e-5}))
    part.dtype = dtype
    return part


@pytest.mark.parametrize("heads,dim,vdim,lengths,spread", [
    (16, 128, 128, [694], True), (16, 128, 128, [694, 694], False), (16, 128, 128, [300] * 4, False), (32, 128, 128, [694], False),
    (4, 128, 128, [300] * 4, True), (4, 128, 128, [300] * 8, False), (8, 256, 256, [2048], True), (8, 256, 256, [694] * 2, False),
    (2, 96, 96, [64] * 8, True), (2, 96, 96, [64] * 24, False),
    (16, 128, 128, [1] * 6 + [1500], False), (16, 128, 128, [1, 694], False), (2, 128, 128, [1] * 6 + [1500], True),
    (16, 64, 64, [694], False)])
def test_delta_rule_spreads_its_columns_while_every_workgroup_has_a_compute_unit(heads, dim, vdim, lengths, spread):
    assert _delta_rule(heads, dim, vdim).spread(_row0(lengths)) == spread
    assert not _delta_rule(heads, dim, vdim, torch.float32).spread(_row0(lengths))


@pytest.mark.parametrize("lengths,chunked", [
    ([95], False), ([96], True), ([64] * 16, False), ([96] * 16, True), ([1111], True), ([1] * 24 + [128], False), ([1] * 24 + [160], True),
    ([1] * 60 + [200], False), ([1] * 60 + [256], True), ([1] * 60 + [500], True), ([1] * 8, False), ([15, 300], True)])
def test_delta_rule_walks_prompts_in_chunks_where_those_are_faster(lengths, chunked):
    assert _delta_rule(16, 128, 128).chunked(_row0(lengths)) == chunked
    assert not _delta_rule(16, 128, 128, torch.float32).chunked(_row0(lengths))


@pytest.mark.parametrize("heads,dim,vdim,lengths,chunked", [
    (48, 128, 128, [1] * 24 + [200], False), (48, 128, 128, [1] * 60 + [400], False), (48, 128, 128, [1] * 60 + [777], True),
    (16, 256, 256, [96], True), (16, 256, 256, [1] * 24 + [256], False), (16, 256, 256, [1] * 24 + [400], True), (16, 256, 256, [1] * 60 + [777], False),
    (16, 256, 256, [17] * 40 + [192], False), (16, 64, 256, [1] * 60 + [200], False), (1, 256, 256, [1] * 60 + [160], True),
    (32, 64, 64, [1] * 60 + [256], False), (2, 16, 16, [1] * 60 + [128], True), (256, 1, 1, [1] * 4 + [200], False)])
def test_many_or_large_heads_beside_short_segments_keep_the_walk_token_by_token(heads, dim, vdim, lengths, chunked):
    assert _delta_rule(heads, dim, vdim).chunked(_row0(lengths)) == chunked


@pytest.mark.parametrize("heads,dim,lengths,cuts", [
    (32, 64, [2048], True), (32, 64, [512] * 4, False), (32, 64, [129] * 2, False), (32, 64, [2048] * 2, True), (32, 64, [128], False),
    (32, 16, [129] * 4, False), (32, 16, [512] * 4, True), (32, 32, [129] * 4, False), (32, 32, [256] * 4, True),
    (16, 128, [129], False), (16, 128, [256] * 2, True), (16, 128, [256] * 4, False),
    (16, 256, [256], False), (16, 256, [1024], True), (4, 256, [129] * 2, False), (4, 256, [256] * 2, True), (4, 256, [256] * 4, False),
    (32, 64, [1] * 24, False), (32, 64, [1] * 24 + [300], True), (8, 64, [128, 200], False)])   # short segments beside a long one
def test_wkv_cuts_long_segments_where_the_chunks_are_faster(heads, dim, lengths, cuts):
    from flyweight_amd.config.spec import PartSpec
    from flyweight_amd.parts.wkv import Wkv
    part = Wkv(PartSpec("wkv", {"hidden_size": 64, "num_heads": heads, "head_dim": dim, "decay_rank": 8, "norm_eps": 1e-5}))
    assert part.cuts(_row0(lengths)) == cuts


@pytest.mark.parametrize("rows,behind,heads,groups,widest,halves", [
    (2048, 2048, 32, 8, 64, True), (2048, 30720, 16, 8, 64, True), (1500, 3072, 32, 8, 64, False), (1700, 2048, 32, 8, 64, True),
    (1500, 3072, 16, 8, 64, True), (777, 0, 32, 8, 64, False), (777, 2048, 32, 8, 64, True), (777, 2048, 16, 8, 64, False),
    (777, 30720, 16, 8, 64, True), (64, 3000, 32, 8, 64, False), (6000, 4096, 32, 8, 64, True), (3500, 4096, 32, 8, 64, False),
    (2048, 8192, 24, 8, 64, False), (2048, 8192, 32, 8, 32, False), (2048, 8192, 32, 8, 48, True), (2048, 8192, 32, 8, 128, False),
    (2048, 8192, 8, 8, 64, False)])
def test_prompt_attention_shares_pages_between_halves_where_its_rounds_are_full(rows, behind, heads, groups, widest, halves):
    from flyweight_amd.kernels import ops
    assert ops.prompt_halves(-(-rows // 64), heads, groups, widest, rows + behind) == halves


@pytest.mark.parametrize("rows,behind,heads,groups,dim,v_dim,window,form", [
    (37, 0, 32, 8, 64, 64, 0, None), (576, 0, 32, 8, 64, 64, 0, None), (777, 0, 32, 8, 64, 64, 0, False), (1111, 0, 32, 8, 64, 64, 0, True),
    (1300, 2048, 32, 8, 64, 64, 0, False), (2048, 0, 32, 8, 64, 64, 0, True), (2048, 2048, 32, 8, 64, 64, 0, False), (3000, 0, 32, 8, 64, 64, 0, False),
    (100, 2000, 32, 8, 64, 64, 0, True), (4096, 0, 16, 8, 64, 64, 0, True), (2048, 30720, 16, 8, 64, 64, 0, True), (2048, 2048, 24, 8, 64, 64, 0, None),
    (2048, 2048, 32, 8, 64, 48, 0, None), (2048, 2048, 32, 8, 80, 80, 0, None), (37, 0, 16, 4, 128, 128, 1024, False), (300, 0, 16, 4, 128, 128, 1024, False),
    (1111, 0, 16, 4, 128, 128, 1024, True), (2048, 0, 16, 4, 128, 128, 1024, True), (3000, 0, 16, 4, 128, 128, 1024, False),
    (4096, 0, 16, 4, 128, 128, 1024, False), (2048, 4096, 16, 4, 128, 128, 0, True), (2048, 4096, 8, 8, 128, 128, 0, None)])
def test_prompt_attention_takes_heads_two_by_two_where_that_is_faster(rows, behind, heads, groups, dim, v_dim, window, form):
    from flyweight_amd.kernels import ops
    context = rows + behind
    assert ops.prompt_pairs(-(-rows // 64), heads, groups, dim, v_dim, min(window or context, context), context) is form


def test_decode_rows_do_not_choose_the_form_of_a_prompt_beside_them(monkeypatch):
    """A new prompt of 777 rows beside a request that decodes behind 20,000 keys takes the form that it takes alone."""
    from types import SimpleNamespace

    from flyweight_amd.kernels import ops
    taken = []
    monkeypatch.setattr(ops, "attention_prefill", lambda *a, halves, **k: taken.append(halves))
    monkeypatch.setattr(ops, "attention_decode", lambda *a, **k: None)
    for decoding, behind, halves in (([], 0, False), ([20000], 0, False), ([20000], 4000, True), ([], 4000, True), ([30], 4000, True)):
        single = len(decoding)
        tiles = torch.zeros(single + 13, dtype=torch.int32)
        rows = single + 777
        ctx = SimpleNamespace(all_decode=False, decode_prefix=single, max_context=max(decoding + [behind + 777]),
                              new_lengths=decoding + [behind + 777], row_seg=None, row_pos=None, seg_row0=None)
        ops.attention(torch.zeros(rows, 32 * 64, dtype=torch.bfloat16), 32, 8, 64, None, None, None, ctx, 0.125, 0, tiles, tiles)
        assert taken.pop() == halves


@pytest.mark.parametrize("mode,M,N,K,splits", [
    (1, 16, 2048, 8192, True), (1, 9, 512, 8192, True), (1, 8, 512, 8192, False),
    (1, 11, 2048, 8192, False), (1, 12, 2048, 8192, True), (1, 9, 2048, 10752, True), (1, 8, 4096, 12288, False), (1, 11, 4096, 12288, True),
    (1, 16, 2048, 4608, False), (1, 16, 4096, 8192, False), (1, 16, 4096, 12288, True),
    (1, 32, 2048, 12288, True), (1, 32, 2048, 8192, False), (1, 48, 2048, 12288, False), (1, 64, 2048, 12288, True),
    (1, 32, 2560, 6144, True), (1, 32, 3072, 8192, False), (1, 16, 3072, 8192, False), (1, 64, 1024, 12288, False), (1, 32, 512, 16384, False),
    (0, 17, 20480, 2048, True), (0, 8, 65536, 2048, True), (0, 64, 65536, 2048, True), (0, 17, 16384, 1024, True), (0, 64, 16384, 1024, False),
    (0, 32, 8192, 2048, True), (0, 32, 10240, 2048, False), (0, 33, 8192, 2048, False), (0, 17, 4096, 1024, False), (0, 4, 6144, 2048, False),
    (2, 32, 4608, 1024, True), (2, 64, 4608, 2048, False), (2, 32, 4096, 1024, False), (2, 17, 10752, 2048, True), (2, 17, 10752, 2056, False)])
def test_products_of_few_rows_split_k_over_workgroups_where_that_is_faster(mode, M, N, K, splits):
    from flyweight_amd.kernels import ops
    assert ops.medium_splits_k(mode, M, N, K) == splits


@pytest.mark.parametrize("M,N,K,takes", [(1, 16, 256, True), (16, 2048, 768, True), (8, 2048, 1024, True), (16, 2048, 1024, False),
                                         (1, 4096, 2048, False), (4, 12288, 512, True), (1, 12288, 640, False), (1, 65536, 64, False)])
def test_products_of_up_to_sixteen_rows_over_a_short_k_take_the_skinny_kernel(M, N, K, takes):
    from flyweight_amd.kernels import ops
    assert ops.skinny_takes(M, N, K) == takes


@pytest.mark.parametrize("mode,M,N,K,fits", [
    (1, 512, 2048, 8192, True), (1, 128, 2560, 10752, True), (0, 192, 6144, 2048, False), (0, 128, 6144, 2048, True), (2, 128, 8192, 2048, False),
    (0, 128, 2560, 7168, True), (0, 128, 2560, 8192, False), (0, 96, 3072, 10752, True), (0, 160, 2560, 10752, True), (0, 256, 2048, 8192, True),
    (0, 256, 2048, 10752, False), (0, 256, 4096, 10752, True), (2, 192, 1536, 5120, True), (2, 192, 1536, 6144, False), (2, 320, 1536, 10752, True),
    (2, 128, 4096, 8192, True), (2, 128, 4096, 10752, False), (2, 96, 1536, 10752, True), (2, 128, 1536, 8192, False), (1, 1025, 64, 64, False)])
def test_products_beyond_64_rows_are_dealt_to_waves_where_that_is_faster(mode, M, N, K, fits):
    from flyweight_amd.kernels import ops
    assert ops.rows_fit(mode, M, N, K) == fits


@pytest.mark.parametrize("mode,M,N,K,plan", [
    (0, 1111, 2048, 8192, ("bigsplit", 0)), (0, 1111, 2048, 2048, ("big", 0)), (0, 640, 2048, 2048, ("deep", 64)), (0, 1111, 1024, 4608, ("deep", 64)),
    (0, 1300, 3072, 2048, ("big", 0)), (0, 801, 3072, 1024, ("big", 0)), (0, 2048, 6144, 2048, ("big", 0)), (0, 512, 6144, 1024, ("big", 0)),
    (0, 320, 6144, 2048, ("big", 0)), (0, 320, 1024, 8192, ("split", 0)), (0, 128, 3072, 8192, ("split", 0)), (0, 300, 2500, 520, ("tiles", 0)),
    (0, 100, 8192, 32, ("tiles", 0)), (2, 801, 1536, 2048, ("tiles", 0)), (2, 1111, 4608, 2048, ("big", 0)), (2, 640, 1536, 2048, ("split", 0)),
    (0, 1111, 64, 4096, ("split", 0)), (0, 2048, 64, 1024, ("deep", 64)), (2, 300, 64, 2048, ("split", 0)),
    (2, 2048, 8192, 2048, ("big", 0)), (2, 128, 8192, 1024, ("tiles", 0)), (2, 2048, 2048, 2048, ("big", 0)),
    (1, 2048, 2048, 8192, ("bigsplit", 0)), (1, 2048, 1024, 1024, ("deep", 64)), (1, 512, 2048, 2048, ("deep", 64)), (1, 256, 2048, 8192, ("split", 0)),
    (1, 2048, 8192, 2048, ("big", 0)),
    # a second round of large tiles that is little full
    (2, 2048, 4608, 1024, ("big", 0)), (2, 2048, 5120, 1024, ("big", 0)), (2, 2048, 4608, 2048, ("big", 0)), (2, 2048, 4096, 1024, ("big", 0)),
    (2, 2048, 7168, 1024, ("big", 0)), (2, 2048, 6144, 2048, ("big", 0)), (2, 1005, 11344, 192, ("big", 0)), (1, 2048, 2048, 2048, ("big", 0)),
    # many rounds of tiles, a short K, odd widths, few rows of tiles over a long K
    (1, 6200, 2048, 7168, ("big", 0)), (1, 8192, 2048, 1024, ("big", 0)), (1, 2690, 1536, 1024, ("big", 0)), (1, 1700, 2048, 7168, ("bigsplit", 0)), (1, 2048, 2048, 4160, ("deep", 128)),
    (2, 13184, 3496, 352, ("big", 0)), (2, 5964, 4032, 128, ("big", 0)), (2, 2304, 1281, 128, ("tiles", 0)), (2, 512, 4480, 2560, ("tiles", 0)),
    (0, 100, 65536, 2048, ("tiles", 0)), (0, 512, 65536, 2048, ("big", 0)), (0, 128, 4480, 2816, ("split", 0)), (1, 256, 2112, 7872, ("bigsplit", 0)),
    # what the GPU tests of these tiles compute
    (1, 2048, 2048, 4096, ("big", 0)), (1, 1800, 1990, 4160, ("deep", 128)), (1, 2048, 1024, 2048, ("deep", 64)), (1, 1152, 2048, 2048, ("big", 0)),
    (1, 576, 2048, 1024, ("deep", 64)), (1, 1100, 1024, 2048, ("deep", 64)), (1, 1664, 2048, 4096, ("deep", 128)), (0, 256, 6144, 2048, ("deep", 64)),
    (0, 1100, 2048, 4096, ("bigsplit", 0)), (0, 130, 6144, 2048, ("deep", 64)), (1, 320, 2048, 2048, ("deep", 64)), (0, 300, 3072, 1024, ("deep", 64)),
    (0, 600, 6144, 2048, ("big", 0)), (0, 700, 6144, 2048, ("big", 0)), (0, 500, 6100, 1984, ("big", 0)), (0, 256, 1024, 2048, ("deep", 64)),
    (0, 1300, 2944, 7680, ("deep", 128))])
def test_tiled_products_take_the_tiles_that_were_the_fastest(mode, M, N, K, plan):
    from flyweight_amd.kernels import ops
    assert ops.tiled_plan(mode, M, N, K) == plan


def _at_an_odd_place(t):
    """The same values from an address that is no multiple of 16 bytes."""
    held = torch.empty(t.numel() + 4, dtype=t.dtype)
    first = next(i for i in range(4) if (held.data_ptr() + i * t.element_size()) % 16)
    odd = held[first:first + t.numel()].view(t.shape)
    return odd.copy_(t)


def _even(*shape):
    t = torch.randn(*shape)
    return t if t.data_ptr() % 16 == 0 else pytest.skip("the host's tensors do not start at 16 bytes")


@pytest.mark.parametrize("odd", ["none", "rows", "weight", "norm"])
def test_few_float32_rows_take_their_norm_in_front_only_where_every_operand_starts_at_16_bytes(odd):
    """The kernel that takes the norm reads x, W and the norm's weight 16 bytes at a time; anything else goes through the norm and the product apart."""
    from flyweight_amd.config.spec import PartSpec
    from flyweight_amd.parts.linear import Linear
    from flyweight_amd.parts.norm import LazyNorm, RMSNorm
    x, w, weight = (_at_an_odd_place(t) if odd == name else t for name, t in (("rows", _even(1, 1024)), ("weight", _even(64, 1024)), ("norm", _even(1024))))
    norm = RMSNorm(PartSpec("rmsnorm", {"size": 1024, "eps": 1e-5}))
    norm.bind({norm.tensor_name: weight}, torch.float32, torch.device("cpu"))
    linear = Linear(w)
    for gated, features in ((False, 64), (True, 32)):
        assert linear._normed(LazyNorm(norm, x, None), features, gated) == (odd == "none")
    assert not linear._normed(LazyNorm(norm, x.view(1, 1, 1024), None), 64, False)       # (rows of another shape, which the norm by itself takes)


@pytest.mark.parametrize("heads,kv_heads,dim,v_dim,rows,fused", [
    (32, 8, 64, 64, 64, True), (32, 8, 64, 64, 65, False), (16, 4, 128, 128, 64, True), (16, 16, 80, 112, 64, True), (16, 4, 144, 144, 32, True),
    (16, 4, 144, 144, 33, False), (8, 8, 256, 256, 32, True), (8, 8, 256, 256, 48, False), (8, 4, 64, 192, 33, False), (8, 4, 192, 64, 33, False),
    (16, 1, 128, 128, 16, True), (16, 1, 128, 128, 17, False), (16, 1, 256, 256, 16, True), (16, 1, 256, 256, 17, False)])
def test_decode_steps_form_queries_inside_the_attention_kernel_where_that_is_faster(monkeypatch, heads, kv_heads, dim, v_dim, rows, fused):
    from types import SimpleNamespace
    from flyweight_amd.config.spec import PartSpec
    from flyweight_amd.kernels import ops
    from flyweight_amd.parts.attention import GQAttention
    took = []
    monkeypatch.setattr(ops, "attention_decode_fused", lambda *a, **k: took.append(True))
    monkeypatch.setattr(ops, "qk_norm_rope_kv_write", lambda *a, **k: None)
    monkeypatch.setattr(ops, "attention", lambda *a, **k: took.append(False))
    part = GQAttention(PartSpec("gqa_attention", {
        "hidden_size": 64, "num_heads": heads, "num_kv_heads": kv_heads, "head_dim": dim, "v_head_dim": v_dim,
        "position": PartSpec("rotary_neox", {"head_dim": dim, "theta": 1e4})}))
    part.dtype, part.sinks, part.slopes, part.conv, part.q_norm_weight, part.k_norm_weight = torch.bfloat16, None, None, None, None, None
    part.qkv = SimpleNamespace(forward=lambda h, out_dtype: torch.empty(0, dtype=out_dtype))
    ctx = SimpleNamespace(all_decode=True, num_rows=rows, max_context=64, row_seg=None, row_pos=None,
                          position_tables=lambda p: (None, None), step_arrays=lambda p: {})
    part.attend(None, ctx, SimpleNamespace(writes=True, k_pages=None, v_pages=None, block_table=None))
    assert took == [fused]


@pytest.mark.parametrize("positions,work", [
    ([1999] * 9, -8), ([1999] * 9 + [0] * 7, -8), ([2000, 2040, 2047, 2048], -9), ([700, 2900, 1500], 21), ([700, 2900, 1500, 0], 21), ([300], -2),
    ([0] * 4, 0), ([2560, 10], 12), ([2999] * 63 + [40], -12)])
def test_decode_steps_tell_rows_of_one_length_from_rows_of_many(positions, work):
    """Whatever rows fill a step up."""
    from types import SimpleNamespace
    from flyweight_amd.parts.attention import QueryTileArrays
    rows = np.asarray(positions, dtype=np.int32)
    assert QueryTileArrays()._decode_work(SimpleNamespace(num_rows=len(rows), all_decode=True, host_row_pos=rows)) == work
    beside = SimpleNamespace(num_rows=len(rows) + 50, all_decode=False, decode_prefix=len(rows), host_row_pos=np.concatenate([rows, np.arange(50, dtype=np.int32)]))
    assert QueryTileArrays()._decode_work(beside) == work
