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
    (16, 128, 128, [1] * 24 + [694], True),     # single rows leave at once
    (16, 128, 128, [1] * 64 + [40], False), (16, 128, 128, [600, 694], False), (16, 128, 128, [50, 694], True),
    (16, 64, 64, [694], False)])
def test_delta_rule_spreads_its_columns_while_every_workgroup_has_a_compute_unit(heads, dim, vdim, lengths, spread):
    assert _delta_rule(heads, dim, vdim).spread(_row0(lengths)) == spread
    assert not _delta_rule(heads, dim, vdim, torch.float32).spread(_row0(lengths))
