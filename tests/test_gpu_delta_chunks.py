"""The gated delta rule's prompts in chunks of sixteen tokens, from the projections to the read-outs, against the plain functions of
tests/plain_koketar.py in float64."""

import numpy as np
import pytest
import torch

import plain_koketar as plain
from test_gpu_koketar_kernels import dev, ints

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,slots_of", [([1, 2, 15, 16, 17, 33, 48], [6, 0, 5, 1, 4, 2, 3]), ([70], [2]), ([5, 100, 1, 1, 64], [1, 0, 4, 3, 2])])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,taps,per_head", [
    (3, 1, 20, 70, 4, False), (2, 2, 64, 64, 1, True), (4, 2, 8, 5, 2, False), (2, 1, 130, 129, 5, False), (2, 2, 128, 128, 4, True), (1, 1, 256, 16, 3, False),
    (1, 1, 200, 256, 17, False)])
def test_prompts_in_chunks(heads, kv_heads, dim, vdim, taps, per_head, lengths, slots_of):
    """Segments at the edges of a chunk beside each other, heads that end inside a tile, convolutions with and without a memory, one decay a
    head; channels that never forget, and some that forget everything at once (a decay that rounds to zero). The tolerance of the
    walk token by token."""
    from flyweight_amd.kernels import ops
    rng = np.random.default_rng(dim + vdim + len(lengths))
    rows, slots = sum(lengths), max(slots_of) + 1
    channels = 2 * kv_heads * dim + heads * vdim
    proj = rng.normal(size=(rows, channels + heads + 3)).astype(np.float32)
    a = rng.normal(size=(rows, heads if per_head else heads * dim)).astype(np.float32) * 2
    weights = rng.normal(size=(channels, taps)).astype(np.float32)
    A_log, dt_bias = rng.uniform(-2, 1, heads).astype(np.float32), rng.normal(size=a.shape[1]).astype(np.float32)
    a[::7, 0] = 300.0                                           # forgets at once
    a[:, -1] = -60.0                                            # never does
    memory = rng.normal(size=(slots, channels, taps - 1)).astype(np.float32)
    start = rng.normal(size=(slots, heads, dim, vdim)).astype(np.float32)
    state, conv_state = dev(start.transpose(0, 1, 3, 2)), dev(memory)
    seg_row0 = np.concatenate([[0], np.cumsum(lengths)])
    wide = dev(np.concatenate([a, rng.normal(size=(rows, 5))], axis=1))      # the decays' arguments as a view of wider rows
    out = ops.delta_chunks(dev(proj), channels, wide[:, :a.shape[1]], dev(weights), conv_state, dev(A_log), dev(dt_bias), state,
                           ints(seg_row0), ints(slots_of), len(lengths), heads, kv_heads, dim, vdim, decay_per_head=per_head)
    out, after, kept = out.cpu().numpy().reshape(rows, heads, vdim), state.cpu().numpy().transpose(0, 1, 3, 2), conv_state.cpu().numpy()
    proj, a, weights, A_log, dt_bias = (x.astype(np.float64) for x in (proj, a, weights, A_log, dt_bias))
    for seg, (length, slot) in enumerate(zip(lengths, slots_of)):
        r0, before = seg_row0[seg], memory[slot].T.astype(np.float64)
        x = proj[r0:r0 + length, :channels]
        y = plain.silu(plain.causal_conv(x, weights, before))
        nq = kv_heads * dim
        q = plain.unit(y[:, :nq].reshape(length, kv_heads, dim)) * dim ** -0.5
        k = plain.unit(y[:, nq:2 * nq].reshape(length, kv_heads, dim))
        v = y[:, 2 * nq:].reshape(length, heads, vdim)
        beta = plain.sigmoid(proj[r0:r0 + length, channels:channels + heads])
        raw = (a[r0:r0 + length] + dt_bias).reshape(length, heads, -1)
        g = np.broadcast_to(np.exp(-np.exp(A_log)[None, :, None] * plain.softplus(raw)), (length, heads, dim))
        if taps > 1:
            np.testing.assert_allclose(kept[slot], np.concatenate([before, x])[-(taps - 1):].T, atol=1e-6)
        for head in range(heads):
            S, group = start[slot, head].astype(np.float64), head // (heads // kv_heads)
            for t in range(length):
                S, o = plain.delta_rule_step(S, q[t, group], k[t, group], v[t, head], beta[t, head], g[t, head])
                np.testing.assert_allclose(out[r0 + t, head], o, rtol=0, atol=2e-5 * max(1.0, np.abs(o).max()))
            np.testing.assert_allclose(after[slot, head], S, rtol=0, atol=2e-5 * max(1.0, np.abs(S).max()))


def test_inputs_far_below_zero_pass_nothing():
    """silu(x) goes to -0 as x falls: a convolution's sum of -1e38 writes nothing and turns no key, one of -90 as good as nothing."""
    from flyweight_amd.kernels import ops
    rng = np.random.default_rng(5)
    rows, dim, vdim = 40, 64, 16
    channels = 2 * dim + vdim
    proj = rng.normal(size=(rows, channels + 1)).astype(np.float32)
    values = np.float32([-3e38, -1e38, -1e30, -1e6, -200, -104, -90, -89, -88.7, -88, -87.5, -87, -80, -60, -20, 1])
    proj[:, 2 * dim:channels] = values
    proj[::3, 5], proj[::4, dim + 7] = -1e38, -3e38
    a, A_log, dt_bias = rng.normal(size=(rows, dim)).astype(np.float32), np.zeros(1, np.float32), np.zeros(dim, np.float32)
    state = dev(np.zeros((1, 1, vdim, dim)))
    out = ops.delta_chunks(dev(proj), channels, dev(a), dev(np.ones((channels, 1))), dev(np.zeros((1, channels, 0))), dev(A_log), dev(dt_bias), state,
                           ints([0, rows]), ints([0]), 1, 1, 1, dim, vdim).cpu().numpy()
    x = proj.astype(np.float64)
    with np.errstate(over="ignore"):
        y = x[:, :channels] / (1.0 + np.exp(-x[:, :channels]))
    q, k = plain.unit(y[:, :dim]) * dim ** -0.5, plain.unit(y[:, dim:2 * dim])
    S = np.zeros((dim, vdim))
    for t in range(rows):
        S, o = plain.delta_rule_step(S, q[t], k[t], y[t, 2 * dim:], plain.sigmoid(x[t, channels]), np.exp(-plain.softplus(a[t].astype(np.float64))))
        # (a sum of fifty factors is 2^-18 off; below 1e-34 a float loses bits, and below 1e-38 all of them)
        assert (np.abs(out[t] - o) <= 2e-5 * np.abs(y[0, 2 * dim:]) + 1e-34).all()
