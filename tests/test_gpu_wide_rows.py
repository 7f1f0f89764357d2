"""The mixes of neighbouring tokens and the experts' sum of a prompt's rows, several rows or channels to a thread, give the bits of the plain forms, which the same
operands take where they lie 4 bytes off."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def off(t):
    """The same numbers 4 bytes behind a 16-byte place."""
    place = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape)
    return place.copy_(t)


@pytest.mark.parametrize("hidden,mixes", [(4, 1), (260, 5), (1024, 6), (2052, 3), (5000, 2)])
@pytest.mark.parametrize("lengths", [[129], [1, 1, 140, 2, 3], [200, 1, 54], [1023], [1, 700, 324], [1030, 1]])
@pytest.mark.parametrize("dtype,normed,one", [(torch.bfloat16, True, True), (torch.float32, True, False), (torch.bfloat16, False, False)])
def test_mixes_of_neighbouring_tokens(hidden, mixes, lengths, dtype, normed, one):
    from flyweight_amd.kernels import ops
    print(hidden, mixes, lengths, dtype, normed, flush=True)
    rows = sum(lengths)
    g = torch.Generator().manual_seed(rows + hidden)
    x, mu, weight, last = (torch.randn(*shape, generator=g).to(DEV) for shape in ((rows, hidden), (mixes, hidden), (hidden,), (len(lengths) + 2, hidden)))
    ints = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)     # noqa: E731
    seg, begin = ints(np.repeat(np.arange(len(lengths)), lengths)), ints(np.concatenate([[0], np.cumsum(lengths)]))
    slots = ints(np.arange(len(lengths))[::-1] + 1)
    last_off = last.clone()
    call = lambda x, last: ops.token_shift_mix(x, weight if normed else None, 1e-5, one, mu, last, seg, begin, slots, len(lengths), dtype)     # noqa: E731
    want = call(off(x), last_off)
    assert torch.equal(call(x, last), want) and torch.equal(last, last_off)


@pytest.mark.parametrize("rows,hidden,top,shared", [(64, 4, 1, False), (65, 2048, 4, False), (300, 1028, 6, True), (77, 2052, 3, True), (64, 66000, 2, False)])
def test_sum_of_a_rows_experts(rows, hidden, top, shared):
    from flyweight_amd.kernels import ops
    print(rows, hidden, top, shared, flush=True)
    g = torch.Generator().manual_seed(rows)
    x, y, b = (torch.randn(n, hidden, generator=g).to(DEV) for n in (rows, rows * top, rows))
    weight, gate = torch.rand(rows, top, generator=g).to(DEV), torch.randn(rows, 1, generator=g).to(DEV)
    place = torch.randperm(rows * top, generator=g).to(torch.int32).view(rows, top).to(DEV)
    more = {"shared": b, "gate": gate} if shared else {}
    want = ops.moe_combine_(off(x), y, weight, place, **more)
    assert torch.equal(ops.moe_combine_(x.clone(), y, weight, place, **more), want)


@pytest.mark.parametrize("table_dtype,places_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, None), (torch.float32, None)])
@pytest.mark.parametrize("rows,hidden", [(64, 4), (65, 1028), (300, 2048), (64, 66000)])
def test_rows_of_a_table(rows, hidden, table_dtype, places_dtype):
    from flyweight_amd.kernels import ops
    print(rows, hidden, table_dtype, places_dtype, flush=True)
    g = torch.Generator().manual_seed(rows)
    table, places = torch.randn(50, hidden, generator=g).to(DEV, table_dtype), torch.randn(400, hidden, generator=g).to(DEV, places_dtype or table_dtype)
    ids, at = (torch.randint(0, n, (rows,), generator=g).to(DEV, torch.int32) for n in (50, 400))
    more = {} if places_dtype is None else {"places_table": places, "places": at}
    want = ops.embed_rows(off(table), ids, scale=1.7, **more)
    assert torch.equal(ops.embed_rows(table, ids, scale=1.7, **more), want)
