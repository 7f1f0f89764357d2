"""The native module of launches: bit for bit what the general paths give, over the forms that it accepts; what it does not take goes to them and is served or refused as
they do."""

import ctypes

import pytest
import torch

DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    assert module.native_launches()
    return module


def draw(*shape, dtype=BF, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def both(ops, monkeypatch, call):
    """What the call gives natively and on the general path."""
    taken = []
    real = ops._native

    class Counted:
        def __getattr__(self, name):
            def function(*args):
                made = getattr(real, name)(*args)
                taken.append(made is not NotImplemented)
                return made
            return function

    monkeypatch.setattr(ops, "_native", Counted())
    native = call()
    monkeypatch.setattr(ops, "_native", None)
    general = call()
    monkeypatch.setattr(ops, "_native", real)
    assert taken and all(taken)
    return native, general


def same(a, b):
    if isinstance(a, tuple):
        return len(a) == len(b) and all(same(x, y) for x, y in zip(a, b))
    return a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tiled,plans", [         # by mode: "rows" waves split K, "split" K over workgroups, "large" a large tile, "cut" K cut on it, None the general path
    (1, 2048, 4096, False, "rows rows rows"), (1, 2048, 4096, True, "rows rows rows"), (16, 2048, 8192, False, "split split rows"), (16, 256, 8192, True, "split split rows"),
    (17, 96, 520, False, "rows rows rows"), (37, 3072, 1024, False, "rows rows rows"), (37, 3072, 1024, True, "rows rows rows"), (64, 515, 168, False, "rows rows rows"),
    (64, 515, 160, True, "rows rows rows"), (65, 1000, 1024, True, "rows rows rows"), (130, 2048, 4608, True, "rows rows rows"), (300, 1536, 512, True, "large large large"),
    (801, 2048, 2048, True, "large large large"), (801, 2048, 7168, True, "cut cut large"), (256, 2048, 8192, True, "cut cut rows"), (65, 1000, 1024, False, "None None None")])
def test_products(ops, monkeypatch, M, N, K, tiled, plans):
    a, w, bias, old = draw(M, K), draw(2 * N, K, seed=1), draw(N, dtype=F32, seed=2), draw(M, N, dtype=F32, seed=3)
    own = w[:N].contiguous()
    t, t2 = (ops.tile_weights(own), ops.tile_weights(w)) if tiled else (None, None)
    assert tiled == (t is not None)

    def named(mode):
        plan = ops._native_plan(False, tiled, mode, M, N, K)
        return "None" if plan is None else ("large" if plan[4] == 1 else "cut") if plan[0] else "split" if plan[1] else "rows"
    found = [named(mode) for mode in range(3)]
    assert " ".join(found) == plans
    if plans == "None None None":
        assert ops._native_product(False, a, own, t, None, None, 0, F32) is NotImplemented
        return
    for how in ({}, {"out_dtype": F32}, {"bias": bias, "out_dtype": F32}, {"gelu": True}):
        assert same(*both(ops, monkeypatch, lambda: ops.gemm(a, own, w_tiled=t, **how)))
    assert same(*both(ops, monkeypatch, lambda: ops.gemm(a, own, bias, accumulate_into=old.clone(), w_tiled=t)))
    for gelu in (False, True):
        assert same(*both(ops, monkeypatch, lambda: ops.gemm_swiglu(a, w, w_tiled=t2, gelu=gelu)))
    if M <= 64:
        squares = draw(5, 16 if M <= 16 else 64, dtype=F32, seed=4).abs()
        weight = draw(N, dtype=F32, seed=5)
        for prepared in ({}, {"squares": squares, "eps": 1e-5}):
            assert same(*both(ops, monkeypatch, lambda: ops.gemm_medium(a, own, ops.EPILOGUE_STORE, bias=bias, out_dtype=F32, w_tiled=t, **prepared)))
            assert same(*both(ops, monkeypatch, lambda: ops.gemm_medium(a, own, ops.EPILOGUE_STORE, gelu=True, w_tiled=t, **prepared)))
            for glu in (None, ops.GEGLU, (7.0, 1.702, 1.0)):
                assert same(*both(ops, monkeypatch, lambda: ops.gemm_medium(a, w, ops.EPILOGUE_SWIGLU, glu=glu, w_tiled=t2, **prepared)))
        assert same(*both(ops, monkeypatch, lambda: ops.gemm_medium(a, own, ops.EPILOGUE_ACCUMULATE, bias=bias, accumulate_into=old.clone(), w_tiled=t)))
        for centered in (False, True):
            def add():
                into = old.clone()
                return (*ops.gemm_medium(a, own, ops.EPILOGUE_ACCUMULATE, accumulate_into=into, next_norm_weight=weight, next_one_centered=centered, w_tiled=t), into)
            (x, sums, into), (x2, sums2, into2) = both(ops, monkeypatch, add)
            assert same(x, x2) and same(into, into2) and same(sums[:, :M], sums2[:, :M])


def ints(*v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@pytest.mark.gpu
def test_norms(ops, monkeypatch):
    x, weight = draw(40, 512, dtype=F32), draw(512, dtype=F32, seed=1)
    for dtype in (BF, F32):
        for rows in (None, ints(3, 39, 3), ints()):
            for rank in (x, x.view(4, 10, 512), x[0]) if rows is None else (x,):
                assert same(*both(ops, monkeypatch, lambda: ops.rmsnorm_rows(rank, weight, 1e-5, dtype, row_index=rows, one_centered=rows is not None)))


@pytest.mark.gpu
@pytest.mark.parametrize("taken,out_dtype", [(F32, BF), (F32, F32), (BF, BF)])
@pytest.mark.parametrize("kernel,with_bias", [(3, True), (4, False), (2, True)])
def test_short_convolutions(ops, monkeypatch, taken, out_dtype, kernel, with_bias):
    bcx, taps, held, bias = draw(40, 3 * 512, dtype=taken), draw(512, kernel, dtype=F32), draw(4, 512, kernel - 1, dtype=F32), draw(512, dtype=F32, seed=1)
    seg, row0, slot = ints(*([0] * 33 + [1] * 7)), ints(0, 33, 40), ints(2, 0)

    def conv():
        own = held.clone()
        return ops.shortconv(bcx, taps, bias if with_bias else None, own, seg, row0, slot, 2, out_dtype=out_dtype), own
    assert same(*both(ops, monkeypatch, conv))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [40, 73])              # from 64 on: rows side by side
@pytest.mark.parametrize("taken,pages", [(F32, BF), (BF, BF), (F32, F32)])
@pytest.mark.parametrize("d,v_dim,rotary,interleaved,normed,scaled,queries", [
    (64, None, 64, False, True, False, False), (64, 128, 32, True, False, True, False), (128, None, 128, True, True, False, False), (128, 64, 64, False, True, True, False),
    (40, None, 16, False, True, False, False), (64, None, 0, False, True, False, False), (128, None, 128, False, True, True, True), (96, None, 96, True, False, False, True)])
def test_queries_keys_and_values(ops, monkeypatch, rows, taken, pages, d, v_dim, rotary, interleaved, normed, scaled, queries):
    heads, kv, first = 6, 2, rows - 7
    dv = v_dim or d
    qkv = draw(rows, heads * d if queries else (heads + kv) * d + kv * dv, dtype=taken)
    weight, scale = draw(d, dtype=F32, seed=2), draw(rows, dtype=F32, seed=5)
    cos, sin = (draw(rows, rotary // 2, dtype=F32, seed=n) if rotary else None for n in (3, 4))
    table, seg, pos = ints(0, 3, 1, 2).view(2, 2), ints(*([0] * first + [1] * 7)), ints(*range(first), *range(60, 67))

    def write():
        k_pages, v_pages = torch.zeros(4, kv, 64, d, dtype=pages, device=DEV), torch.zeros(4, kv, dv, 64, dtype=pages, device=DEV)
        return ops.qk_norm_rope_kv_write(qkv, heads, kv, d, *([weight, weight + 1.0] if normed else [None, None]), 1e-5, cos, sin, rotary, k_pages, v_pages, table,
                                         seg, pos, write_kv=not queries, v_dim=v_dim, interleaved=interleaved, q_only=queries, q_row_scale=scale if scaled else None), k_pages, v_pages
    assert same(*both(ops, monkeypatch, write))


@pytest.mark.gpu
@pytest.mark.parametrize("d,v_dim,how", [
    (64, None, {}), (64, None, {"window": 20}), (64, None, {"window": 20, "keep_first": 3}), (64, None, {"chunk": 32}), (64, None, {"softcap": 5.0, "keep_first": 2}),
    (64, None, {"halves": True}), (64, None, {"paired": True}), (64, None, {"halves": True, "paired": True, "window": 50}), (128, None, {"paired": True, "sinks": True}),
    (64, None, {"heads_together": 4}), (128, 64, {"sinks": True, "slopes": True}), (48, 32, {"slopes": True, "window": 100, "keep_first": 70}), (64, None, {"sinks": True})])
def test_attention_of_prompts(ops, monkeypatch, d, v_dim, how):
    heads, kv, rows = 8, 2, 210
    how, dv = dict(how), v_dim or d
    for name, seed in (("sinks", 6), ("slopes", 7)):
        if how.get(name):
            how[name] = draw(heads, dtype=F32, seed=seed).abs()
    q, k_pages, v_pages = draw(rows, heads * d), draw(6, kv, 64, d, seed=1), draw(6, kv, dv, 64, seed=2)
    tile_seg, tile_row0 = ops.query_tiles([0, 150, 210])
    arrays = ints(5, 0, 3, 1, 2, 4).view(2, 3), ints(*tile_seg), ints(*tile_row0), ints(0, 150, 210), ints(*range(20, 170), *range(60))
    assert same(*both(ops, monkeypatch, lambda: ops.attention_prefill(q, heads, kv, d, k_pages, v_pages, *arrays, d ** -0.5, v_dim=v_dim, **how)))


@pytest.mark.gpu
def test_what_it_does_not_take_is_served_or_refused_as_before(ops):
    a, w = draw(40, 256), draw(96, 256, seed=1)
    with pytest.raises(ops.KernelError, match="contiguous"):
        ops.gemm(a.t().contiguous().t(), w)
    with pytest.raises(ops.KernelError, match="gemm: a is"):
        ops.gemm(a[:, :128].contiguous(), w)
    with pytest.raises(ops.KernelError, match="destination"):
        ops.gemm(a, w, accumulate_into=torch.zeros(40, 95, device=DEV))
    with pytest.raises(ops.KernelError, match="sums of squares"):
        ops.gemm_medium(a, w, ops.EPILOGUE_STORE, squares=torch.zeros(2, 16, device=DEV))
    with pytest.raises(ops.KernelError, match="operand tiles"):
        ops.gemm_medium(a, w, ops.EPILOGUE_STORE, w_tiled=ops.tile_weights(w)[:-1].contiguous())
    for mode, M, N, K in ((0, 300, 1536, 512), (1, 200, 1024, 256), (2, 100, 512, 256)):         # on a large tile, which reads w, where the operand tiles could be read
        assert ops._native_plan(False, True, mode, M, N, K)[0] == 1 and ops.rows_fit(mode, M, N, K)
        x, own, into = draw(M, K), draw(2 * N if mode == 2 else N, K, seed=1), torch.zeros(M, N, device=DEV)
        for wrong in (ops.tile_weights(own)[:-1].contiguous(), ops.tile_weights(own).float()):
            with pytest.raises(ops.KernelError, match="operand tiles"):
                ops.gemm_swiglu(x, own, w_tiled=wrong) if mode == 2 else ops.gemm(x, own, accumulate_into=into if mode else None, w_tiled=wrong)
    with pytest.raises(ops.KernelError, match="row width"):
        ops.rmsnorm_rows(a.float(), torch.zeros(255, device=DEV), 1e-5, BF)
    odd = torch.empty(40 * 256 + 1, dtype=BF, device=DEV)[1:].view(40, 256).copy_(a)       # at no multiple of 16 bytes
    assert torch.allclose(ops.gemm(odd, w, out_dtype=F32), a.float() @ w.float().T, atol=1e-3)


def test_tensors_of_the_host_are_left_to_the_general_path(ops):
    a, w = torch.zeros(20, 64, dtype=BF), torch.zeros(32, 64, dtype=BF)
    assert ops._native_product(False, a, w, None, None, None, 0, BF) is NotImplemented
    with pytest.raises(ops.KernelError, match="GPU only"):
        ops.rmsnorm_rows(torch.zeros(2, 8), torch.zeros(8), 1e-5, BF)
    with pytest.raises(TypeError):
        ops._native.rmsnorm(a)


@pytest.mark.gpu
def test_other_threads_run_while_a_launch_waits(ops):
    """The module lets go of the interpreter's lock around the kernel library's calls, as ctypes does. In place of the entry points here stands
    PyGILState_Check, which says 1 (a refused call) to a thread that holds it."""
    held = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    real = {name: ctypes.cast(getattr(ops._lib, name), ctypes.c_void_p).value for name in ops._NATIVE_ENTRIES}
    x, weight, pages, cos = draw(40, 256, dtype=F32), draw(256, dtype=F32), torch.zeros(2, 1, 64, 64, dtype=BF, device=DEV), draw(40, 32, dtype=F32)
    seg, row0, pos, table = ints(*[0] * 40), ints(0, 40), ints(*range(40)), ints(0, 1).view(1, 2)
    native, stream = ops._native, ops._stream()
    products = [(few, M, N, K, t) for few, M, N, K, t in ((True, 2, 2048, 256, False), (False, 40, 96, 256, False), (True, 16, 256, 8192, True), (False, 300, 1536, 512, True),
                                                          (False, 801, 2048, 7168, True))]
    plans = [ops._native_plan(few, t, 0, M, N, K) for few, M, N, K, t in products]
    assert all(plans) and {plan[0] for plan in plans} == {0, 1} and {plan[1] for plan in plans if not plan[0]} == {False, True} and plans[-1][4] > 1
    operands = [(draw(M, K), w, ops.tile_weights(w) if t else None) for _, M, N, K, t in products for w in (draw(N, K),)]
    counters = ops._medium_counters(x.device, 1)
    calls = [lambda a=a, w=w, t=t, plan=plan: native.product(a, w, t, None, None, 0, ops.F32, False, None, False, None, 0.0, 0.0, 1.0, 0.0, plan, counters, stream)
             for (a, w, t), plan in zip(operands, plans)]
    calls += [lambda: native.rmsnorm(x, weight, None, True, 1e-5, False, stream),
              lambda: native.shortconv(draw(40, 768, dtype=F32), draw(256, 3, dtype=F32), None, draw(1, 256, 2, dtype=F32), seg, row0, ints(0), 1, True, stream),
              lambda: native.qk_norm(draw(40, 256, dtype=F32), 2, 1, 64, None, None, 1e-5, cos, cos, 64, pages, pages, table, seg, pos, True, 64, False, False, None, 64, stream),
              lambda: native.prefill(draw(40, 128), 2, 1, 64, pages, pages, table, ints(0), ints(0), row0, pos, 0.125, 0, 0, 64, 0, 0.0, 0, None, None, 0, 64, stream)]
    try:
        native.bind({name: at if name == "fw_last_error" else held for name, at in real.items()}, ops.KernelError, torch.OutOfMemoryError)
        for call in calls:
            assert isinstance(call(), torch.Tensor)
    finally:
        native.bind(real, ops.KernelError, torch.OutOfMemoryError)
