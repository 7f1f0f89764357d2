"""The product of float32 operands on the float32 matrix instruction: edges of its tiles, of K's quarters and groups of 16,
its three epilogues, and that a row's result does not depend on the rows beside it."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from flyweight_amd.kernels import ops as module
    module.library()
    return module


def draw(*shape, seed=0):
    generator = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=generator)


def bound(a, w):
    """K rounded products and sums: at most (K + 1) * 2^-24 of the sum of the products' sizes."""
    return (a.shape[1] + 1) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


# one row and the last of a tile, one past each tile's edge; outputs that fill no tile; K below a quarter's group, of whole
# groups, with a piece of a group left in the last or in an earlier quarter, and one quarter empty
SHAPES = [(1, 16, 64), (1, 1024, 4608), (16, 33, 100), (17, 64, 4), (32, 65, 20), (33, 130, 132), (64, 96, 208), (65, 1000, 1024),
          (129, 48, 36), (301, 515, 76), (3, 9216, 12)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product_of_float32_operands(ops, M, N, K):
    a, w, bias = draw(M, K), draw(N, K, seed=1), draw(N, seed=2)
    limit, exact = bound(a, w), a.double() @ w.double().T
    A, W, B = a.to(DEV), w.to(DEV), bias.to(DEV)
    assert ((ops.gemm(A, W).cpu().double() - exact).abs() <= limit).all()
    with_bias = ops.gemm(A, W, B).cpu().double()
    assert ((with_bias - exact - bias.double()).abs() <= limit + 2.0 ** -23 * with_bias.abs()).all()
    residual = draw(M, N, seed=3)
    into = residual.to(DEV)
    ops.gemm(A, W, accumulate_into=into)
    total = exact + residual.double()
    assert ((into.cpu().double() - total).abs() <= limit + 2.0 ** -23 * total.abs()).all()
    rounded = ops.gemm(A, W, out_dtype=torch.bfloat16).cpu().double()
    assert ((rounded - exact).abs() <= limit + 2.0 ** -8 * exact.abs()).all()


@pytest.mark.parametrize("M,F,K", [(1, 16, 64), (5, 77, 100), (33, 130, 132), (301, 515, 76), (64, 4608, 1024)])
def test_gated_product_of_float32_operands(ops, M, F, K):
    a, w = draw(M, K) * K ** -0.5, draw(2 * F, K, seed=1)
    limit, sums = bound(a, w), a.double() @ w.double().T
    g, u = sums[:, :F], sums[:, F:]
    exact = torch.nn.functional.silu(g) * u
    # silu's slope is below 1.1; the unit's own roundings are a few units in the last place
    allowed = 1.1 * limit[:, :F] * u.abs() + limit[:, F:] * g.abs() + 2.0 ** -20 * exact.abs() + 1e-12
    assert ((ops.gemm_swiglu(a.to(DEV), w.to(DEV)).cpu().double() - exact).abs() <= allowed).all()


def test_a_row_does_not_depend_on_the_rows_beside_it(ops):
    for N, K in ((1024, 4608), (70, 36), (9216, 1024)):
        a, w = draw(330, K).to(DEV), draw(N, K, seed=1).to(DEV)
        whole = ops.gemm(a, w)
        for first, last in ((0, 1), (7, 23), (40, 57), (3, 36), (250, 330), (17, 301)):
            assert torch.equal(ops.gemm(a[first:last].contiguous(), w), whole[first:last])
        gated = ops.gemm_swiglu(a, w)
        assert torch.equal(ops.gemm_swiglu(a[5:6].contiguous(), w)[0], gated[5])


@pytest.mark.parametrize("K", [16, 64, 128, 192, 260, 272, 300, 512, 520, 4100])
def test_every_part_of_k_is_walked_once(ops, K):
    """Parts of one group and of several, the last of them cut short or empty, for waves that walk one part and waves that walk
    four: the same sums to the bit."""
    a, w = draw(70, K), draw(150, K, seed=1)
    A, W = a.to(DEV), w.to(DEV)
    whole = ops.gemm(A, W)
    assert ((whole.cpu().double() - a.double() @ w.double().T).abs() <= bound(a, w)).all()
    for first, last in ((0, 1), (3, 20), (30, 70)):
        assert torch.equal(ops.gemm(A[first:last].contiguous(), W), whole[first:last])


def test_what_its_loads_cannot_take_goes_to_the_plain_tiles(ops):
    a, w = draw(5, 66), draw(40, 66, seed=1)                       # K no multiple of 4
    exact = a.double() @ w.double().T
    assert ((ops.gemm(a.to(DEV), w.to(DEV)).cpu().double() - exact).abs() <= bound(a, w)).all()
    flat = torch.cat([torch.zeros(1), draw(5, 64).reshape(-1)]).to(DEV)     # rows that do not start at 16 bytes
    b, v = flat[1:].view(5, 64), draw(40, 64, seed=1)
    exact = b.cpu().double() @ v.double().T
    assert ((ops.gemm(b, v.to(DEV)).cpu().double() - exact).abs() <= bound(b.cpu(), v)).all()


# K of whole groups and parts, ending inside a group, inside a part, with parts that have nothing; the deeper ring; outputs at the edges of both tiles
@pytest.mark.parametrize("K", [1024, 1028, 1040, 1280, 2052, 3900, 4096, 4100, 8192])
@pytest.mark.parametrize("N", [1, 5, 1024, 3071, 3072, 3081])
def test_few_rows_have_the_values_of_many(ops, N, K):
    """One row, two over a short K or that add, go to a kernel of their own, more to the matrix instruction: the same bits, with and without the norm in front."""
    # what the threads hold of the rows, and where two rows' multiply-adds in line are still the faster ones
    takes = {(rows, mode): rows * K <= 8192 and (rows == 1 or mode == 1 or K == 1024) for rows in (1, 2) for mode in (0, 1, 2)}
    for rows in (1, 2, 3):
        for mode in (0, 1, 2):
            assert bool(ops.library().fw_gemm_float32_few_rows(mode, rows, N, K)) == takes.get((rows, mode), False)
            if mode != 1:
                assert ops.float32_normed_takes(mode == 2, rows, N, K) == (takes.get((rows, mode), False) and K <= 4096)
    a, w = draw(19, K).to(DEV), draw(2 * N, K, seed=1).to(DEV)
    bias, weight = draw(N, seed=2).to(DEV), draw(K, seed=3).to(DEV)
    old = draw(19, N, seed=4).to(DEV)
    for one_centered in (False, True):
        if K > 4096 or (one_centered and N > 5):
            break
        normed = ops.rmsnorm_rows(a, weight, 1e-5, torch.float32, one_centered=one_centered)
        stored, gated = ops.gemm(normed, w[:N], bias), ops.gemm_swiglu(normed, w)
        index = torch.tensor([11, 4], dtype=torch.int32, device=DEV)
        for rows in (1, 2):
            of = index[:rows].long()
            if takes[rows, 0]:
                assert torch.equal(ops.gemm_float32_normed(a, weight, 1e-5, one_centered, w[:N].contiguous(), bias, row_index=index[:rows]), stored[of])
                assert torch.equal(ops.gemm_float32_normed(a[:rows].contiguous(), weight, 1e-5, one_centered, w[:N].contiguous(), bias), stored[:rows])
            if takes[rows, 2]:
                assert torch.equal(ops.gemm_float32_normed(a, weight, 1e-5, one_centered, w, row_index=index[:rows], gated=True), gated[of])
    stored, gated = ops.gemm(a, w[:N], bias), ops.gemm_swiglu(a, w)
    total = ops.gemm(a, w[:N], accumulate_into=old.clone())
    rounded = ops.gemm(a, w[:N], out_dtype=torch.bfloat16)
    for rows in (1, 2):
        few = a[:rows].contiguous()
        assert torch.equal(ops.gemm(few, w[:N], bias), stored[:rows])
        assert torch.equal(ops.gemm(few, w[:N], out_dtype=torch.bfloat16), rounded[:rows])
        assert torch.equal(ops.gemm(few, w[:N], accumulate_into=old[:rows].clone()), total[:rows])
        assert torch.equal(ops.gemm_swiglu(few, w), gated[:rows])


def test_what_a_normed_product_of_few_rows_refuses(ops):
    assert not ops.float32_normed_takes(False, 3, 64, 1024) and not ops.float32_normed_takes(False, 1, 64, 4100) and not ops.float32_normed_takes(False, 1, 64, 1020)
    a, w, weight = draw(1, 1020).to(DEV), draw(64, 1020, seed=1).to(DEV), draw(1020, seed=2).to(DEV)
    with pytest.raises(ops.KernelError, match="not taken"):
        ops.gemm_float32_normed(a, weight, 1e-5, False, w)
    with pytest.raises(ops.KernelError, match="norm"):
        ops.gemm_float32_normed(a, weight[:1000].contiguous(), 1e-5, False, w)


@pytest.mark.parametrize("odd", ["rows", "weight", "norm"])
def test_one_normed_row_of_operands_at_odd_places(ops, odd):
    """A linear part whose weight, norm or row does not start at 16 bytes: norm and product apart, as with more rows."""
    from flyweight_amd.config.spec import PartSpec
    from flyweight_amd.parts.linear import Linear
    from flyweight_amd.parts.norm import LazyNorm, RMSNorm

    def placed(name, t):
        held = torch.zeros(t.numel() + 1, device=DEV)
        held[1:] = t.to(DEV).reshape(-1)
        return held[1:].view(t.shape) if name == odd else t.to(DEV)

    x, w, weight, bias = draw(1, 1024), draw(64, 1024, seed=1), 1.0 + 0.1 * draw(1024, seed=2), draw(64, seed=3)
    norm = RMSNorm(PartSpec("rmsnorm", {"size": 1024, "eps": 1e-5}))
    norm.bind({norm.tensor_name: placed("norm", weight)}, torch.float32, torch.device(DEV))
    X, W = placed("rows", x), placed("weight", w)
    normed = x.double() * torch.rsqrt(x.double().pow(2).mean() + 1e-5) * weight.double()
    # the row's mean of squares, root and two products are a few roundings each beside those of the product
    limit = bound(normed, w) + 8 * 2.0 ** -24 * (normed.abs() @ w.double().abs().T)
    sums = normed @ w.double().T
    stored = Linear(W, bias.to(DEV)).forward(LazyNorm(norm, X, None), out_dtype=torch.float32).cpu().double()
    assert ((stored - sums - bias.double()).abs() <= limit + 2.0 ** -23 * stored.abs()).all()
    gated = Linear(W).swiglu(LazyNorm(norm, X, None)).cpu().double()
    g, u = sums[:, :32], sums[:, 32:]
    exact = torch.nn.functional.silu(g) * u
    allowed = 1.1 * limit[:, :32] * u.abs() + limit[:, 32:] * g.abs() + 2.0 ** -20 * exact.abs() + 1e-12     # (as the gated product above)
    assert ((gated - exact).abs() <= allowed).all()


@pytest.mark.parametrize("nh,nkv,hd,v_dim,window,keep_first,sink,slope,softcap,chunk", [
    (4, 2, 64, 64, 0, 0, False, False, 0.0, 0), (6, 2, 64, 48, 70, 0, False, False, 0.0, 0), (4, 1, 128, 128, 100, 70, True, False, 0.0, 0),
    (2, 2, 20, 320, 0, 0, False, True, 0.0, 0), (4, 2, 320, 64, 0, 0, False, False, 6.0, 0), (4, 2, 64, 1024, 0, 0, True, False, 0.0, 130)])
def test_attention_of_few_rows_has_the_values_of_many(ops, nh, nkv, hd, v_dim, window, keep_first, sink, slope, softcap, chunk):
    """Eight pages side by side, folded in their order: the same bits as a page after the other, for contexts of one page to more than two rounds of eight."""
    lengths = [1, 63, 64, 65, 300, 512, 513, 1100]
    generator = torch.Generator().manual_seed(1)
    many = 300 // nh + 1                                    # copies of the rows: more rows times heads than compute units
    pages = [(n + 63) // 64 for n in lengths]
    order = torch.randperm(sum(pages), generator=generator).tolist()
    table = torch.zeros(len(lengths), max(pages), dtype=torch.int32)
    for i, n in enumerate(pages):
        table[i, :n] = torch.tensor([order.pop() for _ in range(n)])
    k_pages, v_pages = draw(sum(pages), nkv, 64, hd, seed=2).to(DEV), draw(sum(pages), nkv, v_dim, 64, seed=3).to(DEV)
    for i, n in enumerate(lengths):                         # what lies behind the last key is not a number
        if n % 64:
            v_pages[table[i, pages[i] - 1].item(), :, :, n % 64:] = float("nan")
            k_pages[table[i, pages[i] - 1].item(), :, n % 64:] = float("nan")
    sinks = draw(nh, seed=4).to(DEV) if sink else None
    slopes = (0.05 * torch.rand(nh, generator=generator)).to(DEV) if slope else None
    table = table.to(DEV)
    for i, n in enumerate(lengths):
        q = draw(1, nh * hd, seed=10 + i).to(DEV)
        run = lambda copies: ops.attention_generic(q.repeat(copies, 1), nh, nkv, hd, k_pages, v_pages, table, torch.full((copies,), i, dtype=torch.int32, device=DEV),   # noqa: E731,E501,B023
                                                   torch.full((copies,), n - 1, dtype=torch.int32, device=DEV), hd ** -0.5, window, v_dim=v_dim, chunk=chunk,      # noqa: B023
                                                   softcap=softcap, keep_first=keep_first, sinks=sinks, slopes=slopes)
        few, rows = run(1), run(many)
        assert torch.isfinite(few).all()
        assert torch.equal(rows, few.expand_as(rows))
