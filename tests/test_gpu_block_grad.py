"""The gradient of a block's sum / mean towards its input (every source row written once): widths at the edges of the
lane groups, rows without edges, rows of the lengths at which the way of adding them up changes (8: the lanes of the smallest
group; 16: what a group adds up alone; 512, or a 512th of all edges: what a workgroup adds up alone), hubs, and both edge
orders."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _block(num_dst, fanout, num_src, seed):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    for s, n in ((0, 32), (1, 33), (2, 64), (3, 65), (4, 700)):          # sources with about so many edges
        if s < num_src and n <= r.size // 8:
            r[rng.choice(r.size, n, replace=False)] = s
    r[rng.random(r.size) < 0.2] = -1
    return torch.from_numpy(r.astype(np.int64)).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("num_dst,fanout,num_src,dim", [(1, 1, 1, 1), (700, 15, 5000, 47), (700, 15, 400, 4), (900, 10, 3000, 32),
                                                        (900, 10, 3000, 36), (900, 10, 3000, 100), (500, 25, 9000, 256),
                                                        (300, 20, 2000, 264), (300, 20, 2000, 600), (4000, 5, 70000, 8),
                                                        (40000, 15, 90000, 4)])
@pytest.mark.parametrize("mean", [False, True])
@pytest.mark.parametrize("with_csr", [False, True])
def test_block_aggregate_backward(capi, num_dst, fanout, num_src, dim, dtype, mean, with_csr):
    import apt_amd  # noqa: F401  (loads the operators)
    rel = _block(num_dst, fanout, num_src, num_dst + dim)
    gen = torch.Generator(device=DEV).manual_seed(dim)
    x = torch.randn(num_src, dim, generator=gen, device=DEV).to(dtype).requires_grad_(True)
    up = torch.randn(num_dst, dim, generator=gen, device=DEV).to(dtype)
    f = capi.block_formats(rel, num_dst, fanout, num_src) if with_csr else {}
    out = torch.ops.npc.block_aggregate(rel, num_dst, fanout, x, mean, f.get("csr_indptr"), f.get("csr_indices"))
    dx, = torch.autograd.grad(out, x, up)
    keep = (rel >= 0).nonzero().flatten()
    src, dst = rel[keep], keep // fanout
    xd, w = x.detach().double(), torch.ones(keep.numel(), device=DEV, dtype=torch.float64)
    if mean:
        w = 1.0 / torch.bincount(dst, minlength=num_dst).clamp(min=1).double()[dst]
    want = torch.zeros(num_dst, dim, device=DEV, dtype=torch.float64).index_add(0, dst, xd[src] * w[:, None])
    want_dx = torch.zeros(num_src, dim, device=DEV, dtype=torch.float64).index_add(0, src, up.double()[dst] * w[:, None])
    size = torch.zeros(num_src, dim, device=DEV, dtype=torch.float64).index_add(0, src, up.double().abs()[dst] * w[:, None])
    # fp32 sums of terms adding up to `size` in magnitude, then one rounding to the output's type
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22
    assert out.dtype == dtype and bool(((out.double() - want).abs() <= 1e-5 * (1 + want.abs()) + half * want.abs() + half).all())
    assert dx.dtype == dtype and bool(((dx.double() - want_dx).abs() <= 1e-6 * size + half * want_dx.abs()).all())
    again, = torch.autograd.grad(torch.ops.npc.block_aggregate(rel, num_dst, fanout, x, mean, f.get("csr_indptr"),
                                                               f.get("csr_indices")), x, up)
    assert torch.equal(dx, again)


# Sources with exactly so many edges.  A row of more than 512 is summed in chunks of 256.  With 400 k more edges in a row,
# one of more than 812 is (a 512th of the slots), in chunks of 406.
COUNTS = [0, 1, 7, 8, 9, 15, 16, 17, 18, 31, 32, 33, 64, 65, 255, 256, 257, 511, 512, 513, 514, 767, 768, 769, 811, 812, 813, 814, 1025, 5000, 0, 2]


def _counted_block(counts, fanout, holes, seed):
    """Slots in random order that name source s counts[s] times, and -1."""
    rng = np.random.default_rng(seed)
    r = np.concatenate([np.repeat(np.arange(len(counts)), counts), np.full(holes, -1)])
    r = np.concatenate([r, np.full(-r.size % fanout, -1)])
    return torch.from_numpy(rng.permutation(r).astype(np.int64)).to(DEV), r.size // fanout


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [4, 8, 33, 64, 256, 264])
@pytest.mark.parametrize("with_csr", [False, True])
@pytest.mark.parametrize("last", [0, 400_000])
def test_rows_of_every_length(capi, dim, dtype, with_csr, last):
    import apt_amd  # noqa: F401
    if last and dim not in (8, 64):
        pytest.skip("one narrow and one wide row are enough for the longest")
    counts = COUNTS + [last, 3, 0]
    num_src = len(counts)
    rel, num_dst = _counted_block(counts, 5, 777, dim)
    gen = torch.Generator(device=DEV).manual_seed(dim)
    x = torch.randn(num_src, dim, generator=gen, device=DEV).to(dtype).requires_grad_(True)
    up = torch.randn(num_dst, dim, generator=gen, device=DEV).to(dtype)
    f = capi.block_formats(rel, num_dst, 5, num_src) if with_csr else {}
    grad = lambda: torch.autograd.grad(torch.ops.npc.block_aggregate(rel, num_dst, 5, x, True, f.get("csr_indptr"),  # noqa: E731
                                                                     f.get("csr_indices")), x, up)[0]
    keep = (rel >= 0).nonzero().flatten()
    src, dst = rel[keep], keep // 5
    assert torch.bincount(src, minlength=num_src).tolist() == counts
    w = 1.0 / torch.bincount(dst, minlength=num_dst).clamp(min=1).double()[dst]
    terms = up.double()[dst] * w[:, None]
    pick = (torch.arange(num_src, device=DEV)[:, None] == src).double()
    want, size = pick @ terms, pick @ terms.abs()
    dx = grad()
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22
    assert bool(((dx.double() - want).abs() <= 1e-6 * size + half * want.abs()).all())
    for _ in range(3):      # whichever workgroup adds a row's chunks up
        assert torch.equal(grad(), dx)


def test_a_hub_takes_no_longer_than_an_even_block(capi):
    """100 k edges of one source, 64 features: 13 times the even block's backward pass while one workgroup added a row up
    (1660 against 122 us; the bound leaves room for a busy machine)."""
    import apt_amd  # noqa: F401
    num_dst, fanout, num_src, dim = 100_000, 10, 300_000, 64
    rel = torch.randint(0, num_src, (num_dst * fanout,), device=DEV)
    x = torch.randn(num_src, dim, device=DEV, requires_grad=True)
    up = torch.randn(num_dst, dim, device=DEV)

    def fastest():
        times = []
        for _ in range(8):
            out = torch.ops.npc.block_aggregate(rel, num_dst, fanout, x, False, None, None)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            torch.autograd.grad(out, x, up)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    even = fastest()
    rel.view(num_dst, fanout)[:, 3] = 70_000
    assert fastest() <= 4 * even


def test_block_aggregate_empty_and_wrong_inputs():
    import apt_amd  # noqa: F401
    op = torch.ops.npc.block_aggregate
    x = torch.randn(5, 8, device=DEV, requires_grad=True)
    rel = torch.full((6,), -1, dtype=torch.int64, device=DEV)
    out = op(rel, 3, 2, x, True, None, None)
    dx, = torch.autograd.grad(out.sum(), x)
    assert not out.any() and not dx.any()
    empty = op(rel[:0], 0, 2, x, False, None, None)
    assert empty.shape == (0, 8) and not torch.autograd.grad(empty.sum(), x)[0].any()
    with pytest.raises(TypeError):
        op(rel, 3, 2, x.double(), True, None, None)
    with pytest.raises(TypeError):
        op(rel.cpu(), 3, 2, x, True, None, None)
    with pytest.raises(RuntimeError):
        op(rel, 4, 2, x, True, None, None)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [16, 47, 64, 128, 256, 300])
@pytest.mark.parametrize("num_src", [40, 1100, 9000])
def test_hubs_of_every_class(dim, dtype, num_src):
    """Sources of 0 .. 600 edges around the lengths where another part of the kernel takes them (16, 32, 128 edges, 512 of a
    long row), side by side, in launches with and without a whole slab of neighbouring rows for every XCD."""
    import apt_amd  # noqa: F401  (loads the operators)
    gen = torch.Generator(device=DEV).manual_seed(dim + num_src)
    degrees = [0, 1, 2, 4, 5, 15, 16, 17, 18, 31, 32, 33, 47, 63, 64, 65, 127, 128, 129, 200, 513, 600]
    slots = torch.cat([torch.full((n,), i * 7 % num_src if num_src > 154 else i, dtype=torch.int64) for i, n in enumerate(degrees)]
                      + [torch.arange(num_src, dtype=torch.int64), torch.full((3,), -1, dtype=torch.int64)]).to(DEV)
    fanout = 10
    num_dst = -(-slots.numel() // fanout)
    slots = torch.nn.functional.pad(slots, (0, num_dst * fanout - slots.numel()), value=-1)
    slots = slots[torch.randperm(slots.numel(), generator=gen, device=DEV)].contiguous()
    x = torch.randn(num_src, dim, generator=gen, device=DEV).to(dtype).requires_grad_(True)
    up = torch.randn(num_dst, dim, generator=gen, device=DEV).to(dtype)
    got, = torch.autograd.grad(torch.ops.npc.block_aggregate(slots, num_dst, fanout, x, True, None, None), x, up)
    there = slots.view(num_dst, fanout) >= 0
    weighted = up.double() / there.sum(1, keepdim=True).clamp(min=1)
    edge = there.nonzero()[:, 0], slots[slots >= 0]
    want = torch.zeros(num_src, dim, dtype=torch.float64, device=DEV).index_add_(0, edge[1], weighted[edge[0]])
    size = torch.zeros_like(want).index_add_(0, edge[1], weighted[edge[0]].abs())
    # fp32 sums of n terms in any order: n 2^-24 of the terms' absolute sum, one rounding more for the factor of each; a
    # bf16 result is rounded at 2^-9
    count = torch.bincount(edge[1], minlength=num_src).unsqueeze(1)
    bound = (count + 3) * 2.0 ** -24 * size + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) * want.abs()
    assert got.dtype == dtype and bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [4, 8, 33, 64, 128, 256])
@pytest.mark.parametrize("num_src,hubs", [(40, 40), (600, 90), (3000, 3000), (70000, 700)])
def test_many_hubs(capi, num_src, hubs, dim, dtype):
    """Neighbouring sources of 17 to 140 edges among those of two: whole workgroups of hubs, of which the lane groups take one
    each, workgroups with one or two of them, and grids of rows that come out even and that do not."""
    import apt_amd  # noqa: F401
    rng = np.random.default_rng(num_src + dim)
    counts = np.full(num_src, 2)
    first = min(num_src // 3, num_src - hubs)
    counts[first:first + hubs] = rng.integers(17, 141, size=hubs)
    rel, num_dst = _counted_block(list(counts), 5, 100, num_src)
    gen = torch.Generator(device=DEV).manual_seed(dim)
    x = torch.zeros(num_src, dim, device=DEV, dtype=dtype, requires_grad=True)
    up = torch.randn(num_dst, dim, generator=gen, device=DEV).to(dtype)
    out = torch.ops.npc.block_aggregate(rel, num_dst, 5, x, False, None, None)
    dx, = torch.autograd.grad(out, x, up, retain_graph=True)
    keep = (rel >= 0).nonzero().flatten()
    src, rows = rel[keep], up.double()[keep // 5]
    want = torch.zeros(num_src, dim, device=DEV, dtype=torch.float64).index_add(0, src, rows)
    size = torch.zeros(num_src, dim, device=DEV, dtype=torch.float64).index_add(0, src, rows.abs())
    # fp32 sums of up to 140 terms, one rounding to the result's type
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0      # (half a unit in the last of eight bits)
    assert bool(((dx.double() - want).abs() <= 140 * 2.0 ** -24 * size + half * want.abs()).all())
    assert torch.equal(dx, torch.autograd.grad(out, x, up)[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [16, 33, 256])
def test_edges_without_rows(capi, dim, dtype):
    """No row on the other side, but edges (none of which counts then): zeros, and nothing is read in their place, through
    the C interface as a NULL, or rows that nobody may read."""
    L, es = capi.lib(), 2 if dtype == torch.bfloat16 else 4
    i64 = dict(dtype=torch.int64, device=DEV)
    num_src, counts = 50, torch.arange(50, device=DEV)
    indptr = torch.zeros(num_src + 1, **i64)
    indptr[1:] = torch.cumsum(counts, 0)
    edges = int(indptr[-1])
    index = torch.zeros(edges, **i64)
    dx = torch.full((num_src, dim), 7.0, device=DEV, dtype=dtype)
    stream = capi._stream()
    capi.check(L.apt_block_aggregate_backward(indptr.data_ptr(), index.data_ptr(), 8, 5, num_src, edges, None, None, 1.0, None, 0,
                                              dim, es, dx.data_ptr(), None, 0, stream))
    assert not bool(dx.any())
    keys = torch.repeat_interleave(torch.arange(num_src, device=DEV), counts)
    unreadable = torch.full((1,), float("nan"), device=DEV)
    edata = torch.ones(edges, dim, device=DEV, dtype=dtype)
    for mode in (0, 2):
        for grouped in (1, 0):
            need = int(L.apt_coo_sum_workspace_bytes(edges, num_src, grouped, 0, dim))
            ws = torch.empty(max(need, 256), dtype=torch.uint8, device=DEV)
            dx.fill_(7.0)
            capi.check(L.apt_coo_sum(mode, keys.data_ptr(), index.data_ptr(), edges, grouped, 0, unreadable.data_ptr(), 0,
                                     edata.data_ptr() if mode == 2 else None, dim, es, dx.data_ptr(), num_src, ws.data_ptr(),
                                     ws.numel(), stream))
            assert not bool(dx.any())
