"""The fused GAT layer (scores, edge softmax, weighted sum, bias, and all gradients) against the separate operations in
torch, sums over edges in float64 (bf16 rows: the operations between them in bf16, as a bf16 model has them): heads and widths on every path (a wavefront per destination, lane groups, features that cross a head's
edge inside a vector), hubs, destinations without edges, both edge orders."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _separate(rel, num_dst, fanout, ft_row, al, ar, bias, slope):
    el_row, er_row = (ft_row * al).sum(-1), (ft_row[:num_dst] * ar).sum(-1)
    ft, el, er = ft_row.double(), el_row.double(), er_row.double()
    keep = (rel >= 0).nonzero().flatten()
    src, dst = rel[keep], keep // fanout
    heads, dim = ft.shape[1:]
    e = torch.nn.functional.leaky_relu(el[src] + er[dst], slope)
    top = torch.full((num_dst, heads), -1e30, device=DEV, dtype=ft.dtype).scatter_reduce(0, dst[:, None].expand(-1, heads), e.detach(), "amax")
    w = torch.exp(e - top[dst])
    den = torch.zeros(num_dst, heads, device=DEV, dtype=ft.dtype).index_add(0, dst, w)
    out = torch.zeros(num_dst, heads, dim, device=DEV, dtype=ft.dtype).index_add(0, dst, (w / den[dst])[:, :, None] * ft[src])
    return out.to(ft_row.dtype) + bias


@pytest.mark.parametrize("dtype,attn_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                              (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("num_dst,fanout,num_src,heads,dim", [
    (300, 15, 2500, 4, 64), (300, 10, 2500, 4, 47), (200, 7, 900, 3, 8), (150, 9, 700, 1, 5), (150, 9, 700, 8, 8),
    (100, 25, 800, 2, 100), (100, 20, 800, 8, 64), (64, 64, 500, 1, 256), (1, 1, 1, 1, 1), (90, 5, 400, 4, 6), (80, 5, 300, 5, 3)])
@pytest.mark.parametrize("with_csr", [False, True])
def test_gat_layer(capi, num_dst, fanout, num_src, heads, dim, dtype, attn_dtype, with_csr):
    import apt_amd  # noqa: F401
    rng = np.random.default_rng(num_dst + dim)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    if r.size > 800:
        r[rng.choice(r.size, 300, replace=False)] = min(3, num_src - 1)         # a hub
    r[rng.random(r.size) < 0.2] = -1
    r[:fanout] = -1 if num_dst > 1 else 0                                       # a destination without edges
    rel = torch.from_numpy(r.astype(np.int64)).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(heads * dim)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    ft = rand(num_src, heads, dim).to(dtype).requires_grad_(True)
    al, ar = (rand(heads, dim) * 0.3).to(attn_dtype).requires_grad_(True), (rand(heads, dim) * 0.3).to(attn_dtype).requires_grad_(True)
    bias = rand(heads * dim).to(dtype).requires_grad_(True)
    up = rand(num_dst, heads, dim).to(dtype)
    f = capi.block_formats(rel, num_dst, fanout, num_src) if with_csr else {}
    csr = [f.get(k) for k in ("csr_indptr", "csr_indices", "csr_eids", "csc_indptr")]
    out = torch.ops.npc.gat_layer(rel, num_dst, fanout, ft, al, ar, bias, 0.2, *csr)
    got = torch.autograd.grad(out, [ft, al, ar, bias], up)
    wide = torch.float64 if dtype == torch.float32 else None      # fp32: everything in float64
    leaves = [(t.detach() if wide is None else t.detach().to(wide)).requires_grad_(True) for t in (ft, al, ar, bias.view(heads, dim))]
    ref = _separate(rel, num_dst, fanout, *leaves, 0.2)
    want = torch.autograd.grad(ref, leaves, up.to(ref.dtype))
    # fp32: sums of a few thousand products.  bf16: an fp32 sum next to a rounding boundary may round the other way in
    # another order, 2^-8 of that value; the attention vectors' gradients are sums of terms that cancel, so there
    # it weighs more.
    for a, b, name in zip((out,) + got, (ref,) + want, ("out", "ft", "attn_l", "attn_r", "bias")):
        assert a.dtype == (attn_dtype if name.startswith("attn") else dtype)
        tol = 1e-4 if dtype == torch.float32 else 3e-2 if name.startswith("attn") else 1e-2
        err = (a.double().reshape(-1) - b.double().reshape(-1)).abs().max().item()
        assert err <= tol * (b.abs().max().item() + 1e-2), (name, err, b.abs().max().item())
    with torch.no_grad():
        assert torch.equal(torch.ops.npc.gat_layer(rel, num_dst, fanout, ft, al, ar, bias, 0.2, *csr), out)


@pytest.mark.parametrize("dtype,attn_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                              (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("num_dst,num_src", [(0, 0), (0, 70)])
def test_gat_layer_without_destinations(capi, num_dst, num_src, dtype, attn_dtype):
    """No row and no edge: every gradient is zero, as torch's sums over nothing are."""
    import apt_amd  # noqa: F401
    heads, dim, fanout = 4, 24, 5
    rel = torch.empty(0, dtype=torch.int64, device=DEV)
    ft = torch.randn(num_src, heads, dim, device=DEV).to(dtype).requires_grad_(True)
    al, ar = (torch.randn(heads, dim, device=DEV).to(attn_dtype).requires_grad_(True) for _ in range(2))
    bias = torch.randn(heads * dim, device=DEV).to(dtype).requires_grad_(True)
    out = torch.ops.npc.gat_layer(rel, num_dst, fanout, ft, al, ar, bias, 0.2, None, None, None, None)
    assert out.shape == (num_dst, heads, dim)
    # what the gradients are allocated from: blocks of their sizes that hold something else
    dirty = [torch.full((heads, dim), float("nan"), device=DEV, dtype=t) for t in (dtype, attn_dtype) for _ in range(8)]
    del dirty
    for g, t in zip(torch.autograd.grad(out, [ft, al, ar, bias], torch.zeros_like(out)), (ft, al, ar, bias)):
        assert g.shape == t.shape and g.dtype == t.dtype and bool((g == 0).all())


@pytest.mark.parametrize("heads,dim,fanout", [(4, 16, 9), (3, 24, 9), (2, 100, 9), (4, 64, 20), (1, 5, 7)])
@pytest.mark.parametrize("attn_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("activation", [None, torch.relu])
def test_gat_layer_bf16_without_gradients_keeps_fp32(capi, heads, dim, fanout, attn_dtype, activation):
    """Scores, softmax, sum and result of a bf16 layer are fp32 under no_grad: 1e-5 of the same bf16 rows' float64
    result (a rounding of a score or of the result to bf16 is 4e-3).  The next layer takes that result."""
    from apt_amd.layers import GATConv
    from apt_amd.sampler import Block
    num_dst, num_src = 400, 1500
    rng = np.random.default_rng(heads * dim + fanout)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    r[rng.random(r.size) < 0.2] = -1
    r[:fanout] = -1
    rel = torch.from_numpy(r.astype(np.int64)).to(DEV)
    torch.manual_seed(3)
    layer = GATConv(40, dim, heads, activation=activation).to(DEV, torch.bfloat16)
    with torch.no_grad():
        layer.bias.normal_()
    for p in (layer.attn_l, layer.attn_r):
        p.data = p.data.to(attn_dtype)
    blk = Block(num_src, num_dst, None, rel, fanout)
    feat = torch.randn(num_src, 40, device=DEV).bfloat16()
    with torch.no_grad():
        got = layer(blk, feat)
        ft, al, ar = layer.fc(feat).view(num_src, heads, dim).double(), layer.attn_l.double(), layer.attn_r.double()
        want = _separate(rel, num_dst, fanout, ft, al, ar, layer.bias.view(heads, dim).double(), 0.2)
        want = want if activation is None else activation(want)
        assert got.dtype == torch.float32
        assert (got.double() - want).abs().max().item() <= 1e-5 * want.abs().max().item()
        upper = GATConv(heads * dim, 8, 2).to(DEV, torch.bfloat16)
        top = Block(num_dst, 50, None, torch.randint(0, num_dst, (50 * 4,), device=DEV), 4)
        assert torch.equal(upper(top, got.flatten(1)), upper(top, got.flatten(1).bfloat16()))
    assert layer(blk, feat).dtype == torch.bfloat16     # a training step


@pytest.mark.parametrize("dtype,attn_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("heads,dim", [(4, 64), (8, 8), (3, 6), (1, 5), (5, 3), (2, 100)])
@pytest.mark.parametrize("with_csr", [False, True])
def test_gat_layer_sources_with_given_numbers_of_edges(capi, heads, dim, dtype, attn_dtype, with_csr):
    """Rows of the source half at the lengths where the way of adding them up changes: 8 (the lanes of the smallest group),
    16 (a group alone), 512 (a workgroup alone), several chunks, a 512th of the row to a chunk."""
    import apt_amd  # noqa: F401
    counts = [0, 7, 8, 9, 15, 16, 17, 18, 33, 255, 511, 512, 513, 769, 5000, 140_000 if heads * dim <= 64 else 900, 1]
    fanout, rng = 6, np.random.default_rng(heads * dim)
    r = np.concatenate([np.repeat(np.arange(len(counts)), counts), np.full(1000, -1)])
    r = rng.permutation(np.concatenate([r, np.full(-r.size % fanout, -1)]))
    num_dst, rel = r.size // fanout, torch.from_numpy(r.astype(np.int64)).to(DEV)
    num_src = max(num_dst, len(counts))                     # the destinations are the first sources
    gen = torch.Generator(device=DEV).manual_seed(dim)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    ft = rand(num_src, heads, dim).to(dtype).requires_grad_(True)
    al, ar = ((rand(heads, dim) * 0.3).to(attn_dtype).requires_grad_(True) for _ in range(2))
    up = rand(num_dst, heads, dim).to(dtype)
    f = capi.block_formats(rel, num_dst, fanout, num_src) if with_csr else {}
    csr = [f.get(k) for k in ("csr_indptr", "csr_indices", "csr_eids", "csc_indptr")]
    grads = lambda: torch.autograd.grad(torch.ops.npc.gat_layer(rel, num_dst, fanout, ft, al, ar, None, 0.2, *csr), [ft, al, ar], up)  # noqa: E731
    got = grads()
    wide = torch.float64 if dtype == torch.float32 else None
    leaves = [(t.detach() if wide is None else t.detach().to(wide)).requires_grad_(True) for t in (ft, al, ar)]
    ref = _separate(rel, num_dst, fanout, *leaves, torch.zeros((), device=DEV, dtype=leaves[0].dtype), 0.2)
    want = torch.autograd.grad(ref, leaves, up.to(ref.dtype))
    # As in test_gat_layer; a source's gradient is a sum of up to 140 k terms of its own magnitude: to the sum's norm.
    for a, b, name in zip(got, want, ("ft", "attn_l", "attn_r")):
        tol = 2e-5 if dtype == torch.float32 else 5e-2 if name.startswith("attn") else 1e-2
        a, b = a.double().reshape(-1), b.double().reshape(-1)
        assert bool((a - b).norm() <= tol * b.norm()), (name, ((a - b).norm() / b.norm()).item())
    for a, b in zip(got, grads()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,attn_dtype", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                              (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("num_dst,fanout,num_src,heads,dim", [
    (1, 1, 1, 1, 4), (70, 5, 400, 4, 64), (70, 6, 400, 4, 64), (33, 10, 300, 2, 128), (33, 11, 300, 1, 16), (50, 16, 300, 4, 8),
    (50, 17, 300, 2, 8), (20, 8, 90, 8, 32), (40, 7, 200, 4, 47), (40, 3, 200, 1, 10)])
def test_scores_formed_where_they_are_used(capi, num_dst, fanout, num_src, heads, dim, dtype, attn_dtype):
    """Without gradients: the slots that a wavefront's registers hold (5, 10, 16, and one more), against float64; and fp32
    with the bits of the layer that has gradients, rows with infinities and NaN included."""
    import apt_amd  # noqa: F401
    rng = np.random.default_rng(num_dst * fanout)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    r[rng.random(r.size) < 0.25] = -1
    r[-fanout:] = -1 if num_dst > 1 else 0
    rel = torch.from_numpy(r.astype(np.int64)).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(heads * dim)
    ft = torch.randn(num_src, heads, dim, generator=gen, device=DEV).to(dtype)
    al, ar = ((torch.randn(heads, dim, generator=gen, device=DEV) * 0.3).to(attn_dtype) for _ in range(2))
    bias = torch.randn(heads, dim, generator=gen, device=DEV).to(dtype)
    got = torch.ops.npc.gat_layer(rel, num_dst, fanout, ft, al, ar, bias, 0.2, None, None, None, None, False, True)
    want = _separate(rel, num_dst, fanout, ft.double(), al.double(), ar.double(), bias.double(), 0.2)
    # fp32: dots of up to 128 products move a weight by less than 1e-5, a sum of 16 rows adds 1e-6
    assert got.dtype == torch.float32 and bool(((got.double() - want).abs() <= 2e-5 * (1 + want.abs().max())).all())
    if dtype == torch.float32:
        ft[0, 0, 0], ft[num_src // 2, heads - 1, dim - 1] = float("inf"), float("nan")
        rest = (al, ar, bias, 0.2, None, None, None, None)
        plain = torch.ops.npc.gat_layer(rel, num_dst, fanout, ft, *rest)
        grad = torch.ops.npc.gat_layer(rel, num_dst, fanout, ft.clone().requires_grad_(True), *rest)
        assert torch.equal(plain.isnan(), grad.isnan()) and torch.equal(plain.nan_to_num(7.0), grad.detach().nan_to_num(7.0))


@pytest.mark.parametrize("num_dst,fanout,heads,dim", [(2048, 10, 2, 64), (2049, 10, 2, 64), (8000, 10, 4, 32), (8001, 10, 4, 32),
                                                      (9000, 10, 1, 256), (3300, 5, 1, 64), (13200, 5, 1, 64), (13200, 5, 4, 64),
                                                      (1500, 16, 4, 64), (1500, 16, 2, 128), (5, 16, 1, 4)])
def test_scores_formed_where_they_are_used_or_before(num_dst, fanout, heads, dim):
    """The two ways of a layer without gradients, on either side of where one becomes the faster: the bits of the layer with
    gradients in fp32, and for bf16 rows those of an fp32 layer up to the order of a score's products."""
    import apt_amd  # noqa: F401
    gen = torch.Generator(device=DEV).manual_seed(num_dst)
    num_src = num_dst + 500
    rel = torch.randint(-1, num_src, (num_dst * fanout,), generator=gen, device=DEV)
    ft, al, ar = (torch.randn(*s, heads, dim, generator=gen, device=DEV).bfloat16() for s in ((num_src,), (), ()))
    call = lambda *v: torch.ops.npc.gat_layer(rel, num_dst, fanout, *v, None, 0.2, None, None, None, None, False, True)  # noqa: E731
    whole = [t.float() for t in (ft, al, ar)]
    with torch.no_grad():
        got, half = call(*whole), call(ft, al, ar)
    assert torch.equal(got, call(*(t.clone().requires_grad_(True) for t in whole)))
    # a score is a sum of dim products (|products| up to about 4 sqrt(dim)): its error enters the weights as a factor
    assert half.dtype == torch.float32 and torch.allclose(half, got, rtol=1e-5 * dim ** 0.5, atol=1e-5 * dim ** 0.5)
