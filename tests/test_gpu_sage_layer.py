"""The GraphSAGE layer as one operator against its statement in float64 (forward and every gradient): the product before
and after the mean, with and without bias and CSR, all and few rows as destinations; gradients of gradients keep a graph."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _statement(rel, num_dst, fanout, x, wn, ws, b):
    keep = (rel >= 0).nonzero().flatten()
    src, dst = rel[keep], keep // fanout
    deg = torch.bincount(dst, minlength=num_dst).clamp(min=1).to(x.dtype)
    mean = torch.zeros(num_dst, x.shape[1], device=DEV, dtype=x.dtype).index_add(0, dst, x[src]) / deg[:, None]
    out = x[:num_dst] @ ws.t() + mean @ wn.t()
    return out if b is None else out + b


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("num_dst,fanout,num_src,k,n", [(1, 1, 1, 1, 1), (300, 5, 900, 100, 256), (300, 5, 900, 256, 47),
                                                        (700, 15, 700, 33, 31), (64, 10, 5000, 16, 64), (0, 3, 20, 8, 4)])
@pytest.mark.parametrize("bias,with_csr", [(True, False), (False, True)])
def test_sage_layer(capi, num_dst, fanout, num_src, k, n, dtype, bias, with_csr):
    import apt_amd  # noqa: F401  (loads the operators)
    rng = np.random.default_rng(num_src + k)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    r[rng.random(r.size) < 0.2] = -1
    rel = torch.from_numpy(r.astype(np.int64)).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(k)
    leaves = [torch.randn(num_src, k, generator=gen, device=DEV)] + [torch.randn(n, k, generator=gen, device=DEV) / k ** 0.5
                                                                    for _ in range(2)]
    leaves = [t.to(dtype).requires_grad_(True) for t in leaves]
    if bias:
        leaves.append(torch.randn(n, generator=gen, device=DEV).to(dtype).requires_grad_(True))
    up = torch.randn(num_dst, n, generator=gen, device=DEV).to(dtype)
    f = capi.block_formats(rel, num_dst, fanout, num_src) if with_csr and num_dst else {}
    args = lambda v: (rel, num_dst, fanout, v[0], v[1], v[2], v[3] if bias else None, f.get("csr_indptr"), f.get("csr_indices"))  # noqa: E731
    out = torch.ops.npc.sage_layer(*args(leaves))
    got = torch.autograd.grad(out, leaves, up)
    exact = [t.detach().double().requires_grad_(True) for t in leaves]
    want = _statement(rel, num_dst, fanout, *exact[:3], exact[3] if bias else None)
    grads = torch.autograd.grad(want, exact, up.double())
    # fp32: sums of up to 700 terms; bf16: up to four roundings at 2^-9 on the way to a result, of its own size or of the
    # partial results it is the sum of
    rel_err = 2e-6 if dtype == torch.float32 else 1.2e-2
    for a, b in zip((out,) + got, (want,) + grads):
        assert a.dtype == dtype and a.shape == b.shape
        assert bool((a.double() - b).norm() <= rel_err * b.norm() + 1e-30)
    # a training step has the bits of separate operations 
    lin, agg = torch.nn.functional.linear, lambda t: torch.ops.npc.block_aggregate(rel, num_dst, fanout, t, True, None, None)
    xd, wn, ws = (t.detach() for t in leaves[:3])
    apart = lin(xd[:num_dst], ws, leaves[3].detach() if bias else None) + (agg(lin(xd, wn)) if k > n else lin(agg(xd), wn))
    assert torch.equal(out, apart)
    with torch.no_grad():      # fp32 without gradients: the library's own products
        plain = torch.ops.npc.sage_layer(*args(leaves))
    assert bool((plain.double() - want).norm() <= rel_err * want.norm() + 1e-30)


def test_sage_layer_second_order_and_hooks():
    import apt_amd as npc
    from apt_amd.layers import SAGEConv
    from apt_amd.sampler import Block
    rel = torch.randint(-1, 40, (60,), device=DEV)
    block = Block(40, 12, None, rel, 5)
    for k, n in ((8, 16), (16, 8)):
        layer = SAGEConv(k, n).to(DEV)
        x = torch.randn(40, k, device=DEV, requires_grad=True)
        w = layer.fc_self.weight
        g, = torch.autograd.grad(layer(block, x).square().sum(), w, create_graph=True)
        exact = [t.detach().double().requires_grad_(True) for t in (x, layer.fc_neigh.weight, w, layer.fc_self.bias)]
        want, = torch.autograd.grad(_statement(rel, 12, 5, *exact).square().sum(), exact[2], create_graph=True)
        got2, = torch.autograd.grad(g.sum(), w)
        want2, = torch.autograd.grad(want.sum(), exact[2])
        assert torch.allclose(got2.double(), want2, rtol=1e-4, atol=1e-4)
        plain = layer(block, x)
        seen = []
        layer.fc_neigh.register_forward_hook(lambda *a: seen.append(1))     # a hook takes the layers' own modules
        assert torch.allclose(layer(block, x), plain, rtol=1e-5, atol=1e-5) and seen == [1]
        with pytest.raises(RuntimeError):
            layer(block, x[:5])
    assert npc is not None


def test_sage_layer_gradient_of_wide_results_is_rounded_once(capi):
    """bf16, more columns than the resident product takes: what a destination's row has from its own product is added to the
    sum over the edges before it is rounded.  Everything is whole numbers, so the one rounding is known."""
    import apt_amd  # noqa: F401
    gen = torch.Generator(device=DEV).manual_seed(11)
    num, k, n = 400, 24, 3000
    rel = torch.randperm(num, generator=gen, device=DEV)              # an edge for every row: the mean is the row
    whole = lambda most, *shape: torch.randint(-most, most + 1, shape, generator=gen, device=DEV).bfloat16()
    x = torch.randn(num, k, generator=gen, device=DEV).bfloat16().requires_grad_(True)
    wn = torch.zeros(n, k, device=DEV, dtype=torch.bfloat16)
    wn[:100] = whole(1, 100, k)                                        # sums of at most 100 ones: exact in bf16
    ws, up = whole(8, n, k), whole(1, num, n)
    out = torch.ops.npc.sage_layer(rel, num, 1, x, wn, ws, None, None, None)
    dx, = torch.autograd.grad(out, x, up)
    spread = torch.zeros(num, k, device=DEV, dtype=torch.float64).index_add(0, rel, up.double() @ wn.double())
    assert torch.equal(spread, spread.bfloat16().double())
    assert torch.equal(dx, (spread + up.double() @ ws.double()).bfloat16())
