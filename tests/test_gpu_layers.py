"""Layers over sampled blocks: gradients against torch's own dense arithmetic, a
GAT layer against its textbook statement, and a short training run."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _setup_graph(n=6000, deg=8, seed=0):
    from helpers import small_graph
    import apt_amd as npc
    indptr, indices = small_graph(n, deg, seed=seed)
    npc.set_topology(0, 1)
    e = torch.empty(0, dtype=torch.int64)
    npc.mix_cache_graphs(0, e, e, e, torch.from_numpy(indptr), torch.from_numpy(indices))
    return indptr, indices


def test_block_aggregate_gradients():
    import apt_amd as npc
    from apt_amd.layers import BlockAggregate
    _setup_graph()
    sampler = npc.MixedPSNeighborSampler(0, 1, [7, 4], "DP", replace=False, rng_seed=3)
    seeds = torch.from_numpy(np.random.default_rng(0).permutation(6000)[:300]).to(DEV)
    _, _, blocks = sampler.sample(None, seeds)
    for blk in blocks:
        for mean in (False, True):
            X = torch.randn(blk.num_src, 24, device=DEV, requires_grad=True)
            out = BlockAggregate.apply(blk, X, mean)
            w = torch.randn_like(out)
            (out * w).sum().backward()
            X2 = X.detach().clone().requires_grad_(True)
            ref = torch.zeros(blk.num_dst, 24, device=DEV).index_add(0, blk.col, X2[blk.row])
            if mean:
                cnt = torch.bincount(blk.col, minlength=blk.num_dst).clamp(min=1)
                ref = ref / cnt[:, None]
            (ref * w).sum().backward()
            assert torch.allclose(out, ref, rtol=1e-5, atol=1e-5)
            assert torch.allclose(X.grad, X2.grad, rtol=1e-5, atol=1e-5)
            # the forward is reproducible bit for bit; so is the backward except for source rows whose edges
            # span more than two wavefront ranges (hubs), which are added atomically
            X3 = X.detach().clone().requires_grad_(True)
            out3 = BlockAggregate.apply(blk, X3, mean)
            (out3 * w).sum().backward()
            assert torch.equal(out3, out) and torch.allclose(X3.grad, X.grad, rtol=1e-6, atol=1e-6)
    # a bf16 model: sums are fp32 inside the kernels, results come back in the input's dtype
    X16 = torch.randn(blocks[0].num_src, 32, device=DEV).to(torch.bfloat16).requires_grad_(True)
    out16 = BlockAggregate.apply(blocks[0], X16, True)
    assert out16.dtype == torch.bfloat16
    out16.float().sum().backward()
    assert X16.grad.dtype == torch.bfloat16
    ref16 = BlockAggregate.apply(blocks[0], X16.detach().float(), True)
    assert torch.allclose(out16.float(), ref16, rtol=1e-2, atol=1e-2)


def test_graphconv_matches_dense_statement():
    import apt_amd as npc
    from apt_amd.layers import GraphConv
    _setup_graph(seed=4)
    sampler = npc.MixedPSNeighborSampler(0, 1, [5], "DP", replace=True, rng_seed=6)
    seeds = torch.from_numpy(np.random.default_rng(2).permutation(6000)[:150]).to(DEV)
    _, _, (blk,) = sampler.sample(None, seeds)
    for norm, scale in (("both", 1 / 5.0), ("right", 1 / 5.0), ("left", 1 / 5.0), ("none", 1.0)):
        layer = GraphConv(12, 7, norm=norm).to(DEV)
        feat = torch.randn(blk.num_src, 12, device=DEV, requires_grad=True)
        got = layer(blk, feat)
        h = feat @ layer.weight
        want = torch.zeros(blk.num_dst, 7, device=DEV).index_add(0, blk.col, h[blk.row]) * scale + layer.bias
        assert torch.allclose(got, want, rtol=1e-5, atol=1e-5), norm
        g1, = torch.autograd.grad(got.sum(), feat, retain_graph=True)
        g2, = torch.autograd.grad(want.sum(), feat)
        assert torch.allclose(g1, g2, rtol=1e-5, atol=1e-5), norm


def test_gat_layer_matches_dense_statement():
    import apt_amd as npc
    from apt_amd.layers import GATConv
    _setup_graph(seed=1)
    sampler = npc.MixedPSNeighborSampler(0, 1, [6], "DP", replace=False, rng_seed=5)
    seeds = torch.from_numpy(np.random.default_rng(1).permutation(6000)[:200]).to(DEV)
    _, _, (blk,) = sampler.sample(None, seeds)
    layer = GATConv(16, 8, 3).to(DEV)
    feat = torch.randn(blk.num_src, 16, device=DEV)
    with torch.no_grad():
        got = layer(blk, feat)
        ft = layer.fc(feat).view(-1, 3, 8)
        el, er = (ft * layer.attn_l).sum(-1), (ft[:blk.num_dst] * layer.attn_r).sum(-1)
        e = torch.nn.functional.leaky_relu(el[blk.row] + er[blk.col], 0.2)            # [E, H]
        top = torch.full((blk.num_dst, 3), -1e30, device=DEV).scatter_reduce(0, blk.col[:, None].expand(-1, 3), e, "amax")
        w = torch.exp(e - top[blk.col])
        den = torch.zeros(blk.num_dst, 3, device=DEV).index_add(0, blk.col, w)
        a = w / den[blk.col]
        want = torch.zeros(blk.num_dst, 3, 8, device=DEV).index_add(0, blk.col, a[:, :, None] * ft[blk.row])
        want = want + layer.bias.view(1, 3, 8)
    assert torch.allclose(got, want, rtol=1e-4, atol=1e-5)


def _gat_dense(layer, blk, feat):
    """The layer's textbook statement in plain torch (autograd gives the reference gradients)."""
    H, D = layer.num_heads, layer.out_feats
    ft = layer.fc(feat).view(-1, H, D)
    el, er = (ft * layer.attn_l).sum(-1), (ft[:blk.num_dst] * layer.attn_r).sum(-1)
    e = torch.nn.functional.leaky_relu(el[blk.row] + er[blk.col], layer.negative_slope)
    top = torch.full((blk.num_dst, H), -1e30, device=DEV).scatter_reduce(0, blk.col[:, None].expand(-1, H), e.detach(), "amax")
    w = torch.exp(e - top[blk.col])
    den = torch.zeros(blk.num_dst, H, device=DEV).index_add(0, blk.col, w)
    a = w / den[blk.col]
    out = torch.zeros(blk.num_dst, H, D, device=DEV).index_add(0, blk.col, a[:, :, None] * ft[blk.row])
    return out + layer.bias.view(1, H, D)


@pytest.mark.parametrize("heads,dim,fanout", [(3, 8, 9), (4, 64, 9), (1, 5, 9), (2, 100, 9),      # lane-group kernels
                                              (4, 64, 16), (8, 8, 8), (1, 256, 15), (2, 16, 3)])    # wavefront per destination
def test_gat_layer_gradients(heads, dim, fanout):
    import apt_amd as npc
    from apt_amd.layers import GATConv
    _setup_graph(seed=5)
    sampler = npc.MixedPSNeighborSampler(0, 1, [fanout], "DP", replace=False, rng_seed=8)
    seeds = torch.from_numpy(np.random.default_rng(3).permutation(6000)[:300]).to(DEV)
    _, _, (blk,) = sampler.sample(None, seeds)
    torch.manual_seed(1)
    layer = GATConv(20, dim, heads).to(DEV)
    feat = torch.randn(blk.num_src, 20, device=DEV, requires_grad=True)
    w = torch.randn(blk.num_dst, heads, dim, device=DEV)
    got = layer(blk, feat)
    params = [feat, layer.fc.weight, layer.attn_l, layer.attn_r]
    g_got = torch.autograd.grad((got * w).sum(), params)
    want = _gat_dense(layer, blk, feat)
    g_want = torch.autograd.grad((want * w).sum(), params)
    assert torch.allclose(got, want, rtol=1e-4, atol=1e-5)
    for a, b, name in zip(g_got, g_want, ("feat", "fc", "attn_l", "attn_r")):
        scale = b.abs().max().item() + 1e-12
        assert (a - b).abs().max().item() <= 2e-4 * scale, (name, (a - b).abs().max().item(), scale)


@pytest.mark.parametrize("heads,dim", [(4, 64), (2, 16), (3, 24), (1, 40), (8, 8), (1, 256)])
def test_gat_backward_bf16_matches_fp32_on_rounded_inputs(capi, heads, dim):
    """bf16 features take other kernel variants (8 per lane); on the same (rounded)
    values they must give what the fp32 variants give."""
    rng = np.random.default_rng(heads * 100 + dim)
    n_dst, fanout, n_src = 2000, 11, 9000
    nbr = rng.integers(0, n_src, size=(n_dst, fanout)).astype(np.int64)
    nbr[rng.random(nbr.shape) < 0.2] = -1
    nbr = torch.from_numpy(nbr.reshape(-1)).to(DEV)
    ft16 = torch.randn(n_src, heads, dim, device=DEV).to(torch.bfloat16)
    ft32 = ft16.float()
    el, er = torch.randn(n_src, heads, device=DEV), torch.randn(n_dst, heads, device=DEV)
    d_out = torch.randn(n_dst, heads, dim, device=DEV)
    fmt = capi.block_formats(nbr, n_dst, fanout, n_src, want_csr=False)
    outs = []
    for ft in (ft32, ft16):
        _, attn = capi.gat_block(nbr, n_dst, fanout, ft, el, er, 0.2, want_attn=True)
        outs.append(capi.gat_block_backward(nbr, n_dst, fanout, ft, el, er, 0.2, attn, d_out, fmt["csc_indptr"],
                                            fmt["num_edges"]))
    for a, b in zip(*outs):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5)


def test_sage_trains_on_sampled_batches():
    """Two SAGE layers on sampled blocks + gathered features learn a label that
    depends on the neighbourhood: the loss falls well below its start."""
    import apt_amd as npc
    from apt_amd.layers import SAGEConv
    indptr, indices = _setup_graph(n=4000, deg=10, seed=2)
    n = 4000
    g = torch.Generator().manual_seed(0)
    feats = torch.randn(n, 16, generator=g)
    # label: sign of the mean of feature 0 over the in-neighbours (needs aggregation to predict)
    nb_mean = np.array([feats[indices[indptr[v]:indptr[v + 1]], 0].mean().item() if indptr[v + 1] > indptr[v] else 0.0
                        for v in range(n)])
    labels = torch.from_numpy((nb_mean > 0).astype(np.int64)).to(DEV)
    npc.cache_feats_shared(n, feats, torch.empty(0, 16), torch.empty(0, dtype=torch.int64), torch.arange(n), 0)
    torch.manual_seed(0)
    l1, l2 = SAGEConv(16, 32, activation=torch.relu).to(DEV), SAGEConv(32, 2).to(DEV)
    opt = torch.optim.Adam(list(l1.parameters()) + list(l2.parameters()), lr=0.01)
    sampler = npc.MixedPSNeighborSampler(0, 1, [10, 10], "DP", replace=False, rng_seed=11)
    rng = np.random.default_rng(3)
    losses = []
    for step in range(60):
        seeds = torch.from_numpy(rng.permutation(n)[:256]).to(DEV)
        input_nodes, output_nodes, blocks = sampler.sample(None, seeds)
        x = npc.load_subtensor(input_nodes)
        h = l2(blocks[1], l1(blocks[0], x))
        loss = torch.nn.functional.cross_entropy(h, labels[output_nodes])
        opt.zero_grad()
        loss.backward()
        opt.step()
        losses.append(loss.item())
    assert np.mean(losses[-10:]) < 0.6 * np.mean(losses[:5]), (losses[:5], losses[-10:])


@pytest.mark.parametrize("backend", ["eager", "aot_eager"])
@pytest.mark.parametrize("kind", ["sage", "gcn", "gat", "sage_hooked"])
def test_layers_inside_a_compiled_model(kind, backend):
    """torch.compile breaks its graph around the layers' operators: same outputs and gradients as without it."""
    from apt_amd.layers import GATConv, GraphConv, SAGEConv
    from apt_amd.sampler import Block
    make = dict(sage=SAGEConv, sage_hooked=SAGEConv, gcn=GraphConv, gat=lambda a, b, activation: GATConv(a, b, 1, activation=activation))[kind]
    gen = torch.Generator(device=DEV).manual_seed(7)
    slots = [torch.randint(-1, n, (m * 5,), device=DEV, generator=gen) for n, m in ((900, 300), (300, 40))]
    blocks = [Block(900, 300, None, slots[0], 5), Block(300, 40, None, slots[1], 5)]

    class Model(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.first, self.second = make(16, 32, activation=torch.relu), make(32, 8, activation=None)
            if kind == "sage_hooked":      # the separate operations
                self.first.fc_self.register_forward_hook(lambda module, args, out: out * 2)

        def forward(self, x):
            return self.second(blocks[1], self.first(blocks[0], x).flatten(1) * 0.5).flatten(1)

    torch.manual_seed(5)
    model = Model().to(DEV)
    x = torch.randn(900, 16, device=DEV)
    want = model(x)
    grads = torch.autograd.grad(want.square().sum(), list(model.parameters()))
    torch._dynamo.reset()
    compiled = torch.compile(model, backend=backend)
    got = compiled(x)
    assert torch.allclose(got, want, rtol=1e-6, atol=1e-6)
    for a, b in zip(torch.autograd.grad(got.square().sum(), list(model.parameters())), grads):
        assert torch.allclose(a, b, rtol=1e-5, atol=1e-5)
    with torch.no_grad():
        assert torch.allclose(compiled(x), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("kind", ["aggregate", "aggregate_mean", "sage", "sage_first", "gcn", "gat", "gat_relu"])
@pytest.mark.parametrize("with_csr", [False, True])
def test_gradients_of_gradients(kind, with_csr):
    """A gradient taken with create_graph, squared and differentiated again, against float64: every leaf's first and second
    derivative (fp32 chains of six products and sums of up to a hundred terms: 1e-5 of a result's norm; bound 1e-4)."""
    from apt_amd.layers import BlockAggregate, GATConv, GraphConv, SAGEConv
    from apt_amd.sampler import Block
    gen = torch.Generator(device=DEV).manual_seed(11)
    num_dst, num_src, fanout = 30, 80, 6
    rel = torch.randint(0, num_src, (num_dst * fanout,), device=DEV, generator=gen)
    rel[torch.rand(rel.numel(), device=DEV, generator=gen) < 0.2] = -1
    rel[:fanout] = -1
    blk = Block(num_src, num_dst, None, rel, fanout)
    if with_csr:
        blk.csr()
    keep = (rel >= 0).nonzero().flatten()
    src, dst = rel[keep], keep // fanout
    deg = torch.bincount(dst, minlength=num_dst).clamp(min=1)[:, None].double()
    total = lambda h: torch.zeros(num_dst, h.shape[1], device=DEV, dtype=h.dtype).index_add(0, dst, h[src])  # noqa: E731
    torch.manual_seed(2)
    k, n = (12, 20) if kind != "sage_first" else (20, 12)
    x = torch.randn(num_src, k, device=DEV, generator=gen)
    if kind.startswith("aggregate"):
        layer, mean = torch.nn.Linear(k, n).to(DEV), kind == "aggregate_mean"
        run = lambda: BlockAggregate.apply(blk, layer(leaves[0]), mean)  # noqa: E731
        state = lambda x, w, b: total(x @ w.t() + b) / (deg if mean else 1.0)  # noqa: E731
    elif kind.startswith("sage"):
        layer = SAGEConv(k, n, activation=torch.tanh).to(DEV)
        run = lambda: layer(blk, leaves[0])  # noqa: E731
        state = lambda x, wn, ws, b: torch.tanh(x[:num_dst] @ ws.t() + b + (total(x) / deg) @ wn.t())  # noqa: E731
    elif kind == "gcn":
        layer = GraphConv(k, n, activation=torch.tanh).to(DEV)
        run = lambda: layer(blk, leaves[0])  # noqa: E731
        state = lambda x, w, b: torch.tanh(total(x @ w) / fanout + b)  # noqa: E731
    else:
        layer = GATConv(k, 5, 3, activation=torch.relu if kind == "gat_relu" else None).to(DEV)
        run = lambda: layer(blk, leaves[0])  # noqa: E731

        def state(x, al, ar, b, w):
            ft = (x @ w.t()).view(num_src, 3, 5)
            el, er = (ft * al).sum(-1), (ft[:num_dst] * ar).sum(-1)
            e = torch.exp(torch.nn.functional.leaky_relu(el[src] + er[dst], 0.2))
            den = torch.zeros(num_dst, 3, device=DEV, dtype=e.dtype).index_add(0, dst, e)
            out = torch.zeros(num_dst, 3, 5, device=DEV, dtype=e.dtype).index_add(0, dst, (e / den[dst])[:, :, None] * ft[src])
            out = out + b.view(3, 5)
            return out * (got_out > 0) if kind == "gat_relu" else out
    with torch.no_grad():
        for p in layer.parameters():
            if p.dim() == 1:
                p.normal_()
    names = [name for name, _ in layer.named_parameters()]
    order = {"sage": ["fc_neigh.weight", "fc_self.weight", "fc_self.bias"], "gcn": ["weight", "bias"],
             "gat": ["attn_l", "attn_r", "bias", "fc.weight"], "aggregate": ["weight", "bias"]}[kind.split("_")[0]]
    assert sorted(order) == sorted(names)
    params = dict(layer.named_parameters())
    leaves = [x.requires_grad_(True)] + [params[name] for name in order]
    got_out = run()
    w = torch.randn(got_out.shape, device=DEV, generator=gen)
    exact = [t.detach().double().requires_grad_(True) for t in leaves]
    want_out = state(*exact)
    first = torch.autograd.grad((got_out.square() * w).sum(), leaves, create_graph=True)
    want = torch.autograd.grad((want_out.square() * w.double()).sum(), exact, create_graph=True)
    second = torch.autograd.grad(sum(g.square().sum() for g in first), leaves)
    want2 = torch.autograd.grad(sum(g.square().sum() for g in want), exact)
    for a, b, name in zip(first + second, want + want2, 2 * (["x"] + order)):
        assert (a.double() - b).norm().item() <= 1e-4 * b.norm().item() + 1e-9, name


@pytest.mark.parametrize("kind", ["sage", "sage_first", "gcn", "gat"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_without_edges_whose_csr_was_emitted(kind, dtype):
    """Destinations none of which has a neighbour: the CSR's index arrays are empty, and no gradient crosses the block."""
    from apt_amd.layers import GATConv, GraphConv, SAGEConv
    from apt_amd.sampler import Block
    num_dst, num_src, fanout = 40, 70, 4
    layer = {"sage": lambda: SAGEConv(8, 16), "sage_first": lambda: SAGEConv(16, 8), "gcn": lambda: GraphConv(8, 16),
             "gat": lambda: GATConv(8, 8, 4)}[kind]().to(DEV, dtype)
    x = torch.randn(num_src, 16 if kind == "sage_first" else 8, device=DEV).to(dtype).requires_grad_(True)
    grads = []
    for csr in (False, True):
        blk = Block(num_src, num_dst, None, torch.full((num_dst * fanout,), -1, device=DEV), fanout)
        if csr:
            assert blk.csr()[1].numel() == 0
        out = layer(blk, x)
        grads.append(torch.autograd.grad(out.float().square().sum() + out.float().sum(), [x] + list(layer.parameters())))
    for a, b in zip(*grads):
        assert torch.equal(a, b)
    want = layer.fc_self(x)[:num_dst] if kind.startswith("sage") else layer.bias.view(1, -1).expand(num_dst, -1)
    assert torch.allclose(out.flatten(1).float(), want.float(), rtol=1e-5, atol=1e-6)
    assert bool((grads[0][0][num_dst:] == 0).all())


@pytest.mark.parametrize("kind", ["aggregate", "sage", "sage_first", "gcn", "gat"])
@pytest.mark.parametrize("with_csr", [False, True])
def test_training_on_a_block_made_in_inference_mode(kind, with_csr):
    """Sampling needs no autograd, so a program may do it under torch.inference_mode()."""
    from apt_amd.layers import BlockAggregate, GATConv, GraphConv, SAGEConv
    from apt_amd.sampler import Block
    slots = torch.from_numpy(np.random.default_rng(3).integers(-1, 90, size=30 * 5)).to(DEV)
    torch.manual_seed(4)
    layer = {"aggregate": lambda: torch.nn.Identity(), "sage": lambda: SAGEConv(8, 16), "sage_first": lambda: SAGEConv(8, 4),
             "gcn": lambda: GraphConv(8, 16), "gat": lambda: GATConv(8, 8, 2)}[kind]().to(DEV)
    x = torch.randn(90, 8, device=DEV, requires_grad=True)
    grads = []
    for mode in (False, True):
        with torch.inference_mode(mode):
            blk = Block(90, 30, None, slots.clone(), 5)
            if with_csr:
                blk.csr()
            assert blk.relabeled.is_inference() == mode
        out = BlockAggregate.apply(blk, x, True) if kind == "aggregate" else layer(blk, x)
        grads.append(torch.autograd.grad(out.square().sum(), [x] + list(layer.parameters())))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["sage", "sage_first", "gcn", "gat"])
@pytest.mark.parametrize("change", ["rows", "weights"])
def test_what_no_gradient_needs_may_be_changed_in_place(kind, change):
    """Rows under frozen weights, and weights above rows that need no gradient, between forward and backward: nn.Linear
    keeps neither, and so do the layers."""
    from apt_amd.layers import GATConv, GraphConv, SAGEConv
    from apt_amd.sampler import Block
    blk = Block(90, 30, None, torch.from_numpy(np.random.default_rng(3).integers(-1, 90, size=30 * 5)).to(DEV), 5)
    grads = []
    for touched in (False, True):
        torch.manual_seed(4)
        layer = {"sage": lambda: SAGEConv(8, 16), "sage_first": lambda: SAGEConv(8, 4), "gcn": lambda: GraphConv(8, 16),
                 "gat": lambda: GATConv(8, 8, 2)}[kind]().to(DEV)
        weights = [p for n, p in layer.named_parameters() if n.endswith("weight")]
        leaf = torch.randn(90, 8, device=DEV, requires_grad=change == "rows")
        if change == "rows":
            for p in weights:
                p.requires_grad_(False)
        x = leaf * 1.0
        out = layer(blk, x)
        if touched:
            with torch.no_grad():
                for t in [x] if change == "rows" else weights:
                    t.mul_(3.0)
        wanted = [leaf, layer.bias if kind in ("gcn", "gat") else layer.fc_self.bias] if change == "rows" else weights
        grads.append(torch.autograd.grad((out * torch.linspace(-1, 1, out.numel(), device=DEV).view(out.shape)).sum(), wanted))
    for a, b in zip(*grads):
        assert torch.equal(a, b) and bool((a != 0).any())
