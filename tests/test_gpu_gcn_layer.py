"""The GCN layer as one operator against its statement in float64 (forward and every gradient), and the ReLU that the three
layers' kernels apply against one applied to their results."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _slots(num_dst, fanout, num_src, seed):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    r[rng.random(r.size) < 0.2] = -1
    return torch.from_numpy(r.astype(np.int64)).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("num_dst,fanout,num_src,k,n", [(1, 1, 1, 1, 1), (300, 5, 900, 100, 256), (700, 15, 700, 33, 47),
                                                        (64, 10, 5000, 128, 32), (0, 3, 20, 8, 4)])
@pytest.mark.parametrize("bias,with_csr,relu", [(True, False, True), (False, True, False)])
def test_gcn_layer(capi, num_dst, fanout, num_src, k, n, dtype, bias, with_csr, relu):
    import apt_amd  # noqa: F401  (loads the operators)
    rel = _slots(num_dst, fanout, num_src, k)
    gen = torch.Generator(device=DEV).manual_seed(k)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(dtype).requires_grad_(True)  # noqa: E731
    leaves = [rand(num_src, k), rand(k, n)] + ([rand(n)] if bias else [])
    up = torch.randn(num_dst, n, generator=gen, device=DEV).to(dtype)
    f = capi.block_formats(rel, num_dst, fanout, num_src) if with_csr and num_dst else {}
    scale = 0.3
    out = torch.ops.npc.gcn_layer(rel, num_dst, fanout, leaves[0], leaves[1], leaves[2] if bias else None, 0.5, 0.6,
                                  f.get("csr_indptr"), f.get("csr_indices"), relu)
    got = torch.autograd.grad(out, leaves, up)
    exact = [t.detach().double().requires_grad_(True) for t in leaves]
    keep = (rel >= 0).nonzero().flatten()
    h = exact[0] @ exact[1]
    want = scale * torch.zeros(num_dst, n, device=DEV, dtype=torch.float64).index_add(0, keep // fanout, h[rel[keep]])
    if bias:
        want = want + exact[2]
    # fp32: results within rounding of zero may fall on either side of the ReLU: the mask is the operator's own.
    # bf16: up to four roundings at 2^-9 on the way to a result
    want = want * (out > 0) if relu else want
    grads = torch.autograd.grad(want, exact, up.double())
    rel_err = 2e-6 if dtype == torch.float32 else 1.2e-2
    for a, b in zip((out,) + got, (want,) + grads):
        assert a.dtype == dtype and a.shape == b.shape
        assert bool((a.double() - b).norm() <= rel_err * b.norm() + 1e-30)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["sage", "sage_first", "gcn", "gat", "gat_any"])
def test_relu_in_the_kernels(kind, dtype):
    from apt_amd.layers import GATConv, GraphConv, SAGEConv
    from apt_amd.sampler import Block
    block = Block(500, 120, None, _slots(120, 7, 500, 3), 7)
    torch.manual_seed(4)
    make = {"sage": lambda a: SAGEConv(24, 33, activation=a), "sage_first": lambda a: SAGEConv(33, 24, activation=a),
            "gcn": lambda a: GraphConv(24, 16, activation=a), "gat": lambda a: GATConv(24, 16, 4, activation=a),
            "gat_any": lambda a: GATConv(24, 5, 3, activation=a)}[kind]
    inside, apart = make(torch.relu).to(DEV, dtype), make(lambda h: torch.relu(h)).to(DEV, dtype)
    apart.load_state_dict(inside.state_dict())
    x = torch.randn(500, inside.state_dict()["weight"].shape[0] if kind == "gcn" else 33 if kind == "sage_first" else 24,
                    device=DEV).to(dtype)
    for layer in (inside, apart):
        layer.x = x.clone().requires_grad_(True)
        layer.out = layer(block, layer.x)
        (layer.out.float() * torch.linspace(-1, 1, layer.out.numel(), device=DEV).view(layer.out.shape)).sum().backward()
    assert bool((inside.out == 0).any()) and bool((inside.out > 0).any())
    assert torch.equal(inside.out, apart.out) and torch.equal(inside.x.grad, apart.x.grad)
    for p, q in zip(inside.parameters(), apart.parameters()):
        assert torch.equal(p.grad, q.grad)
