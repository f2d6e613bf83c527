"""The gradient of a block's sum / mean towards its input (every source row written once): widths at the edges of the
lane groups, rows without edges, rows around the length a group adds up alone (32), hubs, and both edge orders."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _block(num_dst, fanout, num_src, seed):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, num_src, size=num_dst * fanout)
    for s, n in ((0, 32), (1, 33), (2, 64), (3, 65), (4, 700)):          # sources with a given number of edges
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
