"""Dense layers over a block's rows: weight and bias gradients of the library's kernel against float64, at the
edges of its tiles (64 columns), steps (16 / 32 rows), vector widths and splits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (31, 64, 64), (33, 65, 63), (64, 16, 50), (65, 10, 32), (1000, 47, 256),
                                   (4099, 188, 101), (9001, 256, 100), (2500, 320, 514), (70000, 3, 7), (3000, 1030, 700),
                                   (65, 47, 47), (8255, 47, 64), (40001, 130, 333)])
def test_linear_wgrad(capi, m, n, k, dtype):
    gen = torch.Generator(device=DEV).manual_seed(m + n + k)
    dy = torch.randn(m, n, generator=gen, device=DEV).to(dtype)
    x = torch.randn(m, k, generator=gen, device=DEV).to(dtype)
    dw, db = capi.linear_wgrad(dy, x)
    want_w, want_b = dy.double().t() @ x.double(), dy.double().sum(0)
    # fp32 sums of m products of magnitude ~1: error ~ eps * m at the worst, sqrt(m) by chance; bf16 results round at 2^-9
    tol = (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
    for got, want in ((dw, want_w), (db, want_b)):
        bound = tol * want.abs() + 2.0 ** -22 * (m ** 0.5) * 16 + 2.0 ** -22 * want.abs()
        assert got.dtype == dtype and bool(((got.double() - want).abs() <= bound).all())
    again, _ = capi.linear_wgrad(dy, x, want_bias=False)
    assert torch.equal(again, dw)      # a fixed order of the sums


def test_linear_wgrad_unaligned_and_empty(capi):
    base = torch.randn(500 * 64 + 1, device=DEV)
    dy = base[1:].view(500, 64)        # rows start at 4-byte, not 16-byte, addresses
    x = torch.randn(500, 64, device=DEV)
    dw, db = capi.linear_wgrad(dy, x)
    assert torch.allclose(dw.double(), dy.double().t() @ x.double(), atol=1e-3) and torch.allclose(db, dy.sum(0), atol=1e-3)
    dw, db = capi.linear_wgrad(torch.empty(0, 5, device=DEV), torch.empty(0, 7, device=DEV))
    assert dw.shape == (5, 7) and not dw.any() and not db.any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kn", [False, True])
def test_block_linear_gradients(dtype, kn):
    import apt_amd  # noqa: F401  (loads the operators)
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(777, 40, generator=gen, device=DEV).to(dtype).requires_grad_(True)
    w = torch.randn((40, 24) if kn else (24, 40), generator=gen, device=DEV).to(dtype).requires_grad_(True)
    b = None if kn else torch.randn(24, generator=gen, device=DEV).to(dtype).requires_grad_(True)
    up = torch.randn(777, 24, generator=gen, device=DEV).to(dtype)
    params = [x, w] + ([] if b is None else [b])
    y = torch.ops.npc.block_linear(x, w, b, kn)
    plain = x @ w if kn else torch.nn.functional.linear(x, w, b)
    # 40 products of magnitude ~1: an fp32 sum is off by a few 2^-24 of their absolute sum; bf16 results round at 2^-9
    want = x.detach().double() @ (w.detach().double() if kn else w.detach().double().t()) + (0 if b is None else b.detach().double())
    bound = (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) * want.abs() + 2.0 ** -22 * 40
    assert y.dtype == dtype and bool(((y.double() - want).abs() <= bound).all())
    got = torch.autograd.grad(y, params, up)
    want = torch.autograd.grad(plain, params, up)
    for g, r in zip(got, want):
        assert g.dtype == r.dtype and torch.allclose(g.float(), r.float(), rtol=2e-2 if dtype == torch.bfloat16 else 1e-5,
                                                     atol=(0.3 if dtype == torch.bfloat16 else 1e-3))
    # gradients of gradients still have a graph
    y = torch.ops.npc.block_linear(x, w, b, kn)
    gw, = torch.autograd.grad(y.float().square().sum(), w, create_graph=True)
    gx, = torch.autograd.grad(gw.float().sum(), x)
    assert gx.shape == x.shape and bool(torch.isfinite(gx).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,m2,n,k,k2", [(1, 1, 1, 1, 1), (129, 65, 65, 129, 64), (6000, 6000, 256, 100, 100), (4097, 900, 47, 256, 256),
                                         (9000, 257, 130, 0, 70), (40000, 40000, 96, 101, 33), (300, 0, 20, 12, 7)])
def test_two_weight_gradients_in_one_launch(capi, m, m2, n, k, k2, dtype):
    """Products of different rows and columns, column sums alone (k = 0), the mask of a ReLU with NaN, infinite and zero
    results, and the edges of both tiles (64, 128) and of a split."""
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    draw = lambda r, c: torch.randn(r, c, generator=gen, device=DEV).to(dtype)
    dy, x, relu = draw(m, n), draw(m, k) if k else None, torch.relu(draw(m, n))
    relu.view(-1)[:3:2] = torch.tensor([float("nan"), float("inf")], device=DEV, dtype=dtype)[:relu.view(-1)[:3:2].numel()]
    dy2, x2 = draw(m2, n + 3), draw(m2, k2)
    (dw, db), (dw2, db2) = capi.linear_wgrads([(dy, x, relu, True), (dy2, x2, None, False)])
    live = torch.where(relu <= 0, torch.zeros_like(dy), dy).double()      # (a NaN passes, as in torch)
    # as in test_linear_wgrad: fp32 sums of m products of magnitude ~1, bf16 results round at 2^-9
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    for got, want, rows in ((dw, None if x is None else live.t() @ x.double(), m), (db, live.sum(0), m),
                            (dw2, dy2.double().t() @ x2.double(), m2)):
        if want is None:
            assert got is None
            continue
        bound = tol * want.abs() + 2.0 ** -22 * (rows ** 0.5) * 16 + 2.0 ** -22 * want.abs()
        assert got.dtype == dtype and bool(((got.double() - want).abs() <= bound).all())
    assert db2 is None


def test_weight_gradient_of_infinite_rows(capi):
    """The parts of an infinity are NaN: the tile is formed again in fp32, and gives what fp32 gives."""
    dy, x = torch.randn(500, 70, device=DEV), torch.randn(500, 80, device=DEV)
    dy[77, 3], x[401, 5], relu = float("inf"), float("-inf"), torch.ones(500, 70, device=DEV)
    relu[401] = 0
    (dw, db), = capi.linear_wgrads([(dy, x, relu, True)])
    live = torch.where(relu <= 0, torch.zeros_like(dy), dy)
    want = live.double().t() @ x.double()     # (0 * inf: NaN, in column 5 and in row 3 where x is not)
    assert torch.equal(dw.isnan(), want.isnan()) and torch.equal(dw.isinf(), want.isinf())
    ok = want.isfinite()
    assert torch.allclose(dw[ok].double(), want[ok], atol=2.0 ** -22 * 500 ** 0.5 * 16) and db[3].isinf()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bias", [False, True])
def test_block_linear_without_columns(dtype, bias):
    """A weight [3, 0]: the product is the bias, its gradients are empty and the column sums."""
    import apt_amd  # noqa: F401
    x, w = torch.zeros(5, 0, device=DEV, dtype=dtype, requires_grad=True), torch.zeros(3, 0, device=DEV, dtype=dtype, requires_grad=True)
    b = torch.tensor([1.0, 2.0, 3.0], device=DEV, dtype=dtype, requires_grad=True) if bias else None
    y = torch.ops.npc.block_linear(x, w, b, False)
    assert torch.equal(y, b.expand(5, 3) if bias else torch.zeros_like(y))
    got = torch.autograd.grad(y, [x, w] + ([b] if bias else []), torch.full_like(y, 2.0))
    assert got[0].shape == (5, 0) and got[1].shape == (3, 0) and (not bias or got[2].tolist() == [10.0, 10.0, 10.0])


@pytest.mark.parametrize("m", [1, 7, 63, 64, 65, 127, 129, 1000, 8193])
@pytest.mark.parametrize("n,k", [(47, 31), (64, 47), (47, 64), (5, 66), (130, 101)])
def test_linear_wgrad_between_what_is_not_finite(capi, m, n, k):
    """bf16 rows of odd lengths and addresses: what shares a dword with their first and their last element is infinite, as is
    what shares one with the ReLU's result."""
    gen = torch.Generator(device=DEV).manual_seed(m + n)

    def rows(cols, shift):
        base = torch.full((m * cols + 8,), float("inf"), device=DEV, dtype=torch.bfloat16)
        part = base[shift:shift + m * cols].view(m, cols)
        part.copy_(torch.randn(m, cols, generator=gen, device=DEV).bfloat16())
        return part

    for shift in (0, 1, 3):
        dy, x, y = rows(n, shift), rows(k, 4 - shift), rows(n, 1 if shift else 2)
        for mask in (None, y):
            (dw, db), = capi.linear_wgrads([(dy, x, mask, True)])
            g = dy.double() if mask is None else torch.where(y.double() > 0, dy.double(), 0.0)
            want, size = g.t() @ x.double(), g.abs().t() @ x.double().abs()
            # fp32 sums of m products, one rounding to bf16
            assert bool(((dw.double() - want).abs() <= (m + 2) * 2.0 ** -24 * size + 2.0 ** -8 * want.abs()).all())
            assert bool(((db.double() - g.sum(0)).abs() <= (m + 2) * 2.0 ** -24 * g.abs().sum(0) + 2.0 ** -8 * g.sum(0).abs()).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [((20000, 256, 600), (3000, 256, 600)), ((500, 64, 64), (90000, 48, 60)), ((64, 300, 1000), (64, 300, 1000)),
                                   ((5000, 256, 0), (30000, 200, 130))])
def test_linear_wgrads_of_different_lengths(capi, sizes, dtype):
    """Two products whose rows are split into different numbers of parts, and more tiles than workgroups."""
    gen = torch.Generator(device=DEV).manual_seed(5)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).to(dtype)  # noqa: E731
    products = [(draw(m, n), draw(m, k) if k else None, None, True) for m, n, k in sizes]
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    for (dw, db), (dy, x, _, _) in zip(capi.linear_wgrads(products), products):
        a, m = dy.double(), dy.shape[0]
        if x is not None:
            want, size = a.t() @ x.double(), a.abs().t() @ x.double().abs()
            assert bool(((dw.double() - want).abs() <= (m / 32 + 40) * 2.0 ** -24 * size + half * want.abs()).all())
        assert bool(((db.double() - a.sum(0)).abs() <= (m / 8 + 8) * 2.0 ** -24 * a.abs().sum(0) + half * a.sum(0).abs()).all())


@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("sizes", [((16411, 33, 4090),), ((16411, 4100, 17),), ((131073, 64, 470), (1000, 3, 65)), ((131073, 470, 64), (77, 65, 1)),
                                   ((131073, 470, 50), (9000, 470, 0)), ((262144, 129, 1),), ((262143, 1, 130),)])
def test_linear_wgrads_of_oblong_tiles(capi, sizes, mask):
    """Long blocks of which one side is at most 64 wide: tiles of 128 x 64 and 64 x 128.  With an infinite element the tiles it
    reaches are formed again in fp32."""
    gen = torch.Generator(device=DEV).manual_seed(9)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV)  # noqa: E731
    for infinite in (False, True):
        products = [(draw(m, n), draw(m, k) if k else None, draw(m, n) if mask else None, True) for m, n, k in sizes]
        if infinite:
            products[0][1][100, 0], products[0][0][100, 0] = float("inf"), 0.5
            if mask:
                products[0][2][100, 0] = 1.0
        for (dw, db), (dy, x, y, _) in zip(capi.linear_wgrads(products), products):
            a, m = dy.double() if y is None else torch.where(y > 0, dy, torch.zeros_like(dy)).double(), dy.shape[0]
            if x is not None:
                # a workgroup's rows (an LDS step of 32 at a time, or one by one) and the partials, each rounded once
                want, size = a.t() @ x.double(), a.abs().t() @ x.double().abs()
                ok = want.isfinite()
                assert torch.equal(dw.isnan(), want.isnan()) and torch.equal(dw.isinf(), want.isinf()) and bool((~ok).any()) == (infinite and x is products[0][1])
                assert bool(((dw.double() - want).abs() <= (m / 32 + 40) * 2.0 ** -24 * size + 2.0 ** -23 * want.abs())[ok].all())
            assert bool(((db.double() - a.sum(0)).abs() <= (m / 8 + 8) * 2.0 ** -24 * a.abs().sum(0) + 2.0 ** -23 * a.sum(0).abs()).all())
