"""Dense products over a block's rows in bf16 against float64: edges of the fragments (16 rows, 32 and 64 columns), steps (32)
and chunks of steps (128) of the depth, both layouts of the weights, odd sizes and addresses, several tiles of columns and
several turns over the rows, and operands whose neighbours in memory are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(got, want, size, k):
    # fp32 sums of k products: at most k 2^-24 of the absolute sum; one rounding to bf16 (2^-9)
    bound = (k + 2) * 2.0 ** -24 * size + 2.0 ** -8 * want.abs()
    assert got.dtype == torch.bfloat16 and bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("m,m2,n,k1,k2", [(1, 1, 1, 1, 1), (17, 0, 31, 33, 0), (129, 65, 65, 100, 100), (300, 300, 47, 256, 256),
                                          (2000, 700, 188, 101, 47), (5000, 5000, 256, 128, 128), (70000, 20000, 256, 64, 50),
                                          (33000, 0, 47, 47, 0), (1000, 1, 600, 300, 20), (4097, 4096, 100, 512, 256), (70001, 3, 10, 16, 3)])
def test_rows_product(capi, m, m2, n, k1, k2, turned):
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).bfloat16()
    weight = lambda k: draw(k, n).t() if turned else draw(n, k)
    x1, w1, bias = draw(m, k1), weight(k1), draw(n)
    x2, w2 = (draw(m2, k2), weight(k2)) if k2 else (None, None)
    want, size = x1.double() @ w1.double().t(), x1.double().abs() @ w1.double().abs().t()
    if k2:
        want[:m2] += x2.double() @ w2.double().t()
        size[:m2] += x2.double().abs() @ w2.double().abs().t()
    _check(capi.rows_gemm(x1, w1, x2, w2), want, size, k1 + k2)
    _check(capi.rows_gemm(x1, w1, x2, w2, bias=bias, relu=True), torch.relu(want + bias.double()), size + bias.double().abs(), k1 + k2)
    y = draw(m, n)
    _check(capi.rows_gemm(x1, w1, x2, w2, out=y.clone()), want + y.double(), size + y.double().abs(), k1 + k2)


@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("k", [50, 47, 96])
def test_rows_product_stays_inside_its_operands(capi, k, turned):
    """Everything around the operands is infinite: rows and weights at odd addresses, weights that are a part of a larger
    matrix, the row behind the second operand's last."""
    n, m, m2 = 40, 200, 77
    hole = lambda *shape: torch.full(shape, float("inf"), device=DEV, dtype=torch.bfloat16)
    gen = torch.Generator(device=DEV).manual_seed(k)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).bfloat16()

    def rows(r):
        base = hole(r * k + 9)
        part = base[3:3 + r * k].view(r, k)
        part.copy_(draw(r, k))
        return part

    def weight():
        base = hole(k + 6, n + 7) if turned else hole(n + 7, k + 6)
        part = base[2:2 + k, 1:1 + n].t() if turned else base[2:2 + n, 1:1 + k]
        part.copy_(draw(n, k))
        return part

    x1, x2, w1, w2 = rows(m), rows(m2), weight(), weight()
    want, size = x1.double() @ w1.double().t(), x1.double().abs() @ w1.double().abs().t()
    want[:m2] += x2.double() @ w2.double().t()
    size[:m2] += x2.double().abs() @ w2.double().abs().t()
    _check(capi.rows_gemm(x1, w1, x2, w2), want, size, 2 * k)
    x1[5, 7], x2[70, 3] = float("inf"), float("nan")      # a row's own stay with it
    got = capi.rows_gemm(x1, w1, x2, w2)
    bad = ~torch.isfinite(got).all(1)
    assert bad[5] and bad[70] and int(bad.sum()) == 2


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("m,m2,n,k", [(200, 77, 40, 48), (200, 77, 40, 47), (2100, 1001, 188, 130), (300, 299, 256, 64)])
def test_rows_product_second_weights_not_finite(capi, m, m2, n, k, turned, bad):
    """The rows behind the second operand's last, in the same fragment of 16, have nothing of its weights."""
    gen = torch.Generator(device=DEV).manual_seed(m + k)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).bfloat16()
    weight = lambda: draw(k, n).t() if turned else draw(n, k)
    x1, x2, w1, w2, bias, y = draw(m, k), draw(m2, k), weight(), weight(), draw(n), draw(m, n)
    w2[n // 2, k - 1], w2[3, 0] = bad, -bad
    want, size = x1.double() @ w1.double().t(), x1.double().abs() @ w1.double().abs().t()
    want[:m2] += x2.double() @ w2.double().t()
    size[:m2] += x2.double().abs() @ w2.double().abs().t()
    for got, ref, total in ((capi.rows_gemm(x1, w1, x2, w2, bias=bias, relu=True), torch.relu(want + bias.double()), size + bias.double().abs()),
                            (capi.rows_gemm(x1, w1, x2, w2, out=y.clone()), want + y.double(), size + y.double().abs())):
        fine = torch.isfinite(ref)
        assert bool(fine[m2:].all()) and int((~fine).sum()) > 0
        assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(got[torch.isinf(got)].double(), ref[torch.isinf(ref)])
        _check(got[fine], ref[fine], total[fine], 2 * k)


@pytest.mark.parametrize("m,k,n", [(19000, 256, 256), (20000, 256, 256), (2000, 333, 970), (3000, 333, 970), (99999, 400, 100), (100000, 400, 100),
                                   (30000, 512, 256), (40000, 129, 256), (70000, 258, 64), (500, 1500, 30)])
def test_products_of_either_kind(m, k, n):
    """A layer's product on both sides of where the resident weights begin to pay, with and without gradients."""
    import apt_amd  # noqa: F401
    gen = torch.Generator(device=DEV).manual_seed(m)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).bfloat16()
    x, w, b = draw(m, k), draw(n, k), draw(n)
    want, size = x.double() @ w.double().t() + b.double(), x.double().abs() @ w.double().abs().t() + b.double().abs()
    with torch.no_grad():
        _check(torch.ops.npc.block_linear(x, w, b, False), want, size, k + 1)
    _check(torch.ops.npc.block_linear(x, w.requires_grad_(True), b, False).detach(), want, size, k + 1)


def test_rows_product_sizes(capi):
    import apt_amd  # noqa: F401  (loads the operators)
    L = capi.lib()
    assert L.apt_rows_product_fits(10, 256, 512, 512) == 1 and L.apt_rows_product_fits(10, 64, 2000, 0) == 0
    assert L.apt_rows_product_fits(10, 0, 5, 0) == 0 and L.apt_rows_product_fits(10, 5, 0, 0) == 0
    # a weight that does not fit takes the library's product
    x, w = torch.randn(50, 2000, device=DEV).bfloat16(), torch.randn(30, 2000, device=DEV).bfloat16()
    assert torch.allclose(torch.ops.npc.block_linear(x, w, None, False).float(), (x.float() @ w.float().t()), rtol=2e-2, atol=0.5)
    assert torch.ops.npc.block_linear(x[:0], w, None, False).shape == (0, 30)
