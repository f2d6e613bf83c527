"""The fp32 product of a layer's rows (one or two operand pairs) against float64: the edges of its tiles (16 / 64 rows and
columns), steps (32), vector widths and workgroup shapes, rows without the second operand, and values that are not
finite, whose bf16 parts would be NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV)


@pytest.mark.parametrize("m,m2,n,k1,k2", [(1, 0, 1, 1, 0), (17, 17, 47, 32, 1), (65, 40, 64, 33, 31), (1000, 1, 65, 100, 100),
                                          (1023, 64, 128, 4, 64), (2049, 2049, 129, 101, 3), (5000, 333, 256, 256, 256),
                                          (40001, 9000, 257, 12, 20), (70001, 70001, 47, 64, 4), (33000, 0, 100, 50, 0),
                                          (300, 200, 600, 512, 40), (40000, 77, 50, 50, 20), (40000, 40000, 100, 64, 0),
                                          (53000, 52990, 300, 90, 20), (32769, 5, 1000, 70, 20)])
@pytest.mark.parametrize("transposed,accumulate", [(False, False), (True, True)])
def test_rows_gemm(capi, m, m2, n, k1, k2, transposed, accumulate):
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    x1, w1, b = _rand(gen, m, k1), _rand(gen, n, k1), _rand(gen, n)
    x2, w2 = (_rand(gen, m2, k2), _rand(gen, n, k2)) if k2 else (None, None)
    base = _rand(gen, m, n) if accumulate else None
    at = [None if w is None else w.t().contiguous().t() if transposed else w for w in (w1, w2)]
    got = capi.rows_gemm(x1, at[0], x2, at[1], b, None if base is None else base.clone())
    want = x1.double() @ w1.double().t() + b.double() + (0 if base is None else base.double())
    size = x1.double().abs() @ w1.double().abs().t() + b.double().abs() + 1
    if k2:
        want[:m2] += x2.double() @ w2.double().t()
        size[:m2] += x2.double().abs() @ w2.double().abs().t()
    # parts left out: below 2^-24 of a product; roundings at 2^-24: one per step of 32 and the partial sums of one step
    steps = (k1 + k2 + 31) // 32
    bound = size * 2.0 ** -24 * (8 + steps)
    assert bool(((got.double() - want).abs() <= bound).all())
    assert torch.equal(got, capi.rows_gemm(x1, at[0], x2, at[1], b, base))


# five steps of depth; four or fewer in the kernel with resident weights, by 32, 64 and 128 columns (200 of 256, of the fewest
# rows that take it: two turns of the CUs, or a good part of one)
@pytest.mark.parametrize("m,m2,n,k1", [(500, 203, 70, 100), (500, 203, 70, 101), (500, 203, 20, 50), (40000, 203, 60, 50),
                                       (40000, 39999, 100, 51), (53000, 1003, 200, 96), (53000, 20, 256, 20)])
def test_rows_gemm_not_finite(capi, m, m2, n, k1):
    gen = torch.Generator(device=DEV).manual_seed(3)
    x1, w1, x2, w2 = _rand(gen, m, k1), _rand(gen, n, k1), _rand(gen, m2, 8), _rand(gen, n, 8)
    x1[3, 5], x1[7, 2], w1[10, 1], w2[n - 9, 3] = float("inf"), float("nan"), float("-inf"), float("inf")
    x1[9] = 0
    x1[9, 0] = torch.finfo(torch.float32).max            # rounds to an infinity in bf16
    w1[:, 0] = 1
    w2[:, :] = torch.where(torch.isinf(w2), w2, w2 * 1e-3)
    got = capi.rows_gemm(x1, w1, x2, w2)
    want = x1.double() @ w1.double().t()
    want[:m2] += x2.double() @ w2.double().t()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)].double(), want[torch.isinf(want)])
    fine = torch.isfinite(want)
    assert bool((got.double() - want)[fine].abs().le(1e-4 + 1e-6 * want[fine].abs()).all())


@pytest.mark.parametrize("scale", [1e-30, 1e15])
def test_rows_gemm_range(capi, scale):
    gen = torch.Generator(device=DEV).manual_seed(5)
    x, w = _rand(gen, 300, 200) * scale, _rand(gen, 50, 200)
    want = x.double() @ w.double().t()
    err = (capi.rows_gemm(x, w).double() - want).norm() / want.norm()
    assert float(err) < 2e-7
