"""The COO sums of the operators (spmm_copy_u / copy_e / u_mul_e) with edges in any order, in segments, with rows out of
range, and the per-edge combine, against float64 torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _edges(E, n_in, n_out, order, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    row = torch.randint(0, n_in, (E,), generator=gen, device=DEV)
    col = (torch.rand(E, generator=gen, device=DEV) ** 3 * n_out).long()      # some rows with many edges, some with none
    if order == "grouped":
        col = col.sort().values
    return row, col


def _sum(key, x, n_out, ok):
    out = torch.zeros(n_out, x.shape[1], device=DEV, dtype=torch.float64)
    return out.index_add(0, key[ok], x[ok]), torch.zeros_like(out).index_add(0, key[ok], x[ok].abs())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("order", ["grouped", "any"])
@pytest.mark.parametrize("E,n_in,n_out,dim", [(1, 1, 1, 1), (5000, 700, 900, 47), (20000, 3000, 70, 100), (3000, 500, 100000, 8),
                                              (9000, 2000, 1500, 256), (60000, 3000, 900, 41), (40000, 3000, 70, 100),
                                              (300000, 500, 200000, 8), (0, 4, 6, 16)])
def test_spmm_operators(E, n_in, n_out, dim, order, dtype):
    import apt_amd as npc
    row, col = _edges(E, n_in, n_out, order, E + dim)
    if E > 100 and order == "any":
        col[5], row[7], row[9] = n_out + 3, n_in, -1                        # not rows of these tensors: left out
    gen = torch.Generator(device=DEV).manual_seed(dim)
    x = torch.randn(n_in, dim, generator=gen, device=DEV).to(dtype)
    ed = torch.randn(E, dim, generator=gen, device=DEV).to(dtype)
    i64 = lambda *v: torch.tensor(v, dtype=torch.int64, device=DEV)
    coo, zero, out_off = i64(0, E), i64(0), i64(0, n_out)
    ok_col = (col >= 0) & (col < n_out)
    ok = ok_col & (row >= 0) & (row < n_in)
    src = x.double()[row.clamp(0, n_in - 1)] if E else torch.zeros(0, dim, device=DEV, dtype=torch.float64)
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22
    for got, term, good in ((npc.ops.spmm_copy_u_sum(row, col, x, coo, zero, out_off), src, ok),
                            (npc.ops.spmm_copy_e_sum(row, col, ed, coo, out_off), ed.double(), ok_col),
                            (npc.ops.spmm_u_mul_e_sum(row, col, x, ed, coo, zero, out_off), src * ed.double(), ok)):
        want, size = _sum(col, term, n_out, good)
        assert got.dtype == dtype and got.shape == (n_out, dim)
        assert bool(((got.double() - want).abs() <= 2e-6 * size + half * want.abs() + 1e-30).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("order", ["grouped", "any"])
@pytest.mark.parametrize("E,n_out,dim", [(40000, 1, 64), (40000, 8, 64), (33000, 64, 64), (300000, 64, 8), (300000, 1, 8), (70000, 137, 33),
                                         (9000, 3, 256)])
def test_spmm_of_few_rows(E, n_out, dim, order, dtype):
    """A readout: every row has hundreds to hundreds of thousands of edges."""
    import apt_amd as npc
    assert E * dim > 2 ** 21      # (fewer are added up edge by edge)
    gen = torch.Generator(device=DEV).manual_seed(E + dim)
    row = torch.randint(0, 5000, (E,), generator=gen, device=DEV)
    col = torch.randint(0, n_out, (E,), generator=gen, device=DEV)
    if order == "grouped":
        col = col.sort().values
    x = torch.randn(5000, dim, generator=gen, device=DEV).to(dtype)
    ed = torch.randn(E, dim, generator=gen, device=DEV).to(dtype)
    i64 = lambda *v: torch.tensor(v, dtype=torch.int64, device=DEV)  # noqa: E731
    coo, zero, out_off = i64(0, E), i64(0), i64(0, n_out)
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22
    pick, src = (torch.arange(n_out, device=DEV)[:, None] == col).double(), x.double()[row]
    for run, term in ((lambda: npc.ops.spmm_copy_u_sum(row, col, x, coo, zero, out_off), src),
                      (lambda: npc.ops.spmm_copy_e_sum(row, col, ed, coo, out_off), ed.double()),
                      (lambda: npc.ops.spmm_u_mul_e_sum(row, col, x, ed, coo, zero, out_off), src * ed.double())):
        want, size = pick @ term, pick @ term.abs()
        got = run()
        assert bool(((got.double() - want).abs() <= 2e-6 * size + half * want.abs()).all())
        assert torch.equal(got, run())


def test_spmm_into_few_rows_takes_no_longer_than_into_many():
    """1 M edges of 64 fp32: into 1 row 11.7 ms, into 8 16 ms, where one workgroup added a row up; into 100 k rows 91 us."""
    import apt_amd as npc
    E, dim = 1_000_000, 64
    row = torch.randint(0, 100_000, (E,), device=DEV)
    x = torch.randn(100_000, dim, device=DEV)
    i64 = lambda *v: torch.tensor(v, dtype=torch.int64, device=DEV)  # noqa: E731

    def fastest(n_out):
        col = torch.randint(0, n_out, (E,), device=DEV)
        coo, zero, out_off, times = i64(0, E), i64(0), i64(0, n_out), []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            npc.ops.spmm_copy_u_sum(row, col, x, coo, zero, out_off)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    many = fastest(100_000)
    assert fastest(1) <= 6 * many and fastest(8) <= 6 * many and fastest(64) <= 6 * many


def test_spmm_segments_and_shared_rows():
    import apt_amd as npc
    E, dim = 4000, 24
    gen = torch.Generator(device=DEV).manual_seed(3)
    row = torch.randint(0, 100, (E,), generator=gen, device=DEV)
    col = torch.randint(0, 50, (E,), generator=gen, device=DEV)
    x = torch.randn(300, dim, generator=gen, device=DEV)
    i64 = lambda *v: torch.tensor(v, dtype=torch.int64, device=DEV)
    coo, x_off, out_off = i64(0, 1500, 1500, E), i64(0, 100, 200), i64(0, 25, 60, 110)   # segments share output rows
    seg = (torch.arange(E, device=DEV) >= 1500).long() * 2
    want = torch.zeros(110, dim, device=DEV, dtype=torch.float64).index_add(0, out_off[seg] + col, x.double()[x_off[seg] + row])
    got = npc.ops.spmm_copy_u_sum(row, col, x, coo, x_off, out_off)
    assert got.shape == (110, dim) and torch.allclose(got.double(), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,dim", [(1, 1), (777, 3), (777, 4), (5000, 100), (300, 41)])
def test_sddmm_operators(E, dim, dtype):
    import apt_amd as npc
    row, col = _edges(E, 300, 200, "any", E)
    gen = torch.Generator(device=DEV).manual_seed(dim)
    a, b = torch.randn(300, dim, generator=gen, device=DEV).to(dtype), torch.randn(200, dim, generator=gen, device=DEV).to(dtype)
    i64 = lambda *v: torch.tensor(v, dtype=torch.int64, device=DEV)
    coo, zero = i64(0, E), i64(0)
    assert torch.equal(npc.ops.sddmm_u_add_v(row, col, a, b, coo, zero, zero), (a.float()[row] + b.float()[col]).to(dtype))
    assert torch.equal(npc.ops.sddmm_u_mul_v(row, col, a, b, coo, zero, zero), (a.float()[row] * b.float()[col]).to(dtype))
