"""COO / CSC / CSR emission of a sampled block: oracle pins (no GPU) and GPU parity."""
import numpy as np
import pytest


def _random_block(rng, num_dst, fanout, num_src, hole=0.3, hub=True):
    """Fixed-stride block with -1 holes (anywhere in a row, not only at its end)."""
    r = rng.integers(0, max(num_src, 1), size=num_dst * fanout)
    if hub and num_src > 3:
        r[rng.random(r.size) < 0.2] = 3                      # one source on a fifth of all edges
    r[rng.random(r.size) < hole] = -1
    if num_src == 0:
        r[:] = -1
    return r.astype(np.int64)


def _closed_form(r, num_dst, fanout, num_src):
    keep = np.nonzero(r >= 0)[0]
    row, col = r[keep], keep // max(fanout, 1)
    order = np.argsort(row, kind="stable")
    return dict(num_edges=len(keep), coo_row=row, coo_col=col,
                csc_indptr=np.concatenate([[0], np.cumsum(np.bincount(col, minlength=num_dst))]),
                csr_indptr=np.concatenate([[0], np.cumsum(np.bincount(row, minlength=num_src))]),
                csr_indices=col[order], csr_eids=order)


def _same(a, b, keys=("coo_row", "coo_col", "csc_indptr", "csr_indptr", "csr_indices", "csr_eids")):
    assert a["num_edges"] == b["num_edges"]
    for k in keys:
        assert np.array_equal(np.asarray(a[k]), np.asarray(b[k])), k


CASES = [(0, 5, 0), (1, 1, 1), (7, 3, 5), (100, 10, 37), (1000, 15, 5000), (257, 16, 70000), (64, 0, 10)]


def test_oracle_block_formats_closed_form(orc):
    rng = np.random.default_rng(0)
    for num_dst, fanout, num_src in CASES:
        r = _random_block(rng, num_dst, fanout, num_src)
        _same(orc.block_formats(r, num_dst, fanout, num_src), _closed_form(r, num_dst, fanout, num_src))
    # scipy agrees on the offsets and on the neighbour sets of a duplicate-free block
    import scipy.sparse as sp
    num_dst, fanout, num_src = 50, 4, 400
    r = rng.permutation(num_src)[:num_dst * fanout].astype(np.int64)
    got = orc.block_formats(r, num_dst, fanout, num_src)
    m = sp.coo_matrix((np.arange(got["num_edges"]) + 1, (got["coo_row"], got["coo_col"])), shape=(num_src, num_dst))
    csr, csc = m.tocsr(), m.tocsc()
    assert np.array_equal(csr.indptr, got["csr_indptr"]) and np.array_equal(csc.indptr, got["csc_indptr"])
    assert np.array_equal(csr.indices, got["csr_indices"]) and np.array_equal(csr.data - 1, got["csr_eids"])
    assert np.array_equal(csc.indices, got["coo_row"][csc.data - 1])          # scipy orders a column by source
    assert np.array_equal(np.sort((csc.data - 1).reshape(num_dst, fanout), axis=1),
                          np.arange(num_dst * fanout).reshape(num_dst, fanout))


@pytest.mark.gpu
def test_gpu_block_formats(orc, capi):
    import torch
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    host = lambda d: {k: (v.cpu().numpy() if hasattr(v, "cpu") else v) for k, v in d.items()}
    rng = np.random.default_rng(1)
    big = [(70000, 15, 300000), (5000, 64, 2 ** 24 + 5), (300000, 5, 17),      # 3 / 4 / 1 digit passes
           (10, 2, 3_000_000), (1, 1, 70_000)]                                # a few edges, sources far apart
    for num_dst, fanout, num_src in CASES + big:
        for hole in (0.0, 0.3, 1.0):
            r = _random_block(rng, num_dst, fanout, num_src, hole)
            want = orc.block_formats(r, num_dst, fanout, num_src)
            got = host(capi.block_formats(dev(r) if r.size else torch.empty(0, dtype=torch.int64, device="cuda:0"),
                                          num_dst, fanout, num_src))
            _same(got, want)
    # the scan launches that large inputs take, forced on small ones; then two inputs large enough by themselves
    capi.check(capi.lib().apt_set_tuning(b"block_fused_scan", 0))
    try:
        for num_dst, fanout, num_src in [(7, 3, 5), (70000, 15, 300000), (5000, 64, 2 ** 24 + 5)]:
            r = _random_block(rng, num_dst, fanout, num_src)
            _same(host(capi.block_formats(dev(r), num_dst, fanout, num_src)), orc.block_formats(r, num_dst, fanout, num_src))
    finally:
        capi.check(capi.lib().apt_set_tuning(b"block_fused_scan", 1))
    for num_dst, fanout, num_src in [(600000, 15, 3000000), (1200000, 15, 70000)]:
        r = _random_block(rng, num_dst, fanout, num_src)
        _same(host(capi.block_formats(dev(r), num_dst, fanout, num_src)), orc.block_formats(r, num_dst, fanout, num_src))
    # no CSR asked for
    r = _random_block(rng, 1000, 7, 900)
    got = host(capi.block_formats(dev(r), 1000, 7, 900, want_csr=False))
    _same(got, orc.block_formats(r, 1000, 7, 900), keys=("coo_row", "coo_col", "csc_indptr"))
    # device-side destination count: buffers at the upper bound, rows past the count are empty
    num_dst, fanout, num_src = 20000, 10, 50000
    r = _random_block(rng, num_dst, fanout, num_src)
    fmt = capi.BlockFormats(num_dst, fanout, num_src)
    for real in (20000, 12345, 1, 0):                        # reuse of the buffers, shrinking
        cnt = torch.tensor([real], dtype=torch.int64, device="cuda:0")
        fmt.emit(dev(r), cnt)
        want = orc.block_formats(r[:real * fanout], real, fanout, num_src)
        e = want["num_edges"]
        assert int(fmt.num_edges.item()) == e
        assert np.array_equal(fmt.csc_indptr.cpu().numpy(), np.concatenate([want["csc_indptr"], np.full(num_dst - real, e)]))
        assert np.array_equal(fmt.csr_indptr.cpu().numpy(), want["csr_indptr"])
        _same(host(fmt.narrow(num_dst=real)), want)


@pytest.mark.gpu
def test_gpu_pipeline_blocks_in_all_formats(orc, capi):
    """The fused driver's blocks, emitted with device-side sizes, equal the
    oracle's formats of the oracle's blocks."""
    import torch
    from helpers import small_graph
    from apt_amd.pipeline import MiniBatchPipeline
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    indptr, indices = small_graph(20000, 6, seed=3)
    feats = torch.randn(20000, 32, device="cuda:0")
    graph = capi.Graph(dev(indptr), dev(indices))
    rng = np.random.default_rng(5)
    for use_graph, what in ((False, True), (True, True), (False, "csc"), (True, "csc")):
        pipe = MiniBatchPipeline(graph, capi.FeatStore(feats), 256, [4, 8, 12], formats=what, use_graph=use_graph)
        for key in (77, 78, 79):                              # buffers and streams are reused batch after batch
            seeds = rng.permutation(20000)[:256]
            pipe.run(dev(seeds), key)
            res = pipe.result()
            inp, blocks = orc.sample_blocks(orc.Graph(indptr, indices), seeds, [4, 8, 12], False, key)
            assert len(res["blocks"]) == 3
            assert torch.equal(res["features"], feats[torch.from_numpy(inp).to("cuda:0")])
            for got, want in zip(res["blocks"], blocks):
                f = got["formats"]
                num_dst, num_src = len(want["seeds"]), len(want["unique"])
                ref = orc.block_formats(want["relabeled"], num_dst, want["fanout"], num_src)
                assert f["csc_indptr"].numel() == num_dst + 1
                if what == "csc":
                    assert "csr_indptr" not in f
                    _same({k: (v.cpu().numpy() if hasattr(v, "cpu") else v) for k, v in f.items()}, ref,
                          keys=("coo_row", "coo_col", "csc_indptr"))
                    continue
                assert f["csr_indptr"].numel() == num_src + 1
                _same({k: (v.cpu().numpy() if hasattr(v, "cpu") else v) for k, v in f.items()}, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("num_dst,fanout,num_src", [
    (3000, 7, 32767), (3000, 7, 32768), (3000, 7, 32769),               # the first piece of source ranges ends at 2^15
    (3000, 7, 2 ** 18 - 1), (3000, 7, 2 ** 18), (3000, 7, 2 ** 18 + 1),  # the second at 2^18
    (2000, 3, 2 ** 18 + 2600 * 1024 - 1), (2000, 3, 2 ** 18 + 2600 * 1024), (2000, 3, 2 ** 18 + 2600 * 2048 - 1),
    (2000, 3, 2 ** 18 + 2600 * 2048), (2000, 3, 2 ** 18 + 2848 * 1024 - 1), (2000, 3, 2 ** 18 + 2848 * 1024),
    (2000, 3, 2 ** 18 + 2848 * 2048 - 1), (2000, 3, 2 ** 18 + 2848 * 2048),   # one source more than the ranges hold: radix passes
    (3000, 7, 255), (3000, 7, 256), (3000, 7, 257),                      # sources with a range each end at 256
    (90000, 10, 40), (90000, 10, 1000), (90000, 10, 3000),               # few sources: radix passes, radix passes, ranges
    (2 ** 21, 1, 50), (2 ** 21 + 1, 1, 50),                              # most destinations a record holds, and one more
    (2048 * 4, 1, 33), (2048 * 4 + 1, 1, 33), (1, 2049, 64)])            # tiles, and a range of more than one chunk
def test_gpu_csr_by_source_ranges(capi, num_dst, fanout, num_src):
    import torch
    rng = np.random.default_rng(num_dst + num_src)
    r = _random_block(rng, num_dst, fanout, num_src)
    # sources at both ends of the id range
    r[: min(r.size, 50)] = np.minimum(np.arange(min(r.size, 50)) % 7, num_src - 1)
    r[-min(r.size, 50):] = num_src - 1 - np.arange(min(r.size, 50)) % min(num_src, 5)
    got = capi.block_formats(torch.from_numpy(r).cuda(), num_dst, fanout, num_src)
    _same({k: (v.cpu().numpy() if hasattr(v, "cpu") else v) for k, v in got.items()},
          _closed_form(r, num_dst, fanout, num_src))


# (a block, a smaller one that takes more ranges of sources, shorter tiles or other passes)
SMALLER = [((3000, 7, 2 ** 18 + 2950 * 1024), (3000, 7, 2 ** 18 + 2847 * 1024)), ((2 ** 21 + 2048, 1, 40000), (2 ** 21, 1, 40000)),
           ((2 ** 20, 9, 2 ** 18 + 2600 * 1024 - 1), (2 ** 20, 8, 2 ** 18 + 2600 * 1024 - 1)),
           ((2 ** 22, 2, 2 ** 22), (2 ** 21, 4, 2 ** 22)), ((300000, 10, 7_000_000), (300000, 10, 2_000_000)),
           ((90000, 10, 3000), (90000, 10, 1000))]


def test_block_workspace_of_a_block_does_for_smaller_ones():
    from apt_amd import capi
    L = capi.lib()
    rng = np.random.default_rng(5)
    pairs = list(SMALLER)
    for _ in range(3000):
        big = [int(np.exp(rng.uniform(0, np.log(m)))) for m in (4e6, 30, 1e7)]
        small = [int(v * rng.choice([1.0, 0.99, 0.5, rng.random()])) for v in big]
        pairs.append((big, small))
    for big, small in pairs:
        for csr in (0, 1):
            assert L.apt_block_workspace_bytes(*small, csr) <= L.apt_block_workspace_bytes(*big, csr), (big, small)
        need = L.apt_block_transpose_workspace_bytes(*big)
        if need:
            assert 0 < L.apt_block_transpose_workspace_bytes(*small) <= need, (big, small)


@pytest.mark.gpu
@pytest.mark.parametrize("big,small", SMALLER[:2])
def test_gpu_formats_of_a_smaller_block_in_the_same_buffers(capi, big, small):
    import torch
    f = capi.BlockFormats(*big)
    r = _random_block(np.random.default_rng(1), *small)
    f.num_dst, f.fanout, f.num_src = small
    f.emit(torch.from_numpy(r).cuda())
    got = f.narrow()
    _same({k: (v.cpu().numpy() if hasattr(v, "cpu") else v) for k, v in got.items()}, _closed_form(r, *small))


@pytest.mark.gpu
@pytest.mark.parametrize("num_dst,fanout,num_src,kind", [
    (8192, 1, 40, "one"), (8193, 1, 40, "one"), (8192 + 4096, 1, 40, "few"), (20481, 1, 33, "few"),   # one workgroup's most, parts
    (60000, 5, 100000, "one"), (60000, 5, 100000, "hub"), (60000, 5, 100000, "hubs"), (60000, 5, 2 ** 18 + 5000, "end"),
    (400000, 1, 70000, "one"), (300000, 2, 64, "few"), (300000, 2, 1000, "few")])
def test_gpu_csr_of_ranges_that_are_sorted_in_parts(capi, num_dst, fanout, num_src, kind):
    """A source with thousands of edges, many such sources, blocks of few sources, all edges in the last range."""
    import torch
    rng = np.random.default_rng(num_dst)
    r = _random_block(rng, num_dst, fanout, num_src, hole=0.1 if fanout > 1 else 0.0, hub=False)
    if kind == "one":
        r[r >= 0] = num_src // 2
    elif kind == "hub":
        r.reshape(num_dst, fanout)[:, 0] = 70
    elif kind == "hubs":
        r[: r.size // 2] = rng.choice([3, 40, 33000, 33001, num_src - 1], r.size // 2)
    elif kind == "end":
        r[r >= 0] = num_src - 1 - (r[r >= 0] % 3)
    want = _closed_form(r, num_dst, fanout, num_src)
    got = capi.block_formats(torch.from_numpy(r).cuda(), num_dst, fanout, num_src)
    _same({k: (v.cpu().numpy() if hasattr(v, "cpu") else v) for k, v in got.items()}, want)
    # the transpose: the same order by slot
    L, rel = capi.lib(), torch.from_numpy(r).cuda()
    indptr = torch.empty(num_src + 1, dtype=torch.int32, device="cuda")
    slots = torch.empty(num_dst * fanout, dtype=torch.int32, device="cuda")
    ws = torch.empty(L.apt_block_transpose_workspace_bytes(num_dst, fanout, num_src), dtype=torch.uint8, device="cuda")
    assert L.apt_block_transpose(rel.data_ptr(), num_dst, fanout, num_src, indptr.data_ptr(), slots.data_ptr(), None, ws.data_ptr(),
                                 ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
    assert np.array_equal(indptr.cpu().numpy(), want["csr_indptr"])
    assert np.array_equal(slots.cpu().numpy()[: want["num_edges"]], np.nonzero(r >= 0)[0][want["csr_eids"]])


def _fastest(f, runs=10):
    import torch
    f()
    times = []
    for _ in range(runs):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


@pytest.mark.gpu
@pytest.mark.parametrize("source", [3, 400_000])
def test_gpu_csr_of_a_hub_takes_no_longer_than_of_an_even_block(capi, source):
    """No workgroup may be left alone with a hub's edges: 8 and 10 times the even block's time for a source in every tenth
    slot, 75 and 92 for a source in all slots, where one workgroup sorted a range (1.0, 1.3, 1.2 and 2.3 since they are
    shared; the bound leaves room for a busy machine)."""
    import torch
    num_dst, fanout, num_src = 100_000, 10, 500_000
    f = capi.BlockFormats(num_dst, fanout, num_src)
    r = torch.randint(0, num_src, (num_dst * fanout,), device="cuda")
    even = _fastest(lambda: f.emit(r))
    r.view(num_dst, fanout)[:, 0] = source
    assert _fastest(lambda: f.emit(r)) <= 4 * even
    r[:] = source
    assert _fastest(lambda: f.emit(r)) <= 5 * even
