"""The pipeline's kernels at the sizes where they can go wrong, against the oracle: edges of tiles,
remainders, the smallest and largest of a branch's range. Structure exact; values within the
bound of any summation order (helpers.compare)."""
import numpy as np
import pytest

import dbd_amd
import oracle
from helpers import check_product, compare, reference

pytestmark = pytest.mark.gpu


def from_lengths(lens, ncols, seed, dtype=np.float64):
    """CSR with the given row lengths, distinct random columns, normal values."""
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens, np.int64)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    idx = np.concatenate([np.sort(rng.choice(ncols, int(n), replace=False)) for n in lens if n] or [np.zeros(0)])
    return dbd_amd.CSR(ptr, idx.astype(np.int32), rng.standard_normal(int(ptr[-1])).astype(dtype), (len(lens), ncols))


# row analysis: rows that end at, before and after the edges of the 2048-nonzero tiles, rows over
# several tiles, and tiles over thousands of empty rows (the bisecting branch)
@pytest.mark.parametrize("lens", [
    [1], [2047], [2048], [2049, 1], [2048] * 3, [1] * 2048 + [5], [2047, 2, 2047, 0, 4096],
    [3] + [0] * 5000 + [7, 0, 2100] + [0] * 9000, [0] * 4095 + [1], [1] + [0] * 4100 + [1] * 20 + [0] * 4200 + [4500, 3],
], ids=lambda v: f"{len(v)}rows{sum(v)}nnz")
def test_row_analysis_tiles(gpu_ok, lens):
    B = from_lengths(np.random.default_rng(5).integers(0, 9, 6000), 700, 6)
    A = from_lengths(lens, 6000, 7)
    with dbd_amd.Context() as ctx:
        ctx.set_operands(A, B)
        info = ctx.plan()
        P = oracle.row_products(A.ptr, A.idx, B.ptr)
        assert np.array_equal(ctx.row_products(A.shape[0]), P) and info["products"] == P.sum()
    check_product(A, B)


def test_device_view_of_a_run_of_rows(gpu_ok):
    """A device view may be rows [r0, r1) of a larger matrix: its row pointer starts past 0 and ends
    before the index array does."""
    import torch
    M = from_lengths(np.random.default_rng(8).integers(0, 40, 900), 500, 9)
    B = dbd_amd.gen_er(500, 800, 6, seed=10)
    r0, r1 = 211, 640
    dM, dB = dbd_amd.DeviceCSR.from_host(M), dbd_amd.DeviceCSR.from_host(B)
    V = dbd_amd.DeviceCSR(dM.ptr[r0:r1 + 1].clone(), dM.idx, dM.val, (r1 - r0, 500))
    with dbd_amd.Context(stream=torch.cuda.current_stream()) as ctx:
        ctx.set_operands(V, dB)
        ctx.plan()
        p = torch.empty(r1 - r0 + 1, dtype=torch.int64, device="cuda")
        n = ctx.symbolic(p)
        i, v = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, dtype=torch.float64, device="cuda")
        ctx.numeric(p, i, v)
        C = dbd_amd.CSR(p.cpu().numpy(), i.cpu().numpy(), v.cpu().numpy(), (r1 - r0, 800))
    e0, e1 = int(M.ptr[r0]), int(M.ptr[r1])
    S = dbd_amd.CSR(M.ptr[r0:r1 + 1] - e0, M.idx[e0:e1], M.val[e0:e1], (r1 - r0, 500))
    compare(C, reference(S, B), np.float64, "rows of a larger matrix")


# hub rows (long rows in column ranges of 8192): widths at the edges of a range, of the 131072-column
# count window and of the bucketed form (more than 8 ranges); rows of many entries (over several
# split chunks of 1024), rows of few entries with many products, and long rows that stay in the windows
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ncols", [8191, 8192, 8193, 40000, 65536, 65537, 131072, 131073, 300001])
def test_hub_rows_in_ranges(gpu_ok, ncols, dtype):
    rng = np.random.default_rng(ncols)
    blen = np.concatenate([rng.integers(0, 64, 2400), rng.integers(64, 600, 500), [min(ncols, 9000)] * 8, [63, 64, 65]])
    B = from_lengths(rng.permutation(blen), ncols, 11, dtype)
    A = from_lengths([1, 2900, 1025, 1024, 700, 300, 0, 60, 12, 2049], B.shape[0], 12, dtype)
    _, _, info = check_product(A, B, what=f"{ncols} columns")
    # rows of many entries are hub rows (a row of at most 8192 columns fits a hash table)
    assert info["num_rows"][-1] >= 3 if ncols > 8192 else info["num_rows"][-1] == 0


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ncols", [20000, 100000])
def test_hub_sums_of_special_values(gpu_ok, ncols, dtype):
    """Entries whose sum is zero, -0.0, denormal, infinite or NaN are entries of C like any other.
    The values are small multiples of one number, so every order of summation gives the same sum."""
    rng = np.random.default_rng(13)
    B = from_lengths(rng.permutation([10, 40, 63, 64, 900, 2500] * 60), ncols, 14, dtype)
    A = from_lengths([360, 200, 2, 360], B.shape[0], 15, dtype)
    A.val[:] = rng.choice([1.0, -1.0, 0.0, -0.0], A.nnz)
    tiny = np.finfo(dtype).smallest_subnormal
    for what, vals in (("zeros", [0.0, -0.0]), ("signs", [1.0, -1.0, 0.0, -0.0]), ("subnormal", [tiny, -tiny, 0.0, -0.0]),
                       ("infinite", [1.0, np.inf, 2.0, 0.0]), ("nan", [1.0, np.nan, -0.0, 3.0])):
        B.val[:] = rng.choice(np.array(vals, dtype), B.nnz)
        Cptr, Cidx, Cval, _ = reference(A, B)
        with dbd_amd.Context(dtype=dtype) as ctx:
            ctx.set_operands(A, B)
            ctx.run("compute")
            C = ctx.result()
        assert np.array_equal(C.ptr, Cptr) and np.array_equal(C.idx, Cidx), what
        assert np.array_equal(C.val, Cval.astype(dtype), equal_nan=True), what


# binning: one launch up to 64 tiles of 256 rows, by tile beyond; the scan in one launch up to 32768
# counters, in three beyond; block tables over both
@pytest.mark.parametrize("block_rows", [256, 4096])
@pytest.mark.parametrize("nrows", [1, 63, 64, 65, 255, 257, 16383, 16384, 16385, 16640, 700_001])
def test_bins_and_block_tables(gpu_ok, nrows, block_rows):
    rng = np.random.default_rng(nrows)
    B = from_lengths(rng.integers(0, 70, 300), 5000, 16)
    lens = np.minimum(rng.geometric(0.3, nrows) - 1, 40) if nrows > 1 else [7]
    ptr = np.concatenate([[0], np.cumsum(lens)])
    idx = np.concatenate([np.sort(rng.permutation(300)[:n]) for n in range(41)])  # a row of n entries: the n-th list
    at = np.concatenate([[0], np.cumsum(np.arange(41))])
    idx = idx[np.repeat(at[np.asarray(lens)] - ptr[:-1], lens) + np.arange(ptr[-1])]
    A = dbd_amd.CSR(ptr, idx.astype(np.int32), rng.standard_normal(int(ptr[-1])), (nrows, 300))
    P = oracle.row_products(A.ptr, A.idx, B.ptr)
    ref = reference(A, B)
    with dbd_amd.Context(block_rows=block_rows) as ctx:
        ctx.set_operands(A, B)
        info = ctx.plan()
        bptr, bprod, binfo = dbd_amd.plan_blocks(P, block_rows)
        gptr, gprod = ctx.blocks(info["num_blocks"])
        assert np.array_equal(gptr, bptr) and np.array_equal(gprod, bprod)
        assert all(info[k] == binfo[k] for k in ("products", "criteria", "max_block_products", "blocks_any"))
        ctx.run("compute")
        compare(ctx.result(), ref, np.float64, f"{nrows} rows")
        assert sum(ctx.plan_info()["num_rows"]) == nrows
    if nrows > 60000:  # several chunks: the offsets by tile
        with dbd_amd.Context(block_rows=block_rows, chunks_hint=5) as ctx:
            ctx.set_operands(A, B)
            assert ctx.run("d2h")["chunks"] > 1
            compare(ctx.result(), ref, np.float64, "chunks")


# several rows per wave (more than 8192 rows of a category): groups cut off at the end of a bin, rows
# with more entries than their lanes, with one long B row, and full tables; one-wave rows below that
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nrows", [8100, 8193, 30011])
def test_several_rows_per_wave(gpu_ok, nrows, dtype):
    rng = np.random.default_rng(nrows)
    blen = rng.permutation([0] * 20 + [1] * 300 + [2, 3, 5, 8, 13, 16, 31, 32, 33, 63, 64, 65, 127, 128] * 20)
    for ncols, per_row in ((700, 6), (40, 40), (3_000_000, 12)):  # duplicates; full tables of 32 columns; distinct
        B = from_lengths(np.minimum(blen, ncols), ncols, 17, dtype)
        lens = rng.integers(0, per_row, nrows)
        idx = np.concatenate([np.sort(rng.choice(B.shape[0], n, replace=False)) for n in lens])
        A = dbd_amd.CSR(np.concatenate([[0], np.cumsum(lens)]), idx.astype(np.int32),
                        rng.standard_normal(idx.size).astype(dtype), (nrows, B.shape[0]))
        check_product(A, B, what=f"{ncols} columns")


# backward of hub rows: in windows of one range (up to 8 ranges), of several (up to 16 windows), and by
# the window kernel beyond; the forward pass again afterwards (it shares workspace with the latter)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ncols", [8193, 65536, 65537, 200_000, 262_145, 600_000])
def test_backward_hub_rows(gpu_ok, ncols, dtype):
    import torch
    from test_gpu_backward import check_grads, run_backward
    rng = np.random.default_rng(ncols)
    B = from_lengths(rng.permutation(np.concatenate([rng.integers(0, 64, 1500), rng.integers(64, 700, 400)])), ncols, 18,
                     dtype)
    A = from_lengths([1, 1800, 64, 65, 300, 0, 1025, 30], B.shape[0], 19, dtype)
    check_grads(A, B, *run_backward(A, B))
    ref = reference(A, B)
    dA, dB = dbd_amd.DeviceCSR.from_host(A), dbd_amd.DeviceCSR.from_host(B)
    with dbd_amd.Context(dtype=dtype, stream=torch.cuda.current_stream()) as ctx:
        ctx.set_operands(dA, dB)
        ctx.plan()
        p = torch.empty(A.shape[0] + 1, dtype=torch.int64, device="cuda")
        n = ctx.symbolic(p)
        i, v = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, dtype=dA.val.dtype, device="cuda")
        ctx.numeric(p, i, v)
        ctx.backward(p, i, v, torch.empty_like(dA.val), torch.zeros_like(dB.val))
        i.fill_(-1), v.fill_(0)
        ctx.numeric(p, i, v)
        compare(dbd_amd.CSR(p.cpu().numpy(), i.cpu().numpy(), v.cpu().numpy(), (A.shape[0], ncols)), ref, dtype)


def test_backward_sums_in_parts_add_to_db(gpu_ok):
    """Many FP32 products per value of B are summed in parts; dB is added to, as without them, and each
    value is as near the FP64 gradient as a sum of few parts."""
    import torch
    A, B = dbd_amd.gen_rmat(12, 48, seed=20, dtype=np.float32), dbd_amd.gen_er(4096, 600, 5, seed=21, dtype=np.float32)
    dA, dB = dbd_amd.DeviceCSR.from_host(A), dbd_amd.DeviceCSR.from_host(B)
    with dbd_amd.Context(dtype="f32", stream=torch.cuda.current_stream()) as ctx:
        ctx.set_operands(dA, dB)
        assert ctx.plan()["products"] >= 32 * B.nnz  # the parts are in use
        p = torch.empty(A.shape[0] + 1, dtype=torch.int64, device="cuda")
        n = ctx.symbolic(p)
        i, v = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, device="cuda")
        ctx.numeric(p, i, v)
        gB = torch.full_like(dB.val, 3.0)
        ctx.backward(p, i, v, None, gB)
    _, db, miss = oracle.backward(A, B, p.cpu().numpy(), i.cpu().numpy(), v.double().cpu().numpy())
    assert miss == 0
    scale = np.abs(db) + 3.0
    assert np.all(np.abs(gB.cpu().numpy() - 3.0 - db) <= 1e-5 * scale)


# rows of 1024 columns and more without a hash table: at the edges of the width of a window of values
# (4096 columns), of a window of ranks (65536) and of four windows of values; rows of up to 64 entries
# (shared by the waves), up to 512 (one per lane) and more; short, banded and mixed B rows; products of
# zeros, whose sums must not pass for absent columns
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ncols, base, width", [
    (4096, 0, 4096), (4097, 0, 4097), (8192, 2048, 4096), (16384, 0, 16384), (16385, 1, 16384), (65536, 0, 65536),
    (65537, 0, 65537), (65537, 1, 65536), (200000, 70001, 4095), (200000, 70001, 4097), (200000, 131071, 65537),
    (400000, 0, 400000)])
def test_rank_windows(gpu_ok, dtype, ncols, base, width):
    rng = np.random.default_rng(ncols + width)
    lens = np.concatenate([rng.integers(0, 64, 1500), rng.integers(64, 300, 1400), rng.integers(2500, 3000, 100)])
    B = from_lengths(lens, width, 21, dtype)
    B.idx += base
    B.val[rng.random(len(B.val)) < 0.05] = -0.0
    B = dbd_amd.CSR(B.ptr, B.idx, B.val, (len(lens), ncols))
    groups = [np.arange(1500), np.arange(3000), np.arange(2900, 3000)]  # short, mixed, long B rows
    rows = []
    for nA, k in [(1, 2), (2, 2), (4, 2), (12, 1), (30, 1), (63, 1), (64, 0), (64, 1), (65, 0), (65, 1), (150, 0), (200, 0),
                  (511, 0), (512, 0), (513, 0), (700, 0), (1024, 0)]:
        rows.append(np.sort(rng.choice(groups[k], nA, replace=False)))
    A = dbd_amd.CSR(np.concatenate([[0], np.cumsum([len(r) for r in rows])]), np.concatenate(rows).astype(np.int32),
                    rng.standard_normal(sum(map(len, rows))).astype(dtype), (len(rows), len(lens)))
    check_product(A, B)


# symbolic tables of 1024 slots and more, which take one wave, 256 or 512 threads a row where rows are many:
# counts of rows on both sides of that, products at the tables' limits
@pytest.mark.parametrize("few", [True, False])
def test_symbolic_tables_by_row_count(gpu_ok, few):
    rng = np.random.default_rng(23)
    limits, counts = (256, 512, 1024, 2048, 4096), (40, 40, 40, 40) if few else (8193, 8193, 1025, 1025)
    edge = [m + d for m in limits for d in (-1, 0, 1)]
    B = from_lengths(rng.permutation(edge + list(rng.integers(1, 4096, 200))), 9001, 24)
    order = np.argsort(np.diff(B.ptr), kind="stable")
    lens = np.diff(B.ptr)[order]
    rows = []
    for (lo, hi), n in zip(zip(limits, limits[1:]), counts):
        one = order[(lens >= lo - 1) & (lens <= hi + 1)]  # one entry a row
        rows += [np.array([b]) for b in one]
        small = order[lens <= hi // 2]
        for _ in range(n):  # one or two entries, up to hi products
            r = rng.choice(one, 1) if len(small) < 3 or rng.random() < 0.5 else rng.choice(small, 2, replace=False)
            rows.append(np.sort(r))
    A = dbd_amd.CSR(np.concatenate([[0], np.cumsum([len(r) for r in rows])]), np.concatenate(rows).astype(np.int32),
                    rng.standard_normal(sum(map(len, rows))), (len(rows), B.shape[0]))
    check_product(A, B)


# backward of long rows over up to 65536 columns: C's row by rank, 14336 FP32 or 7168 FP64 values at a time
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ncols", [65535, 65536, 65537])
def test_backward_ranked_rows(gpu_ok, ncols, dtype):
    from test_gpu_backward import check_grads, run_backward
    rng = np.random.default_rng(ncols)
    edge = [4096, 4097, 7167, 7168, 7169, 14335, 14336, 14337, 16000]
    B = from_lengths(np.concatenate([edge, rng.integers(0, 200, 400)]), ncols, 25, dtype)
    B.idx[B.ptr[8]], B.idx[B.ptr[9] - 1] = 0, ncols - 1  # a row from the first column to the last
    rows = [np.array([e]) for e in range(9)] + [np.array([0, 2]), np.array([1, 3, 20])]
    rows += [np.sort(rng.choice(np.arange(9, 409), n, replace=False)) for n in (64, 65, 100)]
    A = dbd_amd.CSR(np.concatenate([[0], np.cumsum([len(r) for r in rows])]), np.concatenate(rows).astype(np.int32),
                    rng.standard_normal(sum(map(len, rows))).astype(dtype), (len(rows), B.shape[0]))
    check_grads(A, B, *run_backward(A, B))
    # the entries of C's rows in another order, as the hash tables take them
    import torch
    dA, dB = dbd_amd.DeviceCSR.from_host(A), dbd_amd.DeviceCSR.from_host(B)
    with dbd_amd.Context(dtype=dtype, stream=torch.cuda.current_stream()) as ctx:
        ctx.set_operands(dA, dB)
        ctx.plan()
        p = torch.empty(A.shape[0] + 1, dtype=torch.int64, device="cuda")
        n = ctx.symbolic(p)
        i, v = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, dtype=dA.val.dtype, device="cuda")
        ctx.numeric(p, i, v)
        h = p.cpu().numpy()
        hub = h[1:] - h[:-1] > 4096  # hub and wide long rows: in order only
        order = np.concatenate([np.arange(a, b) if w else np.arange(a, b)[::-1] for a, b, w in zip(h, h[1:], hub)])
        if ncols > 65536:
            order = np.arange(n)
        order = torch.from_numpy(order).cuda()
        gA, gB = torch.empty_like(dA.val), torch.zeros_like(dB.val)
        ctx.backward(p, i[order], v[order], gA, gB)
        check_grads(A, B, h, i.cpu().numpy(), v.cpu().numpy(), gA.cpu().numpy(), gB.cpu().numpy())
