"""GPU parity of the sum-of-products SpMM (mamtorch_kernel_sparsev1::cusparsemm) through the C ABI and
through the operator.  The reference checks it by printing the max-abs error against the dense
``a @ b`` (test/test_sparse.py:33-44); here every cell must be within rtol 1e-5 of the fp64 oracle plus
the rounding floor of an fp32 sum in any order, 2^-22 x the sum of |terms| of that cell."""
import numpy as np
import ctypes

import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _random_sparse(rows, k, sparse_rate, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(rows, k, generator=g)
    return a * torch.bernoulli(torch.full((rows, k), 1 - sparse_rate), generator=g)


def _check(got, want, floor, what):
    err = np.abs(got.cpu().numpy().astype(np.float64) - want)
    bound = 1e-5 * np.abs(want) + 2.0 ** -22 * floor + 1e-30
    assert (err <= bound).all(), "%s: worst excess %g at %s" % (what, (err - bound).max(),
                                                                 np.unravel_index((err - bound).argmax(), err.shape))


SHAPES = [(37, 53, 29, 0.9), (200, 310, 64, 0.7), (5, 1, 3, 0.0), (64, 64, 100, 0.99), (1, 40, 256, 0.5),
          (300, 1000, 260, 0.9), (129, 17, 4, 0.2), (33, 90, 1, 0.5), (0, 5, 7, 0.5), (6, 5, 0, 0.5)]


@pytest.mark.parametrize("rows,k,cols,rate", SHAPES)
def test_csr_and_coo_against_oracle(rows, k, cols, rate):
    from mamtorch_amd import capi

    a = _random_sparse(rows, k, rate, seed=rows + cols)
    b = torch.randn(k, cols, generator=torch.Generator().manual_seed(k))
    csr = a.to_sparse_csr()
    crow, col, val = csr.crow_indices(), csr.col_indices(), csr.values()
    want, floor = oracle.csr_spmm(crow.numpy(), col.numpy(), val.numpy(), b.numpy())
    c = capi.csr_spmm(crow.to(DEV), col.to(DEV), val.to(DEV), b.to(DEV), rows)
    torch.cuda.synchronize()
    _check(c, want, floor, "csr")
    coo = a.to_sparse_coo().coalesce()
    idx = coo.indices()
    c2 = capi.coo_spmm(idx[0].contiguous().to(DEV), idx[1].contiguous().to(DEV), coo.values().to(DEV), b.to(DEV), rows)
    torch.cuda.synchronize()
    _check(c2, want, floor, "coo")


@pytest.mark.parametrize("cols", [2, 3, 63, 64, 65, 126, 128, 131, 255, 257, 516])
def test_column_counts_around_the_panels(cols):
    """One, two or four entries per load, ragged last panels, b rows of any alignment; rows of 0 to 70 entries end in
    every remainder of a group, and the last row of b ends the allocation."""
    from mamtorch_amd import capi

    rows, k = 71, 150
    g = torch.Generator().manual_seed(cols)
    a = torch.zeros(rows, k)
    for r in range(rows):
        a[r, torch.randperm(k, generator=g)[:r]] = torch.randn(r, generator=g)
    a[:, k - 1] = 1.0
    csr = a.to_sparse_csr()
    crow, col, val = (t.to(DEV) for t in (csr.crow_indices(), csr.col_indices(), csr.values()))
    coo = a.to_sparse_coo().coalesce()
    idx, values = coo.indices().to(DEV), coo.values().to(DEV)
    for offset in (0, 1):                       # words past a 16-byte boundary
        store = torch.randn(offset + k * cols, generator=g)
        b = store[offset:].view(k, cols)
        want, floor = oracle.csr_spmm(crow.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy(), b.numpy())
        bd = store.to(DEV)[offset:].view(k, cols)
        _check(capi.csr_spmm(crow, col, val, bd, rows), want, floor, "csr, offset %d" % offset)
        _check(capi.coo_spmm(idx[0].contiguous(), idx[1].contiguous(), values, bd, rows), want, floor, "coo, offset %d" % offset)


@pytest.mark.parametrize("cols", [129, 130, 131, 257, 385, 386, 5121, 5122, 5123])
def test_last_columns_are_read_inside_b(cols):
    """Four columns a lane where their number is no multiple of four, a last panel of one to three columns among them: lanes at the
    end take the last four columns, each written by one lane, and no load leaves its row, which for the last row is the end of b."""
    from mamtorch_amd import capi

    rows, k = 21, 40
    g = torch.Generator().manual_seed(cols)
    a = _random_sparse(rows, k, 0.3, seed=cols)
    a[:, k - 1] = 1.0
    store = torch.full((k * cols + 4,), float("nan"))
    store[: k * cols] = torch.randn(k * cols, generator=g)
    b = store[: k * cols].view(k, cols)
    bd = store.to(DEV)[: k * cols].view(k, cols)
    csr, coo = a.to_sparse_csr(), a.to_sparse_coo().coalesce()
    crow, col, val = (t.to(DEV) for t in (csr.crow_indices(), csr.col_indices(), csr.values()))
    row = coo.indices()[0].contiguous().to(DEV)
    want, floor = oracle.csr_spmm(csr.crow_indices().numpy(), csr.col_indices().numpy(), csr.values().numpy(), b.numpy())
    _check(capi.csr_spmm(crow, col, val, bd, rows), want, floor, "csr")
    _check(capi.coo_spmm(row, col, val, bd, rows), want, floor, "coo")
    c, by_rows = capi.coo_spmm_by_rows(row, col, val, bd, rows)
    assert by_rows
    _check(c, want, floor, "by rows")


@pytest.mark.parametrize("k,cols", [(32768, 2000), (32769, 2000), (70000, 600), (90000, 600), (300000, 64)])
def test_panels_by_xcd_and_in_turn(k, cols):
    """Workgroups are numbered panel by panel up to 2^18 rows of b in the (at most eight) panels, and have a grid row per panel
    above: 8, 8, 3, 3 panels and one."""
    from mamtorch_amd import capi

    rows, each = 90, 70
    g = torch.Generator(device=DEV).manual_seed(k)
    crow, col = torch.arange(rows + 1, device=DEV) * each, torch.randint(0, k, (rows * each,), generator=g, device=DEV)
    col[::7] = k - 1
    val, b = torch.randn(rows * each, generator=g, device=DEV), torch.randn(k, cols, generator=g, device=DEV)
    terms = (val.double()[:, None] * b[col].double()).view(rows, each, cols)
    _check(capi.csr_spmm(crow, col, val, b, rows), terms.sum(1).cpu().numpy(), terms.abs().sum(1).cpu().numpy(), "csr")


@pytest.mark.parametrize("n", [63, 64, 65, 127, 4000, 20000, 32768])
@pytest.mark.parametrize("cols", [4, 100, 200])
@pytest.mark.parametrize("layout", [torch.sparse_csr, torch.sparse_coo])
def test_long_rows_are_added_up_in_short_sums(n, cols, layout):
    """Equal terms round the same way each time: n of them in one running sum are off by up to n roundings (0.1 and 0.7, 4000 to
    32768 terms: 4e-5 to 3e-4), sums of 64 that are then added by 64 + n / 64, and a few for the parts of a row."""
    import mamtorch_amd as mt

    rows, k = 20, n + 300
    a = torch.zeros(rows, k)
    a[7, 100:100 + n] = 1.0
    a[12, :3] = 1.0
    b = torch.full((k, cols), 0.1)
    b[:, 1::2] = 0.7
    got = mt.sparse.kernel.v1.cusparsemm(a.to(DEV).to_sparse(layout=layout), b.to(DEV)).cpu().double()
    want = a.double() @ b.double()
    assert bool(((got - want).abs() <= (64 + n / 64 + 4) * 2.0 ** -24 * want).all())


@pytest.mark.parametrize("nnz,rows", [(0, 5), (1, 1), (63, 9), (64, 300), (65, 3), (4096, 70), (4097, 1), (300000, 4001), (0, 256), (70, 255),
                                      (70, 256), (1000, 300000), (2000000, 100003)])
def test_row_offsets(nnz, rows):
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(nnz)
    row = torch.randint(0, rows, (nnz,), generator=g) ** 2 // max(rows - 1, 1)      # crowded first rows, empty ones
    row = row.clamp(max=rows - 1).sort()[0]
    got = capi.coo_row_offsets(row.to(DEV), rows).cpu()
    assert torch.equal(got, torch.searchsorted(row, torch.arange(rows + 1)))


@pytest.mark.parametrize("cols", [1, 40, 100, 260])                       # four, two, one entry per load; two panels
@pytest.mark.parametrize("spoil", ["nothing", "first", "middle", "last", "reversed", "shuffled"])
def test_operands_flagged_as_coalesced_whatever_their_order(cols, spoil):
    """The flag is the caller's word (is_coalesced=True is not checked): rows out of order add up all the same."""
    import mamtorch_amd as mt

    rows, k, nnz = 90, 130, 70000 if spoil == "middle" else 900          # more entries than the check has threads, too
    g = torch.Generator().manual_seed(cols)
    row = torch.randint(0, rows, (nnz,), generator=g).sort()[0]
    col = torch.randint(0, k, (nnz,), generator=g)
    val = torch.randn(nnz, generator=g)
    order = torch.arange(nnz)
    if spoil in ("first", "middle", "last"):
        at = {"first": 0, "middle": 65536 + 77, "last": nnz - 2}[spoil]
        row[at], row[at + 1] = rows - 1, 0
    elif spoil == "reversed":
        order = order.flip(0)
    elif spoil == "shuffled":
        order = torch.randperm(nnz, generator=g)
    row, col, val = row[order], col[order], val[order]
    b = torch.randn(k, cols, generator=g)
    want, floor = oracle.coo_spmm(row.numpy(), col.numpy(), val.numpy(), b.numpy(), rows)
    a = torch.sparse_coo_tensor(torch.stack([row, col]).to(DEV), val.to(DEV), (rows, k), is_coalesced=True)
    assert a.is_coalesced()
    _check(mt.sparse.kernel.v1.cusparsemm(a, b.to(DEV)), want, floor, spoil)


@pytest.mark.parametrize("rows,k,cols,each", [(64, 4096, 64, 41), (300, 1000, 260, 10), (5, 90, 3, 2), (40, 2000, 129, 0)])
@pytest.mark.parametrize("at", [0, 1, -1])
@pytest.mark.parametrize("more", [0, 1])
def test_crowded_rows_are_not_one_wave_s(rows, k, cols, each, at, more):
    """Rows of the most entries that a wave takes, and of one more: nnz * cols / 2^18 + 256.  The result either way,
    and which way it was."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(rows)
    lengths = [each] * rows
    longest = lambda n: 256 + int(n * cols / 2 ** 18)
    while longest(sum(lengths)) != lengths[at % rows]:          # (it counts into nnz itself)
        lengths[at % rows] = longest(sum(lengths))
    lengths[at % rows] += more
    row = torch.repeat_interleave(torch.arange(rows), torch.tensor(lengths))
    nnz = row.numel()
    assert (longest(nnz) < max(lengths)) == bool(more)
    col, val = torch.randint(0, k, (nnz,), generator=g), torch.randn(nnz, generator=g)
    b = torch.randn(k, cols, generator=g)
    want, floor = oracle.coo_spmm(row.numpy(), col.numpy(), val.numpy(), b.numpy(), rows)
    c, by_rows = capi.coo_spmm_by_rows(row.to(DEV), col.to(DEV), val.to(DEV), b.to(DEV), rows)
    assert by_rows == (not more)
    _check(c, want, floor, "crowded" if more else "not crowded")


@pytest.mark.parametrize("cols", [1, 4, 16, 64, 260])
@pytest.mark.parametrize("nnz", [0, 700, 130000, 1300000])
@pytest.mark.parametrize("rows", [65536, 262147])
def test_operands_of_many_rows(rows, nnz, cols):
    """Coalesced COO operands of many rows, most of them empty or not: by rows or by entries, as the operator chooses (both
    within these), and the CSR operator."""
    import mamtorch_amd as mt

    k = 60
    g = torch.Generator().manual_seed(nnz + cols)
    row, col = torch.randint(0, rows, (nnz,), generator=g), torch.randint(0, k, (nnz,), generator=g)
    a = torch.sparse_coo_tensor(torch.stack([row, col]), torch.randn(nnz, generator=g), (rows, k)).coalesce()
    b = torch.randn(k, cols, generator=g)
    idx, val = a.indices(), a.values()
    want, floor = oracle.coo_spmm(idx[0].numpy(), idx[1].numpy(), val.numpy(), b.numpy(), rows)
    _check(mt.sparse.kernel.v1.cusparsemm(a.to(DEV), b.to(DEV)), want, floor, "coo")
    _check(mt.sparse.kernel.v1.cusparsemm(a.to(DEV).to_sparse_csr(), b.to(DEV)), want, floor, "csr")


def test_coo_unsorted_with_duplicates_and_strided_b():
    from mamtorch_amd import capi

    rows, k, cols = 70, 90, 48
    g = torch.Generator().manual_seed(3)
    nnz = 2000
    row = torch.randint(0, rows, (nnz,), generator=g)
    col = torch.randint(0, k, (nnz,), generator=g)
    val = torch.randn(nnz, generator=g)
    wide = torch.randn(k, cols + 16, generator=g)
    b = wide[:, 8:8 + cols]                      # a view: row stride cols + 16, 32-byte offset
    want, floor = oracle.coo_spmm(row.numpy(), col.numpy(), val.numpy(), b.contiguous().numpy(), rows)
    bd = wide.to(DEV)[:, 8:8 + cols]
    c = capi.coo_spmm(row.to(DEV), col.to(DEV), val.to(DEV), bd, rows)
    torch.cuda.synchronize()
    _check(c, want, floor, "coo unsorted")
    # the same matrix through CSR with unsorted columns inside the rows
    order = torch.argsort(row, stable=True)
    crow = torch.zeros(rows + 1, dtype=torch.int64)
    crow[1:] = torch.cumsum(torch.bincount(row, minlength=rows), 0)
    c2 = capi.csr_spmm(crow.to(DEV), col[order].to(DEV), val[order].to(DEV), bd, rows)
    torch.cuda.synchronize()
    _check(c2, want, floor, "csr unsorted columns")


@pytest.mark.parametrize("layout", [torch.sparse_csr, torch.sparse_coo])
def test_operator_name_keys_and_reference_style_check(layout):
    """The reference's own check (test/test_sparse.py:21-44) with seeds: random sizes in [10, 1000], 90 %
    zeros, result against the dense product."""
    import mamtorch_amd as mt

    rng = np.random.default_rng(7)
    n, l, m = (int(v) for v in rng.integers(10, 1000, 3))
    a = _random_sparse(n, l, 0.9, seed=n).to(DEV)
    b = torch.randn(l, m, generator=torch.Generator().manual_seed(m)).to(DEV)
    asparse = a.to_sparse(layout=layout)
    res = torch.ops.mamtorch_kernel_sparsev1.cusparsemm(asparse, b)
    assert res.shape == (n, m) and res.dtype == torch.float32 and res.device == b.device
    res2 = mt.sparse.kernel.v1.cusparsemm(asparse, b)
    want = a.double() @ b.double()
    floor = a.abs().double() @ b.abs().double()
    for r in (res, res2):
        assert bool(((r.double() - want).abs() <= 1e-5 * want.abs() + 2.0 ** -22 * floor).all())
    with pytest.raises(RuntimeError):
        torch.ops.mamtorch_kernel_sparsev1.cusparsemm(asparse, b[:-1])


def test_full_size_against_dense_matmul():
    from mamtorch_amd import capi

    n = 4096
    a = _random_sparse(n, n, 0.9, seed=1).to(DEV)
    b = torch.randn(n, n, generator=torch.Generator().manual_seed(2)).to(DEV)
    csr = a.to_sparse_csr()
    c = capi.csr_spmm(csr.crow_indices(), csr.col_indices(), csr.values(), b, n)
    want = a.double() @ b.double()
    floor = a.abs().double() @ b.abs().double()
    assert bool(((c.double() - want).abs() <= 1e-5 * want.abs() + 2.0 ** -22 * floor).all())
    # linearity, a size-independent property: (2A) @ b == 2 (A @ b) bit for bit (scaling by 2 is exact)
    c2 = capi.csr_spmm(csr.crow_indices(), csr.col_indices(), csr.values() * 2, b, n)
    assert torch.equal(c2, c * 2)


@pytest.mark.parametrize("rows,k,rate", [(37, 53, 0.5), (200, 310, 0.7), (5, 1, 0.0), (64, 1000, 0.3), (0, 5, 0.5), (300, 7, 0.99)])
def test_sparse_operand_written_out_dense(rows, k, rate):
    """mam_csr_to_dense / mam_coo_to_dense: exact (every cell is one stored value, or the sum of a repeated
    coordinate's values)."""
    from mamtorch_amd import capi

    a = _random_sparse(rows, k, rate, seed=rows + k)
    csr = a.to_sparse_csr()
    d = capi.csr_to_dense(csr.crow_indices().to(DEV), csr.col_indices().to(DEV), csr.values().to(DEV), rows, k)
    assert torch.equal(d.cpu(), a + 0.0)           # a + 0.0: the cleared cells are +0
    coo = a.to_sparse_coo().coalesce()
    idx = coo.indices()
    # every coordinate twice, halved values, shuffled: repeated coordinates add up
    perm = torch.randperm(2 * idx.shape[1], generator=torch.Generator().manual_seed(1))
    row2, col2 = torch.cat([idx[0], idx[0]])[perm], torch.cat([idx[1], idx[1]])[perm]
    val2 = torch.cat([coo.values() * 0.5, coo.values() * 0.5])[perm]
    d2 = capi.coo_to_dense(row2.contiguous().to(DEV), col2.contiguous().to(DEV), val2.contiguous().to(DEV), rows, k)
    assert torch.equal(d2.cpu(), a + 0.0)


@pytest.mark.parametrize("layout", [torch.sparse_csr, torch.sparse_coo])
@pytest.mark.parametrize("n,l,m,rate", [(300, 500, 260, 0.6), (1024, 2048, 512, 0.7), (129, 64, 64, 0.0), (64, 100, 63, 0.5)])
def test_operator_at_high_density(layout, n, l, m, rate):
    """From one stored entry in eight on (and 64 columns of b) the operator writes the operand out dense and
    calls the library GEMM; (64, 100, 63) stays on the sparse kernels.  Same bar as everywhere: the fp64 product
    within rtol 1e-5 plus the rounding floor of an fp32 sum."""
    a = _random_sparse(n, l, rate, seed=n + m).to(DEV)
    b = torch.randn(l, m, generator=torch.Generator().manual_seed(m)).to(DEV)
    asparse = a.to_sparse(layout=layout)
    res = torch.ops.mamtorch_kernel_sparsev1.cusparsemm(asparse, b)
    assert res.shape == (n, m) and res.dtype == torch.float32
    want = a.double() @ b.double()
    floor = a.abs().double() @ b.abs().double()
    assert bool(((res.double() - want).abs() <= 1e-5 * want.abs() + 2.0 ** -22 * floor).all())


@pytest.mark.parametrize("operand,one_in", [("csr", 8), ("coo", 8), ("coo in any order", 16), ("wide coo", 16)])
@pytest.mark.parametrize("above", [False, True])
def test_operator_either_side_of_the_density_threshold(operand, one_in, above):
    """The operator changes route at one stored entry in eight (CSR, and coalesced COO up to K = 32768; other COO operands at
    one in sixteen): sparse kernel below, dense copy + library GEMM from there on, and with it the order of summation: one entry
    below and exactly at the threshold, both against the fp64 defining sum within rtol 1e-5 plus the rounding floor of an fp32 sum."""
    R, K, C = (2, 32784, 64) if operand == "wide coo" else (96, 256, 128)
    nnz = R * K // one_in + (0 if above else -1)
    g = torch.Generator().manual_seed(17 + int(above))
    where = torch.randperm(R * K, generator=g)[:nnz]
    a = torch.zeros(R * K)
    a[where] = torch.randn(nnz, generator=g)
    a = a.view(R, K).to(DEV)
    assert int((a != 0).sum()) == nnz
    b = torch.randn(K, C, generator=g).to(DEV)
    if operand == "coo in any order":
        coo = a.to_sparse()
        order = torch.randperm(nnz, generator=g).to(DEV)
        sparse = torch.sparse_coo_tensor(coo.indices()[:, order], coo.values()[order], a.shape)
    else:
        sparse = a.to_sparse(layout=torch.sparse_csr if operand == "csr" else torch.sparse_coo)
    assert operand == "csr" or sparse.is_coalesced() == (operand != "coo in any order")
    res = torch.ops.mamtorch_kernel_sparsev1.cusparsemm(sparse, b)
    want = a.double() @ b.double()
    floor = a.abs().double() @ b.abs().double()
    assert bool(((res.double() - want).abs() <= 1e-5 * want.abs() + 2.0 ** -22 * floor).all())


@pytest.mark.parametrize("rows,k,cols,nnz", [(50, 60, 64, 150), (50, 60, 70, 186), (50, 60, 70, 188), (300, 32768, 130, 9000),
                                             (300, 32769, 130, 9000)])
@pytest.mark.parametrize("order", ["coalesced", "shuffled", "repeated"])
def test_coo_operands_of_the_operator(rows, k, cols, nnz, order):
    """Coalesced, in any order, and with coordinates that occur up to three times, below and above one entry in sixteen, and on
    either side of the K up to which coalesced operands are summed by rows."""
    import mamtorch_amd as mt

    g = torch.Generator().manual_seed(nnz + cols)
    where = torch.randperm(rows * k, generator=g)[:nnz].sort()[0]
    val = torch.randn(nnz, generator=g)
    if order != "coalesced":
        shuffle = torch.randperm(nnz, generator=g)
        where, val = where[shuffle], val[shuffle]
    if order == "repeated":
        where = torch.cat([where[: nnz // 3], where[: nnz // 3], where[: nnz - 2 * (nnz // 3)]])
    row, col, b = where // k, where % k, torch.randn(k, cols, generator=g)
    want, floor = oracle.coo_spmm(row.numpy(), col.numpy(), val.numpy(), b.numpy(), rows)
    a = torch.sparse_coo_tensor(torch.stack([row, col]), val, (rows, k))
    a = a.coalesce() if order == "coalesced" else a
    _check(mt.sparse.kernel.v1.cusparsemm(a.to(DEV), b.to(DEV)), want, floor, order)


@pytest.mark.parametrize("cols,ldb", [(8, 2 ** 27 + 4), (300, 2 ** 27 + 4), (7, 2 ** 27 + 4), (129, 2 ** 27 + 4), (64, 2 ** 27 + 3)])
def test_b_of_more_than_4_gib(cols, ldb):
    """b rows whose byte offsets do not fit 32 bits: four columns a lane where everything is aligned, else one; 9 rows of b in
    4.8 GB, all three entry points."""
    from mamtorch_amd import capi

    rows, k = 37, 9
    g = torch.Generator().manual_seed(cols)
    a = _random_sparse(rows, k, 0.4, seed=cols)
    b = torch.randn(k, cols, generator=g)
    wide = torch.empty((k - 1) * ldb + cols, device=DEV)
    bd = wide.as_strided((k, cols), (ldb, 1))
    bd.copy_(b)
    csr, coo = a.to_sparse_csr(), a.to_sparse_coo().coalesce()
    crow, col, val = (t.to(DEV) for t in (csr.crow_indices(), csr.col_indices(), csr.values()))
    want, floor = oracle.csr_spmm(csr.crow_indices().numpy(), csr.col_indices().numpy(), csr.values().numpy(), b.numpy())
    row = coo.indices()[0].contiguous().to(DEV)
    _check(capi.csr_spmm(crow, col, val, bd, rows), want, floor, "csr")
    _check(capi.coo_spmm(row, col, val, bd, rows), want, floor, "coo")
    c, by_rows = capi.coo_spmm_by_rows(row, col, val, bd, rows)
    assert by_rows
    _check(c, want, floor, "by rows")
    back = torch.arange(val.numel() - 1, -1, -1, device=DEV)
    c, by_rows = capi.coo_spmm_by_rows(row[back], col[back], val[back], bd, rows)
    assert not by_rows
    _check(c, want, floor, "rows that fall")


@pytest.mark.parametrize("ldb", [0, 2 ** 27 + 5])
@pytest.mark.parametrize("cols,blocks", [(1, 300), (100, 255), (100, 256), (300, 127), (300, 128), (300, 511), (300, 512), (513, 342),
                                         (600, 1300)])
@pytest.mark.parametrize("ascending", [False, True])
def test_entries_by_columns_per_lane(cols, blocks, ldb, ascending):
    """One column a lane below 256 workgroups of four columns a lane (256 entries and columns each), two below 1024, four from
    there on; b of more and of less than 4 GiB; more workgroups than the fallback launches, in turns."""
    from mamtorch_amd import capi

    rows, k, nnz = 500, 9, 256 * (blocks - 1) + 1
    g = torch.Generator().manual_seed(cols + blocks)
    row = torch.randint(0, rows, (nnz,), generator=g)
    row = row.sort()[0] if ascending else row
    col, val, b = torch.randint(0, k, (nnz,), generator=g), torch.randn(nnz, generator=g), torch.randn(k, cols, generator=g)
    want, floor = oracle.coo_spmm(row.numpy(), col.numpy(), val.numpy(), b.numpy(), rows)
    if ldb:
        bd = torch.empty((k - 1) * ldb + cols, device=DEV).as_strided((k, cols), (ldb, 1))
        bd.copy_(b)
    else:
        bd = b.to(DEV)
    row, col, val = row.to(DEV), col.to(DEV), val.to(DEV)
    _check(capi.coo_spmm(row, col, val, bd, rows), want, floor, "coo")
    c, by_rows = capi.coo_spmm_by_rows(row, col, val, bd, rows)
    assert ascending or not by_rows
    _check(c, want, floor, "by rows" if by_rows else "after the look")


def test_to_dense_skips_coordinates_outside_the_matrix():
    """mam_csr_to_dense / mam_coo_to_dense write at the coordinates they are given: an entry outside the
    matrix (a malformed tensor) is dropped instead of written out of range."""
    R, K = 4, 8
    crow = torch.tensor([0, 2, 3, 3, 5], dtype=torch.int64, device=DEV)
    col = torch.tensor([1, 8, -1, 7, 1 << 40], dtype=torch.int64, device=DEV)
    val = torch.tensor([1.0, 2.0, 3.0, 4.0, 5.0], device=DEV)
    guard = torch.full((R + 2, K), 9.0, device=DEV)          # rows before and after the matrix must stay
    from mamtorch_amd import capi

    l = capi.lib()
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert l.mam_csr_to_dense(P(crow), P(col), P(val), P(guard[1]), K, R, K, st) == 0
    torch.cuda.synchronize()
    want = torch.full((R + 2, K), 9.0)
    want[1:R + 1] = 0.0
    want[1, 1] = 1.0
    want[4, 7] = 4.0
    assert torch.equal(guard.cpu(), want)
    row = torch.tensor([0, 4, -1, 3, 2], dtype=torch.int64, device=DEV)
    col2 = torch.tensor([1, 0, 0, 7, 8], dtype=torch.int64, device=DEV)
    guard.fill_(9.0)
    assert l.mam_coo_to_dense(P(row), P(col2), P(val), 5, P(guard[1]), K, R, K, st) == 0
    torch.cuda.synchronize()
    want = torch.full((R + 2, K), 9.0)
    want[1:R + 1] = 0.0
    want[1, 1] = 1.0
    want[4, 7] = 4.0
    assert torch.equal(guard.cpu(), want)
