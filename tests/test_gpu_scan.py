"""GPU: the count scan that sizes a CSR (one block up to 32768 rows, three passes above), the numbers
it leaves for the host, and the row-candidate calls that use them."""

import pytest
import torch

from saeflow_amd import kernels
from saeflow_amd.kernels import dense_to_csr, encode_rows, exclusive_scan, row_lists, rows_to_csr, scan_counts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [0, 1, 15, 16, 17, 4095, 4096, 4097, 16384, 16385, 32768, 32769, 300001])
@pytest.mark.parametrize("offset", [0, 1])  # counts that are 16-B aligned or not
def test_scan_counts(M, offset):
    g = torch.Generator().manual_seed(M)
    counts = torch.randint(0, 1000, (M + offset,), generator=g, dtype=torch.int32)[offset:]
    if M > 2:
        counts[M // 2] = 70000  # sums beyond 2^31 at the largest M would not show otherwise
    dev = torch.cat([torch.zeros(offset, dtype=torch.int32), counts]).cuda()[offset:]
    indptr, nnz, longest = scan_counts(dev)
    want = torch.cat([torch.zeros(1, dtype=torch.int64), counts.long().cumsum(0)])
    assert torch.equal(indptr.cpu(), want) and torch.equal(exclusive_scan(dev).cpu(), want)
    assert nnz == int(want[-1]) and longest == (int(counts.max()) if M else 0)


@pytest.mark.parametrize("M", [3, 40000])
def test_scan_counts_of_large_counts(M):
    """Sums past 2^31; a largest count of 2^20 and more is reported as 2^20 - 1."""
    counts = torch.full((M,), 1 << 20, dtype=torch.int32)
    counts[-1] = 2 ** 31 - 1
    indptr, nnz, longest = scan_counts(counts.cuda())
    assert nnz == (M - 1) * (1 << 20) + 2 ** 31 - 1 == int(indptr[-1]) and longest == (1 << 20) - 1
    counts[-1] = 5
    assert scan_counts(counts.cuda())[2] == (1 << 20) - 1


@pytest.mark.parametrize("M", [1, 300])
def test_row_candidates_count_from_zero_and_sort_with_a_known_bound(M):
    """encode_rows clears its counts whatever the memory held; rows_to_csr with the longest list known
    equals the call without it, with and without lists above 256 entries."""
    for b in (-1.0, 1.0):  # few and nearly all of the 600 features kept
        x = torch.randn(M, 64, generator=torch.Generator().manual_seed(1)).cuda()
        W = torch.randn(64, 600, generator=torch.Generator().manual_seed(2)).cuda() / 8
        b_enc = torch.full((600,), b, device="cuda")
        junk = torch.full((M,), 12345, dtype=torch.int32, device="cuda")
        del junk  # its block is what the counts are likely to get
        cnt, idx, val = encode_rows(x, W, b_enc, torch.zeros(64, device="cuda"), cap=1024)
        f = torch.relu(x.double() @ W.double() + b)
        assert torch.equal(cnt.cpu(), (f > 0).sum(1).int().cpu())
        indptr, nnz, longest = scan_counts(cnt)
        assert (longest > 256) == (b > 0)
        for a, c in zip(rows_to_csr(cnt, idx, val, indptr, nnz, longest), rows_to_csr(cnt, idx, val, indptr, nnz)):
            assert torch.equal(a, c)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N", [8, 2048, 2051, 16384, 16392, 40003])  # rows of one group of loads, of several, with a tail
def test_dense_to_csr_counts_and_lists_in_one_read(dtype, N, monkeypatch):
    """Without counts: rows that fit their lists (up to 256 nonzeros) and batches with some that do
    not, against the CSR by hand; -0.0 is a zero, NaN and infinities are kept. The lists are for large
    f alone, so the sizes they start at are lowered here."""
    monkeypatch.setattr(kernels.decode, "LIST_MIN_BYTES", 0)
    monkeypatch.setattr(kernels.decode, "LIST_MIN_ROW_BYTES", 0)
    M, pad = 5, -N % 8
    for longest in (0, 1, 255, 256, 257, N):
        longest = min(longest, N)
        f = torch.zeros(M, N + pad, dtype=dtype)[:, :N]  # rows stay 16-B aligned
        for m, n in enumerate((longest, longest // 2, 0, min(longest, 3), longest)):
            g = torch.Generator().manual_seed(7 * m + n)
            f[m, torch.randperm(N, generator=g)[:n]] = torch.rand(n, generator=g).to(dtype) + 1
        if longest >= 3:
            f[3, f[3].nonzero().flatten()] = torch.tensor([float("nan"), float("-inf"), -2.0], dtype=dtype)
        f[2, N - 1] = -0.0
        dev = torch.empty(M, N + pad, dtype=dtype, device="cuda")[:, :N].copy_(f)
        counts = (f != 0).sum(1)
        lists, idx, val = row_lists(dev)
        assert torch.equal(lists.cpu(), counts.int())
        indptr, indices, values = dense_to_csr(dev)
        where = (f != 0).nonzero()
        assert torch.equal(indptr.cpu(), torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)]))
        assert torch.equal(indices.cpu(), where[:, 1].int())
        bits = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(values.cpu().view(bits), f[where[:, 0], where[:, 1]].view(bits))


def test_dense_to_csr_of_rows_the_vector_loads_do_not_take(monkeypatch):
    monkeypatch.setattr(kernels.decode, "LIST_MIN_BYTES", 0)
    monkeypatch.setattr(kernels.decode, "LIST_MIN_ROW_BYTES", 0)
    f = torch.zeros(4, 1001).index_fill_(1, torch.tensor([0, 17, 1000]), 2.5).cuda()
    for g in (f, f[:, 1:], f.t().contiguous().t()):
        indptr, indices, values = dense_to_csr(g)
        want = g.to_sparse_csr()
        assert torch.equal(indptr, want.crow_indices()) and torch.equal(indices.long(), want.col_indices())
        assert torch.equal(values, want.values())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_dense_to_csr_of_rows_around_the_list_length(dtype, monkeypatch):
    """Whole 16-B chunks of one thread nonzero (its count of a group of loads is 64 or 32), which fill
    a row's list exactly or pass it by one; half of the rows past their list; all of them a little past
    it; and so far past it on average that everything is compacted from f."""
    monkeypatch.setattr(kernels.decode, "LIST_MIN_BYTES", 0)
    monkeypatch.setattr(kernels.decode, "LIST_MIN_ROW_BYTES", 0)
    M, N = 6, 3 * 256 * 8 * 8
    epc = 8 if dtype == torch.bfloat16 else 4

    def check(f):
        indptr, indices, values = dense_to_csr(f.cuda())
        where = (f != 0).nonzero()
        assert torch.equal(indptr.cpu(), torch.cat([torch.zeros(1, dtype=torch.int64), (f != 0).sum(1).cumsum(0)]))
        assert torch.equal(indices.cpu(), where[:, 1].int()) and torch.equal(values.cpu(), f[where[:, 0], where[:, 1]])

    f = torch.zeros(M, N, dtype=dtype)
    for m in range(M):
        for t in range(256 // (8 * epc)):  # threads of one wavefront, or of several, in the group m // 2
            for u in range(8):
                at = ((m // 2) * 2048 + u * 256 + (t if m % 2 else 37 * t % 256)) * epc
                f[m, at:at + epc] = torch.arange(1, epc + 1).to(dtype) + m
    assert (f != 0).sum(1).tolist() == [256] * M
    check(f)
    f[::2, N - 1] = 1  # every second row passes its list
    f[1::2, f[1].nonzero()[0]] = 0
    check(f)
    f[1::2, N - 2:] = 3
    check(f)
    f = torch.zeros(M, N, dtype=dtype)
    for m in range(M):
        f[m, torch.randperm(N, generator=torch.Generator().manual_seed(m))[:265 + m]] = 1
    check(f)
    f[:, f.sum(0) == 0] = torch.cat([torch.ones(30), torch.zeros(N)])[:int((f.sum(0) == 0).sum())].to(dtype)
    monkeypatch.setattr(kernels.decode, "rows_to_csr", None)  # 295 and more a row: not sorted at all
    check(f)
