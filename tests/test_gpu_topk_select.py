"""GPU: the top-k select's early stop (the elements at or above the k-th one's leading digits are
sorted once they fit) and its two block sizes, on rows and on candidate lists, against a stable sort."""

import pytest
import torch

from saeflow_amd.kernels import rows_topk, topk_rows

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def rows(kind, M, N, dtype, g):
    x = torch.randn(M, N, generator=g)
    if kind == "relu":  # mostly zeros, fewer positives than the larger k
        x = torch.relu(x - 2.0)
    elif kind == "ties":  # a handful of values: ties at the cut, resolved by column
        x = (x * 2).round() / 2
    elif kind == "equal":
        x = torch.full((M, N), 0.75)
    elif kind == "narrow":  # one leading digit holds every value
        x = 1.0 + torch.rand(M, N, generator=g) * 0.05
    elif kind == "special":
        x[:, ::7] = -0.0
        x[:, 3::50] = float("nan")
        x[:, 5::40] = float("inf")
        x[:, 6::40] = -float("inf")
    return x.to(dtype)


def want(x, k):
    """The first k by value (any NaN above inf, -0 = 0), then column, and their stored bits."""
    key = torch.where(x.isnan(), torch.tensor(float("inf"), dtype=torch.float64), x.double() * 0.5 + 0.0)
    key = torch.where(x.isinf() & (x > 0), torch.tensor(1e300, dtype=torch.float64), key)
    idx = key.sort(dim=1, descending=True, stable=True).indices[:, :k]
    return bits(x).gather(1, idx), idx.int()  # (as integers: float copies may change a NaN's bits)


def bits(t):
    return t.view({4: torch.int32, 2: torch.int16}[t.element_size()])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["normal", "relu", "ties", "equal", "narrow", "special"])
@pytest.mark.parametrize("M,N", [(3, 4096), (2, 12291), (513, 4100), (2, 40000), (5, 700)])
def test_topk_rows_select(M, N, kind, dtype):
    x = rows(kind, M, N, dtype, torch.Generator().manual_seed(M + N))
    xg = x.cuda()
    for k in (1, 48, 511, 512, 513, 700, 1024):
        if k > N:
            continue
        v, i = topk_rows(xg, k)
        wv, wi = want(x, k)
        assert torch.equal(i.cpu(), wi) and torch.equal(bits(v.cpu()), wv), k


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["normal", "relu", "ties", "equal", "narrow", "special"])
def test_rows_topk_select(kind, dtype):
    """Lists of 0 to 4096 candidates (positive or NaN, as the encode keeps them) in shuffled order."""
    g = torch.Generator().manual_seed(9)
    cap, N = 4096, 50000
    lens = [0, 1, 31, 511, 512, 513, 700, 1025, 2048, 4095, 4096]
    x = rows(kind, len(lens), cap, dtype, g).abs()
    x[x == 0] = 1e-3
    cols = torch.stack([torch.randperm(N, generator=g)[:cap] for _ in lens]).int()
    cnt = torch.tensor(lens, dtype=torch.int32)
    for k in (1, 32, 512, 600, 2000):
        v, i = (t.cpu() for t in rows_topk(cnt.cuda(), cols.cuda(), x.cuda(), k, N))
        for r, n in enumerate(lens):
            order = cols[r, :n].argsort()
            take = min(k, n)
            wv, wi = want(bits(x)[r, :n][order][None].view(dtype), take)
            assert torch.equal(i[r, :take], cols[r, :n][order][wi[0].long()]), (k, n)
            assert torch.equal(bits(v)[r, :take], wv[0]), (k, n)
            assert not v[r, take:].any() and len(set(i[r].tolist())) == k, (k, n)
