"""GPU: the line-slab decode's two round lengths (one workgroup per CU or fewer, and more) against the
one-row-per-wavefront kernel, bit for bit."""

import pytest
import torch

from saeflow_amd.kernels import sparse_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d_in", [512, 4160])  # buffer-resource gathers; fp32 4160: 64-bit addresses
@pytest.mark.parametrize("M", [1, 3, 17, 130, 1025, 4100])
def test_line_slab_rounds_match_the_row_kernel(M, d_in, dtype):
    """1 to 4100 tokens are 4 to far more than 256 workgroups; rows of 0 to 150 entries end inside a round
    and a batch, with invalid indices among them; with and without a bias, and a strided fp32 output."""
    g = torch.Generator().manual_seed(M + d_in)
    n = torch.randint(0, 151, (M,), generator=g)
    n[0] = 150
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), n.cumsum(0)]).cuda()
    nnz = int(indptr[-1])
    idx = torch.randint(-1, 701, (nnz,), generator=g).int().cuda()  # 700 features: -1 and 700 are invalid
    val = torch.randn(nnz, generator=g).to(dtype).cuda()
    W = torch.randn(700, d_in, generator=g).to(dtype).cuda()
    b = torch.randn(d_in, generator=g).to(dtype).cuda()
    rows = {"BLOCK_NNZ": 64, "BLOCK_D": 512}
    for bias in (b, None):
        for out in (None, torch.float32):
            got = sparse_decode(indptr, idx, val, W, bias, out_dtype=out)
            assert torch.equal(got, sparse_decode(indptr, idx, val, W, bias, out_dtype=out, config=rows))
