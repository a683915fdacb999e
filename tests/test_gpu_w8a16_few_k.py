"""int8 products of 33 to 64 rows whose k gives fewer splits than there are idle CUs (tiled GEMM, 64-row tile)."""

import pytest
import torch

from pypto_amd import workloads
from pypto_amd.runtime import w8a16_matmul

pytestmark = pytest.mark.gpu


# k below one split's worth, exactly two splits', a ragged last split, and as many splits as the CUs allow
@pytest.mark.parametrize("m,k,n", [(33, 192, 256), (64, 512, 264), (40, 1088, 1000), (64, 2048, 2048), (57, 4096, 512)])
def test_few_k_products(worker, m, k, n):
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16)
    q, s = workloads.quantize_w8(torch.randn((k, n), generator=g))
    out = torch.full((m, n), float("nan"), device="cuda")
    worker.register(w8a16_matmul)(x.cuda(), q.cuda(), s.cuda(), out)
    torch.cuda.synchronize()
    xd, qd, sd = x.double(), q.double(), s.double()
    # products of bf16 and int8 are exact in fp32: k roundings of partial sums, one of the scale
    bound = (k + 1) * 2.0 ** -24 * (xd.abs() @ qd.abs()) * sd
    assert ((out.cpu().double() - (xd @ qd) * sd).abs() <= bound).all()
