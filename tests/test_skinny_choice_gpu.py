"""The products and the scaled outputs of the kernels that 3 to 64 rows are given, where their blocks are ragged."""
import pytest
import torch

import quadmul_amd as qm
from test_gemm_gpu import fp32_matmul_on_gpu
from util import SEED_BASE, make_operands, pack_cpu, poisoned_c

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("m,n,k", [
    (3, 4097, 6144), (16, 8191, 8160), (3, 1023, 16416), (16, 4095, 16448), (17, 33, 1024), (32, 2047, 2048), (17, 2049, 1056), (31, 4095, 2016), (17, 16385, 3584),
    (32, 20481, 4064), (17, 8193, 4128), (31, 12287, 4128), (32, 12289, 4128), (17, 16383, 4128), (33, 16385, 2048), (47, 22527, 2080), (49, 10753, 2048), (59, 12287, 2080)], ids=str)
def test_int32_and_scaled(m, n, k):
    a, b = make_operands(m, n, k, SEED_BASE + 44000 + m + n + k)
    want = fp32_matmul_on_gpu(a, b)
    ap, bp = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV)
    c = poisoned_c(m, n, DEV)
    qm.gemm(ap, bp, c, m, n, k)
    assert torch.equal(c, want)
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 44500)
    rs, cs = (torch.rand(size, device=DEV, generator=gen) + 0.5 for size in (m, n))
    got = torch.full((m, n), -1.0, device=DEV, dtype=torch.float16)
    scale = 2.0 ** -8
    qm.gemm_scaled(ap, bp, got, m, n, k, rs * scale, cs * scale)
    # one product of the scales, one with the sum, one rounding to half: 2^-24 each and 2^-11 relative, 2^-25 where the half is subnormal
    exact = want.double() * (rs * scale).double()[:, None] * (cs * scale).double()[None, :]
    assert ((got.double() - exact).abs() <= exact.abs() * (2.0 ** -11 + 3 * 2.0 ** -24) + 2.0 ** -25).all()
