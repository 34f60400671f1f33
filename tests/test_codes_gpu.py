"""A re-coded in parts, one workgroup per eight or sixteen rows and part, and quantised to codes: where the parts, the pairs of fragments
and the rows end."""
import pytest
import torch

import quadmul
import quadmul_amd as qm
from test_gemm_gpu import fp32_matmul_on_gpu
from util import SEED_BASE, make_operands, pack_cpu, poisoned_c

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# a part of one wave, of some and of all; a last one with fewer K-steps than the others; five parts; groups of 32 rows of which
# one row, half or all are there
# (from 32 million elements on by sixteen rows)
@pytest.mark.parametrize("m,k", [(1, 256), (17, 512 + 32), (33, 1280), (48, 4224), (255, 4352), (64, 8192), (49, 8320), (31, 17024),
                                 (32001, 1024), (7905, 4064), (7999, 4032), (2001, 16032), (1911, 17024), (490, 65504)], ids=str)
def test_every_part_of_the_re_coding(m, k):
    n = 256
    a, b = make_operands(m, n, k, SEED_BASE + 41000 + m + k)
    a_d, b_d = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV)
    want = fp32_matmul_on_gpu(a, b)   # (64 k < 2^24: exact)
    for cfg in (qm.CFG_RECODE, qm.CFG_RECODE_NARROW):
        c = poisoned_c(m, n, DEV)
        qm.gemm_cfg(a_d, b_d, c, m, n, k, cfg)
        assert torch.equal(c, want), cfg


@pytest.mark.parametrize("m,n,k,off", [(8001, 1300, 4098, 0), (7777, 1290, 4130, 1), (4001, 2001, 8014, 0), (4001, 2001, 8024, 2), (1531, 3307, 4100, 0)], ids=str)
def test_rows_at_any_address_by_eight_and_by_sixteen(m, n, k, off):
    """On padded steps, loaded as they are and as shifted dwords, B copied in the same launch."""
    a, b = make_operands(m, n, k, SEED_BASE + 41300 + m + k)
    room = torch.empty(m * (k // 2) + off, dtype=torch.int8, device=DEV)
    a_d = room[off:].view(m, k // 2)
    a_d.copy_(pack_cpu(a))
    assert qm.recode_bytes(m, n, k, ptr_align=1 if off & 1 else 2) > 0
    c = poisoned_c(m, n, DEV)
    quadmul.gemm(a_d, pack_cpu(b).to(DEV), c, m, n, k)
    assert torch.equal(c, fp32_matmul_on_gpu(a, b))


@pytest.mark.parametrize("m,n,k", [(1599, 4096, 2080), (2047, 2080, 4128), (1100, 4096, 10240)], ids=str)
def test_rows_quantised_to_codes(m, n, k):
    """The layer's rows as codes give what the packed rows give, bit for bit."""
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 41500 + k)
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    x = torch.randn(m, k, device=DEV, generator=gen, dtype=torch.float16)
    xq, xs = quadmul.quantize_pack(x)
    want = torch.empty(m, n, dtype=torch.float16, device=DEV)
    qm.gemm_scaled(xq, w, want, m, n, k, xs, ws)
    got = quadmul.linear(x, w, n, ws, None, False)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
