"""Rows off the multiples of four bytes, loaded as aligned dwords and shifted into place (Shifted16 in csrc/qm_common.hpp): every
offset of the operands against the dwords, the first and the last bytes of them, both kernels that load so."""
import pytest
import torch

import quadmul
import quadmul_amd as qm
from test_gemm_gpu import fp32_matmul_on_gpu
from util import SEED_BASE, make_operands, pack_cpu, poisoned_c

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def at_offset(packed, off):
    """The bytes of `packed` from `off` bytes into an allocation on, other bytes all around them."""
    room = torch.full((packed.numel() + off + 9,), 0x5A, dtype=torch.uint8, device=DEV)
    room[off:off + packed.numel()] = packed.view(torch.uint8).flatten().to(DEV)
    return room[off:off + packed.numel()].view(packed.shape).view(torch.int8)


# one row of the fewest bytes; rows of every length modulo four; a last chunk of one byte, of 63, of 64; one row of each block and one more than all
SHAPES = [(1, 1, 32), (1, 17, 34), (2, 33, 126), (15, 300, 130), (16, 301, 250), (17, 700, 1022), (33, 129, 514), (65, 2100, 262), (130, 2050, 1030), (3, 40, 8998)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_any_address(shape):
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 43000 + m + n + k)
    want = fp32_matmul_on_gpu(a, b)
    ap, bp = pack_cpu(a), pack_cpu(b)
    for oa, ob in ((0, 0), (1, 0), (0, 3), (2, 1), (3, 2), (4, 4), (7, 5)):
        c = poisoned_c(m, n, DEV)
        qm.gemm(at_offset(ap, oa), at_offset(bp, ob), c, m, n, k, workspace=None)
        assert torch.equal(c, want), (oa, ob)


@pytest.mark.parametrize("shape", [(1537, 3300, 2078), (1300, 3301, 4098)], ids=str)
def test_rows_re_coded_at_any_address(shape):
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 43500 + m + n + k)
    want = fp32_matmul_on_gpu(a, b)
    ap, bp = pack_cpu(a), pack_cpu(b)
    for oa, ob in ((0, 0), (1, 2), (3, 0), (2, 3)):
        assert qm.recode_bytes(m, n, k, ptr_align=1) > 0
        c = poisoned_c(m, n, DEV)
        quadmul.gemm(at_offset(ap, oa), at_offset(bp, ob), c, m, n, k)
        assert torch.equal(c, want), (oa, ob)
