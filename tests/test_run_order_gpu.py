"""Rows of 4096 bytes and multiples of them, whose workgroups begin at different places of K (first_of_runs in csrc/qm_common.hpp): every
kernel that does so, waves with one, two and many runs, numbers of waves that do and do not divide the runs."""
import pytest
import torch

import quadmul_amd as qm
from test_gemm_gpu import fp32_matmul_on_gpu
from util import SEED_BASE, make_operands, pack_cpu, poisoned_c

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
KERNELS = [i for i, name in enumerate(qm.config_names()) if name[0] in "dp"]


@pytest.mark.parametrize("m,n,k", [(3, 2048, 8192), (16, 2049, 8192), (17, 2065, 8192), (32, 2048, 16384), (48, 2049, 24576), (64, 2063, 8192), (65, 2048, 16384), (256, 2048, 8192)], ids=str)
def test_every_kernel(m, n, k):
    a, b = make_operands(m, n, k, SEED_BASE + 45000 + m + n + k)
    want = fp32_matmul_on_gpu(a, b)
    ap, bp = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV)
    ran = 0
    for cfg in KERNELS:
        if not qm.config_supports(cfg, m, n, k):
            continue
        c = poisoned_c(m, n, DEV)
        qm.gemm_cfg(ap, bp, c, m, n, k, cfg)
        assert torch.equal(c, want), qm.config_name(cfg)
        ran += 1
    assert ran >= 10


@pytest.mark.parametrize("m,n,k", [(2, 8192, 8192), (31, 33000, 8192), (33, 4100, 32768), (65, 2048, 57344), (257, 2048, 8192)], ids=str)
def test_automatic_choice(m, n, k):
    a, b = make_operands(m, n, k, SEED_BASE + 45500 + m + n + k)
    c = poisoned_c(m, n, DEV)
    qm.gemm(pack_cpu(a).to(DEV), pack_cpu(b).to(DEV), c, m, n, k)
    assert torch.equal(c, fp32_matmul_on_gpu(a, b))
