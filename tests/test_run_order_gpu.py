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


@pytest.mark.parametrize("m,n,k", [(3, 2048, 8192), (16, 2049, 8192), (17, 2065, 8192), (32, 2048, 16384), (48, 2049, 24576), (64, 2063, 8192), (65, 2048, 16384), (256, 2048, 8192),
                                   (16, 2561, 8192), (17, 3073, 8192), (24, 4097, 16384), (48, 3081, 24576), (64, 3087, 8192), (32, 3077, 49152)], ids=str)
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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("m,n,k", [(2, 2561, 8192), (16, 2577, 8192), (31, 4098, 16384), (64, 3087, 8192), (100, 3073, 8192)], ids=str)
def test_scaled_output_with_and_without_a_bias(m, n, k, dtype):
    a, b = make_operands(m, n, k, SEED_BASE + 45700 + m + n + k)
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 45800 + m)
    rs, cs = (torch.rand(r, device=DEV, generator=gen) * 1e-3 + 1e-4 for r in (m, n))
    bias = torch.randn(n, device=DEV, generator=gen).to(dtype)
    plain = (fp32_matmul_on_gpu(a, b).float() * rs[:, None] * cs[None]).to(dtype)
    ap, bp = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV)
    ran = 0
    for cfg, name in enumerate(qm.config_names()):
        if name[0] not in "dpv" or not qm.config_supports(cfg, m, n, k):
            continue
        for extra, want in ((None, plain), (bias, plain + bias)):
            d = torch.full((m, n), float("nan"), dtype=dtype, device=DEV)
            qm.gemm_scaled(ap, bp, d, m, n, k, rs, cs, cfg, bias=extra)
            assert torch.equal(d.view(torch.int16), want.view(torch.int16)), (name, extra is None)
        ran += 1
    assert ran >= 10
