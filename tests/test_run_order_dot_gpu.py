"""One or two rows on a K of whole 8192: workgroups that begin at different places of K, the GEMM and the linear layer in one launch."""
import pytest
import torch

import quadmul
import quadmul_amd as qm
from test_dot_linear_gpu import both
from test_gemm_gpu import fp32_matmul_on_gpu
from util import SEED_BASE, make_operands, pack_cpu, poisoned_c

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SIZES = [(1, 2048, 8192), (2, 2065, 8192), (1, 4099, 16384), (2, 2048, 24576), (1, 2049, 57344), (1, 2561, 57344), (2, 2579, 8192)]


@pytest.mark.parametrize("m,n,k", SIZES, ids=str)
def test_every_dot_kernel(m, n, k):
    a, b = make_operands(m, n, k, SEED_BASE + 46000 + m + n + k)
    want = fp32_matmul_on_gpu(a, b)
    ap, bp = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV)
    ran = 0
    for cfg, name in enumerate(qm.config_names()):
        if name[0] == "v" and qm.config_supports(cfg, m, n, k):
            c = poisoned_c(m, n, DEV)
            qm.gemm_cfg(ap, bp, c, m, n, k, cfg)
            assert torch.equal(c, want), name
            ran += 1
    assert ran >= 2


@pytest.mark.parametrize("m,n,k", SIZES[:3] + SIZES[5:], ids=str)
def test_linear_layer(m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 46500 + k)
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    for dtype in (torch.float16, torch.bfloat16):
        got, want = both(torch.randn(m, k, device=DEV, generator=gen).to(dtype), w, n, ws, dtype, None)
        assert torch.equal(got, want)
