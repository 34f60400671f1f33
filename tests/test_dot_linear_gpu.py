"""The linear layer for one or two rows (csrc/qm_dot_linear.hpp): one launch, the values of the quantisation and the GEMM
one after the other, bit for bit."""
import pytest
import torch

import quadmul
import quadmul_amd as qm
from util import SEED_BASE

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TYPES = {torch.float16: 1, torch.bfloat16: 2, torch.float32: 3}


def both(x, w, n, ws, out, bias):
    xq, xs = quadmul.quantize_pack(x)
    want = torch.empty(x.shape[0], n, dtype=out, device=DEV)
    qm.gemm_scaled(xq, w, want, x.shape[0], n, x.shape[1], xs, ws, bias=bias)
    got = quadmul.linear(x, w, n, ws, bias, out == torch.bfloat16)
    return got.view(torch.int16), want.view(torch.int16)


# a K of less than one chunk pair, of one, of part of one more; every number of waves; more elements than a workgroup keeps in
# registers (8192 per row for four waves); columns that are no multiple of sixteen; the longest rows it is given
@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("n,k", [(1, 32), (17, 96), (64, 256), (33, 288), (100, 2048), (250, 2080), (4096, 4096), (130, 4128), (77, 8192), (64, 11008),
                                 (40, 16384), (4096, 11008)], ids=str)
def test_one_launch_gives_what_two_give(m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 35000 + k + m)
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    for dtype in TYPES:
        room = torch.randn(m * k + 1, device=DEV, generator=gen).to(dtype)
        room[k // 2 + 3] = 40.0
        for x in (room[:m * k].view(m, k), room[1:].view(m, k)):   # (the second aligned to an element only)
            assert qm.library().qm_linear_workspace_bytes(m, n, k, TYPES[dtype], 256) == 0
            for out in (torch.float16, torch.bfloat16):
                for bias in (None, torch.randn(n, device=DEV, generator=gen).to(out)):
                    got, want = both(x, w, n, ws, out, bias)
                    assert torch.equal(got, want), (dtype, out, bias is None)


def test_rows_of_zeros_infinities_and_nan():
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 35500)
    n, k = 64, 4096
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    for dtype in TYPES:
        for value in (0.0, -0.0, float("inf"), -float("inf"), float("nan"), 6e-8):
            for where in (slice(0, k), slice(5, 6), slice(k - 1, k)):
                x = torch.randn(2, k, device=DEV, generator=gen).to(dtype) if where != slice(0, k) else torch.zeros(2, k, device=DEV, dtype=dtype)
                x[1, where] = value
                got, want = both(x, w, n, ws, torch.float16, None)
                assert torch.equal(got, want), (dtype, value, where)


def test_three_rows_and_operands_it_cannot_take_run_as_before():
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 35600)
    lib = qm.library()
    for m, n, k, off in ((3, 64, 512, 0), (1, 64, 514, 0), (2, 40, 512, 4), (1, 16, 16384 + 32, 0), (2, 8192, 8192, 0),
                         (2, 14336, 4096, 0)):
        assert lib.qm_linear_workspace_bytes(m, n, k, 1, 4 if off else 256) > 0
        x = torch.randn(m, k, device=DEV, generator=gen, dtype=torch.float16)
        w0, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
        w = torch.zeros(w0.numel() + 16, dtype=torch.int8, device=DEV)[off:off + w0.numel()].view(n, k // 2).copy_(w0)
        got, want = both(x, w, n, ws, torch.float16, None)
        assert torch.equal(got, want), (m, n, k, off)


def test_captured_and_replayed():
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 35700)
    n, k = 4096, 4096
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    x = torch.randn(1, k, device=DEV, generator=gen, dtype=torch.float16)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = quadmul.linear(x, w, n, ws, None, False)
    for i in range(3):
        x.copy_(torch.randn(1, k, device=DEV, generator=gen))
        y.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        got, want = both(x, w, n, ws, torch.float16, None)
        assert torch.equal(y.view(torch.int16), want) and torch.equal(got, want), i
