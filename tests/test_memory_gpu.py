"""Memory that only makes a call faster is asked for, not required: where the allocator does not have it, the call runs
without and gives the same values."""
import contextlib

import pytest
import torch

import quadmul
import quadmul_amd as qm
from util import SEED_BASE

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
MIB = 1 << 20


@contextlib.contextmanager
def room_for(extra):
    """The allocator may reserve `extra` bytes more than it has."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + extra) / total)
    try:
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def packed(gen, rows, k):
    return torch.randint(-128, 128, (rows, k // 2), dtype=torch.int8, device=DEV, generator=gen)


def captured(call):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


M, N, K = 8192, 4096, 8192   # 48 MiB of codes, 32 of packed rows; no workspace that it must have


def test_a_large_product_runs_without_the_room_for_its_codes():
    assert qm.recode_bytes(M, N, K) > 48 * MIB < qm.recode_bytes(M, N, K, True) and qm.workspace_bytes(M, N, K) == 0
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 38000)
    a, b = packed(gen, M, K), packed(gen, N, K)
    want = torch.empty(M, N, dtype=torch.int32, device=DEV)
    qm.gemm(a, b, want, M, N, K, workspace=None)
    want16 = torch.empty(M, N, dtype=torch.float16, device=DEV)
    qm.gemm_scaled(a, b, want16, M, N, K, workspace=None)
    c, d = torch.zeros_like(want), torch.zeros_like(want16)
    for module in (quadmul, qm):
        with room_for(24 * MIB):
            module.gemm(a, b, c, M, N, K)
            module.gemm_scaled(a, b, d, M, N, K)
        assert torch.equal(c, want) and torch.equal(d, want16), module.__name__
        c.zero_(), d.zero_()
    with room_for(24 * MIB):
        graph, _ = captured(lambda: quadmul.gemm(a, b, c, M, N, K))
    for _ in range(3):
        c.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)


def test_the_linear_layer_runs_on_packed_rows_without_the_room_for_codes():
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 38100)
    x = torch.randn(M, K, device=DEV, generator=gen, dtype=torch.float16)
    w, ws = quadmul.quantize_pack(torch.randn(N, K, device=DEV, generator=gen))
    bias = torch.randn(N, device=DEV, generator=gen).to(torch.bfloat16)
    assert qm.library().qm_linear_workspace_bytes(M, N, K, 1, 256) > 48 * MIB
    want = quadmul.linear(x, w, N, ws, bias, True)
    with room_for((64 + 40) * MIB):   # the output, the packed rows and scales
        got = quadmul.linear(x, w, N, ws, bias, True)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    with room_for((64 + 8) * MIB):    # ... and what it cannot do without is still an error
        with pytest.raises(torch.cuda.OutOfMemoryError):
            quadmul.linear(x, w, N, ws, bias, True)
    assert torch.equal(quadmul.linear(x, w, N, ws, bias, True).view(torch.int16), want.view(torch.int16))
