"""The linear layer for 3 to 16 rows in one launch (csrc/qm_skinny_linear.hpp): the values of the quantisation and the GEMM one
after the other, bit for bit."""
import pytest
import torch

import quadmul
import quadmul_amd as qm
from test_dot_linear_gpu import both
from util import SEED_BASE

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TYPES = {torch.float16: 1, torch.bfloat16: 2}

# the rows of every kernel, all there and one short; a K of one short run, of one run and a part, of every wave's run or not, of two runs per
# wave; columns that are no multiple of sixteen or of four, fewer blocks of them than CUs and more
CASES = [(3, 1024, 32), (4, 1031, 288), (5, 1040, 96), (8, 1025, 1280), (9, 1030, 160), (16, 8192, 2048), (11, 4099, 1056), (7, 8185, 4096), (8, 4096, 3872),
         (4, 12288, 4064), (3, 4096, 4096), (4, 4093, 4128), (3, 2050, 8192)]


def one_launch(m, n, k, dtype):
    return qm.library().qm_linear_workspace_bytes(m, n, k, TYPES[dtype], 256) == 0


@pytest.mark.parametrize("m,n,k", CASES, ids=str)
def test_one_launch_gives_what_two_give(m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 42000 + k + m)
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    for dtype in TYPES:
        room = torch.randn(m * k + 1, device=DEV, generator=gen).to(dtype)
        room[k // 2 + 3] = 40.0
        for x in (room[:m * k].view(m, k), room[1:].view(m, k)):   # (the second aligned to an element only)
            assert one_launch(m, n, k, dtype)
            for out in (torch.float16, torch.bfloat16):
                for bias in (None, torch.randn(n, device=DEV, generator=gen).to(out)):
                    got, want = both(x, w, n, ws, out, bias)
                    assert torch.equal(got, want), (dtype, out, bias is None)


@pytest.mark.parametrize("m,n,k", [(4, 1024, 4096), (8, 1024, 512), (16, 1024, 256)], ids=str)
def test_rows_of_zeros_infinities_and_nan(m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 42500)
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    for dtype in TYPES:
        for value in (0.0, -0.0, float("inf"), -float("inf"), float("nan"), 6e-8):
            for where in (slice(0, k), slice(5, 6), slice(k - 1, k)):
                x = torch.randn(m, k, device=DEV, generator=gen).to(dtype) if where != slice(0, k) else torch.zeros(m, k, device=DEV, dtype=dtype)
                x[m - 1, where] = value
                got, want = both(x, w, n, ws, torch.float16, None)
                assert torch.equal(got, want), (dtype, value, where)


def test_captured_and_replayed():
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 42700)
    m, n, k = 8, 4096, 4096
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen))
    x = torch.randn(m, k, device=DEV, generator=gen, dtype=torch.float16)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = quadmul.linear(x, w, n, ws, None, False)
    for i in range(3):
        x.copy_(torch.randn(m, k, device=DEV, generator=gen))
        y.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        got, want = both(x, w, n, ws, torch.float16, None)
        assert torch.equal(y.view(torch.int16), want) and torch.equal(got, want), i


@pytest.mark.parametrize("m,k,shift", [(1, 4096, 0), (2, 2048, 0), (4, 4096, 0), (4, 4096, 2048), (8, 4096, -2048), (16, 2048, 0)], ids=str)
def test_in_place(m, k, shift):
    """The output over the rows, or some of them."""
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 42900 + m)
    w, ws = quadmul.quantize_pack(torch.randn(k, k, device=DEV, generator=gen))
    room = torch.randn(3, m * k, device=DEV, generator=gen).to(torch.float16)
    x = room.flatten()[m * k:2 * m * k].view(m, k)
    _, want = both(x, w, k, ws, torch.float16, None)
    assert one_launch(m, k, k, torch.float16)
    need = (4 * m + 255) // 256 * 256 + m * k // 2
    scratch = torch.empty(need, dtype=torch.uint8, device=DEV)
    d = room.flatten()[m * k + shift:2 * m * k + shift]
    assert qm.library().qm_linear_i4(x.data_ptr(), 1, w.data_ptr(), d.data_ptr(), m, k, k, ws.data_ptr(), None, 1, torch.cuda.current_stream().cuda_stream, scratch.data_ptr(), need) == 0
    assert torch.equal(d.view(m, k).view(torch.int16), want)
