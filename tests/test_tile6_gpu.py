"""The tile kernel on 6-bit floats (csrc/qm_tile6.hpp): bit-exact against exact products, through the explicit
configurations QM_CFG_RECODE and QM_CFG_RECODE_NARROW, at the edges of its tiles, K-steps and work items, in every output form."""
import numpy as np
import pytest
import torch

import quadmul
import quadmul_amd as qm
from test_gemm_gpu import fp32_matmul_on_gpu
from util import SEED_BASE, make_operands, pack_cpu, poisoned_c

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
both_tiles = pytest.mark.parametrize("cfg", [qm.CFG_RECODE, qm.CFG_RECODE_NARROW], ids=["256x256", "256x128"])

# one row, one tile and one element more or less, K-steps short by 32, 64 and 96 nibbles, odd and even numbers of them, a K
# of more than one part of the row sums and of more than four, columns that are no multiple of four, more tiles than CUs
SHAPES = [(1, 256, 256), (15, 257, 288), (33, 300, 320), (255, 511, 352), (256, 256, 384), (257, 260, 416), (300, 512, 4096 + 32),
          (64, 258, 20480 + 128), (2100, 9001, 256), (1030, 18000, 640)]


def operands(m, n, k, seed):
    a, b = make_operands(m, n, k, SEED_BASE + seed)
    return a, b, pack_cpu(a).to(DEV), pack_cpu(b).to(DEV)


@both_tiles
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_every_output_form_is_exact(shape, cfg):
    m, n, k = shape
    a, b, a_d, b_d = operands(m, n, k, 31000 + m + n + k)
    want = fp32_matmul_on_gpu(a, b)   # (64 k < 2^24: exact)
    c = poisoned_c(m, n, DEV)
    qm.gemm_cfg(a_d, b_d, c, m, n, k, cfg)
    assert torch.equal(c, want)
    # a C that is 4-byte aligned only
    room = torch.full((m * n + 1,), -1, dtype=torch.int32, device=DEV)
    c = room[1:].view(m, n)
    qm.gemm_cfg(a_d, b_d, c, m, n, k, cfg)
    assert torch.equal(c, want) and room[0].item() == -1
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + k)
    rs, cs = (torch.rand(x, device=DEV, generator=gen) * 1e-3 + 1e-4 for x in (m, n))
    for dtype in (torch.float16, torch.bfloat16):
        for rows, cols in ((rs, cs), (None, cs), (rs, None)):
            for bias in (None, torch.randn(n, device=DEV, generator=gen).to(dtype)):
                d = torch.empty(m, n, dtype=dtype, device=DEV)
                qm.gemm_scaled(a_d, b_d, d, m, n, k, rows, cols, cfg=cfg, bias=bias)
                e = want.float()
                if rows is not None:
                    e = e * rows[:, None]
                if cols is not None:
                    e = e * cols[None, :]
                e = e.to(dtype)
                if bias is not None:
                    e = e + bias
                assert torch.equal(d.view(torch.int16), e.view(torch.int16)), (dtype, rows is None, cols is None, bias is None)


@both_tiles
@pytest.mark.parametrize("k", [256, 4096, 65504])
def test_extremes_in_closed_form(k, cfg):
    """The largest and the most negative accumulators there are, up to the largest K."""
    m, n = 40, 260
    fill = lambda rows, v: pack_cpu(torch.full((rows, k), v, dtype=torch.int8)).to(DEV)
    for va, vb in ((-8, -8), (-8, 7), (7, -8), (7, 7), (0, 7), (-8, 0)):
        c = poisoned_c(m, n, DEV)
        qm.gemm_cfg(fill(m, va), fill(n, vb), c, m, n, k, cfg)
        assert (c == va * vb * k).all(), (va, vb)


@both_tiles
def test_every_product_of_two_nibbles_at_every_place_of_a_k_step(cfg):
    """One element of A against one of B: the place of each in its 6-bit fields, alone in its row."""
    k, n = 256, 256
    values = torch.arange(-8, 8, dtype=torch.int8)
    for pos in range(0, k, 1 if k < 64 else 7):
        a = torch.zeros(16, k, dtype=torch.int8)
        a[:, pos] = values
        b = torch.zeros(n, k, dtype=torch.int8)
        b[:, pos] = values.repeat(n // 16)
        b[:, pos ^ 1] = 7   # (meets zeros of A only)
        c = poisoned_c(16, n, DEV)
        qm.gemm_cfg(pack_cpu(a).to(DEV), pack_cpu(b).to(DEV), c, 16, n, k, cfg)
        assert torch.equal(c.cpu(), values.int()[:, None] * b[:, pos].int()[None, :]), pos


def test_the_automatic_choice_takes_it_with_the_workspace_and_leaves_it_without():
    m, n, k = 1280, 8192, 4096
    assert qm.recode_bytes(m, n, k) > 0 and qm.workspace_bytes(m, n, k) < qm.recode_bytes(m, n, k)
    a, b, a_d, b_d = operands(m, n, k, 32000)
    want = fp32_matmul_on_gpu(a, b)
    for call in (lambda c: quadmul.gemm(a_d, b_d, c, m, n, k), lambda c: qm.gemm(a_d, b_d, c, m, n, k),
                 lambda c: qm.gemm(a_d, b_d, c, m, n, k, workspace=None),
                 lambda c: qm.gemm(a_d, b_d, c, m, n, k, workspace=torch.empty(qm.recode_bytes(m, n, k) - 16, dtype=torch.uint8, device=DEV))):
        c = poisoned_c(m, n, DEV)
        call(c)
        assert torch.equal(c, want)
    # captured, replayed between other work
    c = poisoned_c(m, n, DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        quadmul.gemm(a_d, b_d, c, m, n, k)
    for _ in range(3):
        c.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)
    d = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    quadmul.gemm_scaled(a_d, b_d, d, m, n, k)
    assert torch.equal(d, want.float().to(torch.bfloat16))


def test_two_streams_have_a_workspace_each():
    m, n, k = 1280, 8192, 4096
    assert qm.recode_bytes(m, n, k) > 0
    sets = [operands(m, n, k, 33000 + i) for i in range(2)]
    want = [fp32_matmul_on_gpu(a, b) for a, b, _, _ in sets]
    outs = [poisoned_c(m, n, DEV) for _ in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sets]
    for _ in range(4):
        for st, (_, _, a_d, b_d), c in zip(streams, sets, outs):
            with torch.cuda.stream(st):
                quadmul.gemm(a_d, b_d, c, m, n, k)
    torch.cuda.synchronize()
    assert all(torch.equal(c, w) for c, w in zip(outs, want))


# K that fills its last 16-byte piece, K-step or pair of them by little, all but little, or not at all; operands at odd addresses
@pytest.mark.parametrize("m,n,k,a_off,b_off", [(1531, 3307, 4100, 0, 0), (1531, 3307, 4098, 1, 2), (1531, 3307, 4222, 0, 0), (1500, 3300, 4224, 8, 0),
                                               (1500, 3300, 4222, 0, 5), (1531, 3307, 4352 - 2, 0, 0), (1531, 3307, 4096, 3, 0), (1300, 8192, 1534, 0, 0)], ids=str)
def test_rows_of_any_k_and_at_any_address(m, n, k, a_off, b_off):
    """... are re-coded and copied padded, where the operands would be copied anyway."""
    a, b = make_operands(m, n, k, SEED_BASE + 36000 + k)
    place = lambda x, off: torch.full((x.numel() + 16,), 0x7F, dtype=torch.int8, device=DEV)[off:off + x.numel()].view(x.shape).copy_(x)
    a_d, b_d = place(pack_cpu(a), a_off), place(pack_cpu(b), b_off)
    align = min((x.data_ptr() & -x.data_ptr()) for x in (a_d, b_d))
    assert qm.recode_bytes(m, n, k, ptr_align=align) > 0 and qm.recode_bytes(m, n, k, True, align) > 0
    want = fp32_matmul_on_gpu(a, b)
    for workspace in (True, torch.full((qm.recode_bytes(m, n, k, ptr_align=align),), 0x55, dtype=torch.uint8, device=DEV)):
        c = poisoned_c(m, n, DEV)
        qm.gemm(a_d, b_d, c, m, n, k, workspace=workspace)
        assert torch.equal(c, want)
    rs, cs = (torch.rand(x, device=DEV) * 1e-3 + 1e-4 for x in (m, n))
    bias = torch.randn(n, device=DEV).to(torch.bfloat16)
    d = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    qm.gemm_scaled(a_d, b_d, d, m, n, k, rs, cs, bias=bias)
    assert torch.equal(d, ((want.float() * rs[:, None]) * cs[None, :]).to(torch.bfloat16) + bias)


@both_tiles
def test_what_it_cannot_take_is_refused(cfg):
    def status(m, n, k, a_off=0, ws=True):
        a = torch.zeros(m * (k // 2) + 16, dtype=torch.int8, device=DEV)[a_off:a_off + m * (k // 2)].view(m, k // 2)
        b = torch.zeros(n, k // 2, dtype=torch.int8, device=DEV)
        c = poisoned_c(m, n, DEV)
        with pytest.raises(qm.QuadmulError):
            qm.gemm_cfg(a, b, c, m, n, k, cfg, ws)
    status(16, 256, 224)
    status(16, 255, 256)
    status(16, 256, 272)
    status(16, 256, 65536)
    status(16, 256, 256, a_off=4)
    status(16, 256, 256, ws=None)
    status(16, 256, 256, ws=torch.empty(qm.workspace_bytes(16, 256, 256, cfg) - 1, dtype=torch.uint8, device=DEV))


# rows that are no multiple of eight, K-steps short and odd in number, each number of chunks per lane, each type
@pytest.mark.parametrize("m,n,k,dtype", [(1283, 8200, 4096, torch.float16), (1100, 8192, 4128, torch.bfloat16), (2048, 14336, 1984, torch.bfloat16),
                                         (1100, 8192, 7200, torch.float16), (1031, 8192, 12320, torch.bfloat16), (2048, 14336, 2016, torch.float32),
                                         (1283, 8192, 4000, torch.float32), (1283, 8192, 6176, torch.float32)], ids=str)
def test_the_linear_layer_quantises_straight_to_codes(m, n, k, dtype):
    """... with the values of the two calls one after the other, bit for bit."""
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 34000 + k)
    room = torch.randn(m * k + 1, device=DEV, generator=gen).to(dtype)
    room[5:5 + k] = 0                       # (most of two rows)
    x = room[1:].view(m, k)                 # aligned to an element only
    x[7] = 0
    x[9, 3] = 3e4
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, generator=gen).to(dtype))
    align = w.data_ptr() & -w.data_ptr()
    groups, steps = (m + 31) // 32, -(-k // 128) + (-(-k // 128) & 1)
    types = {torch.float16: 1, torch.bfloat16: 2, torch.float32: 3}
    assert qm.library().qm_linear_workspace_bytes(m, n, k, types[dtype], align) - (4 * m + 255) // 256 * 256 >= groups * steps * 3072   # codes
    xq, xs = quadmul.quantize_pack(x)
    for out in (torch.float16, torch.bfloat16):
        for bias in (None, torch.randn(n, device=DEV, generator=gen).to(out)):
            want = torch.empty(m, n, dtype=out, device=DEV)
            qm.gemm_scaled(xq, w, want, m, n, k, xs, ws, workspace=None, bias=bias)
            got = quadmul.linear(x, w, n, ws, bias, out == torch.bfloat16)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (out, bias is None)


def test_the_linear_call_refuses_what_it_cannot_do():
    lib = qm.library()
    m, n, k = 16, 64, 256
    x = torch.randn(m, k, device=DEV, dtype=torch.float16)
    w, ws = quadmul.quantize_pack(torch.randn(n, k, device=DEV, dtype=torch.float16))
    d = torch.full((m, n), 7.0, dtype=torch.float16, device=DEV)
    need = lib.qm_linear_workspace_bytes(m, n, k, 1, 256)
    work = torch.empty(need + 256, dtype=torch.uint8, device=DEV)
    call = lambda x_ptr, in_type, ws_ptr, ws_bytes, kk=k, out=1: lib.qm_linear_i4(x_ptr, in_type, w.data_ptr(), d.data_ptr(), m, n, kk, ws.data_ptr(), None, out, None,
                                                                                  ws_ptr, ws_bytes)
    assert call(x.data_ptr(), 1, work.data_ptr(), need - 1) == -7 and call(x.data_ptr(), 1, None, 0) == -7
    assert call(x.data_ptr(), 1, work.data_ptr() + 16, need) == -7
    assert call(x.data_ptr(), 4, work.data_ptr(), need) == call(x.data_ptr(), 1, work.data_ptr(), need, out=3) == -6
    assert call(x.data_ptr(), 1, work.data_ptr(), need, kk=255) == -2
    assert call(x.data_ptr() + 1, 1, work.data_ptr(), need) == -5 and call(None, 1, work.data_ptr(), need) == -1
    torch.cuda.synchronize()
    assert (d == 7.0).all()
    assert lib.qm_linear_workspace_bytes(0, n, k, 1, 256) == 0
