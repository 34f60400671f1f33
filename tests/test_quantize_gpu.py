"""GPU parity of the fused quantise + pack kernel (through the C ABI) against the CPU oracle:
packed bytes and scales bit-exact; then the whole int4 linear layer end to end."""
import numpy as np
import pytest
import torch

import quadmul_amd as qm
from util import SEED_BASE

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SHAPES = [(1, 2), (3, 6), (7, 30), (16, 64), (33, 130), (64, 4096), (5, 4104), (9, 8192), (4, 16384), (3, 16392), (2, 40960), (257, 1184), (0, 64), (5, 0)]


def make_x(rows, k, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((rows, k), generator=g) * (torch.rand((rows, 1), generator=g) * 20 + 0.01)
    if rows > 2:
        x[1] = 0                      # an all-zero row
        x[2] = torch.round(x[2])      # exact ties after scaling are likely here
    return x.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_quantize_pack_matches_oracle(oracle_mod, shape, dtype):
    rows, k = shape
    x = make_x(rows, k, dtype, SEED_BASE + 8000 + rows + k)
    want_p, want_s = oracle_mod.quantize_pack(x.to(torch.float32).numpy())
    packed, scales = qm.quantize_pack(x.to(DEV))
    torch.cuda.synchronize()
    assert packed.shape == (rows, k // 2) and packed.dtype == torch.int8 and scales.shape == (rows,)
    assert (scales.cpu().numpy() == want_s).all()
    got = packed.cpu().numpy().view(np.uint8)
    bad = np.flatnonzero(got != want_p)
    assert bad.size == 0, f"{bad.size} packed bytes differ, first at {bad[0]}: got {got.flat[bad[0]]:#04x} want {want_p.flat[bad[0]]:#04x}"


def test_quantize_pack_unaligned_input(oracle_mod):
    rows, k = 6, 72
    x = make_x(rows, k, torch.float16, SEED_BASE + 8100)
    buf = torch.zeros(rows * k + 8, dtype=torch.float16, device=DEV)
    view = buf[1:1 + rows * k].view(rows, k)      # 2-byte aligned only: the element-wise kernel
    view.copy_(x)
    want_p, want_s = oracle_mod.quantize_pack(x.to(torch.float32).numpy())
    packed, scales = qm.quantize_pack(view)
    torch.cuda.synchronize()
    assert (packed.cpu().numpy().view(np.uint8) == want_p).all() and (scales.cpu().numpy() == want_s).all()


# k that is no multiple of 8 (the last chunk of a row overlaps the one before), either side of every change of
# waves per row and chunks per lane, rows around the four of a workgroup
ANY_ROW = [(1, 8), (1025, 10), (1026, 512), (1027, 514), (1025, 1026), (1026, 1536), (1030, 1538), (1024, 514), (3, 2046), (2, 2050), (3, 4098),
           (2, 6146), (3, 8190), (2, 8194), (3, 10242), (2, 12288), (3, 12290), (2, 16382), (3, 16386)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("shape", ANY_ROW, ids=lambda s: "x".join(map(str, s)))
def test_quantize_pack_any_row(oracle_mod, shape, dtype):
    """Input one element and output one byte off alignment, the bytes around the output untouched."""
    rows, k = shape
    x = make_x(rows, k, dtype, SEED_BASE + 8300 + rows + k)
    buf = torch.zeros(rows * k + 1, dtype=dtype, device=DEV)
    buf[1:].copy_(x.reshape(-1))
    out = torch.full((rows * k // 2 + 33,), 0x5A, dtype=torch.uint8, device=DEV)
    scales = torch.empty(rows, device=DEV)
    kind = {torch.float16: 1, torch.bfloat16: 2, torch.float32: 3}[dtype]
    st = qm.library().qm_quantize_pack_i4(buf.data_ptr() + x.element_size(), kind, out.data_ptr() + 17, scales.data_ptr(), rows, k,
                                          torch.cuda.current_stream().cuda_stream)
    assert st == 0
    want_p, want_s = oracle_mod.quantize_pack(x.to(torch.float32).numpy())
    got = out.cpu().numpy()
    assert (got[17:17 + rows * k // 2].reshape(rows, -1) == want_p).all() and (scales.cpu().numpy() == want_s).all()
    assert (got[:17] == 0x5A).all() and (got[17 + rows * k // 2:] == 0x5A).all()


@pytest.mark.parametrize("k", [6, 600, 2600])
def test_quantize_pack_special_values(k):
    """A NaN counts for nothing in a row's maximum and becomes -7; an infinity makes the scale infinite and
    everything finite 0; where 7 / amax overflows the values saturate (and a zero, times infinity, is a NaN)."""
    x = torch.ones((1100, k))
    x[0, 1] = float("nan")
    x[1] = float("nan")
    x[2, 2], x[2, 3] = float("inf"), -2.0
    x[3] = 1e-39
    x[3, 4], x[3, 5] = 0.0, -1e-39
    packed, scales = qm.quantize_pack(x.to(DEV))
    v = qm.unpack_int4(packed).cpu()
    assert v[0, 1] == -7 and (v[0, 2:] == 7).all() and (v[1] == -7).all()
    assert v[2, 2] == -7 and v[2, 3] == 0 and (v[2, 4:] == 0).all()
    assert v[3, 4] == -7 and v[3, 5] == -7 and v[3, 0] == 7
    s = scales.cpu()
    assert s[0] == np.float32(1) / np.float32(7) and s[1] == 0 and s[2] == float("inf")


def test_int4_linear_layer_end_to_end(oracle_mod):
    """activations -> quantize_pack -> gemm_scaled(row_scale = activation scales, col_scale =
    weight scales) against the oracle's chain of the same three steps (bit-exact), and against
    the float product (within the quantisation error)."""
    m, n, k = 96, 320, 1024
    g = torch.Generator().manual_seed(SEED_BASE + 8200)
    x = (torch.randn((m, k), generator=g) * 0.5).to(torch.float16)
    w = (torch.randn((n, k), generator=g) * 0.05).to(torch.float16)
    import quadmul

    xq, xs = quadmul.quantize_pack(x.to(DEV))   # the extension module's entry point
    wq, ws = qm.quantize_pack(w.to(DEV))        # the ctypes binding of the same C function
    y = torch.empty((m, n), dtype=torch.float16, device=DEV)
    qm.gemm_scaled(xq, wq, y, m, n, k, xs, ws)
    torch.cuda.synchronize()
    oxq, oxs = oracle_mod.quantize_pack(x.float().numpy())
    owq, ows = oracle_mod.quantize_pack(w.float().numpy())
    want = oracle_mod.scale_round16(oracle_mod.gemm_i4(oxq, owq), oxs, ows, oracle_mod.OUT_F16)
    assert (y.view(torch.int16).cpu().numpy().view(np.uint16) == want).all()
    ref = x.float() @ w.float().t()
    err = (y.float().cpu() - ref).norm() / ref.norm()
    assert err < 0.25, err  # int4 x int4 with per-row scales: about 15 % relative error on gaussian data


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_w4a4_linear_module(oracle_mod, out_dtype):
    """The module form of the same chain: leading dimensions flattened, weights quantised once,
    bias added to the rounded output; bit-exact against the oracle's chain; no rows -> no launch."""
    from quadmul_amd.linear import W4A4Linear

    n, k = 272, 1056
    g = torch.Generator().manual_seed(SEED_BASE + 8300)
    x = (torch.randn((3, 5, k), generator=g) * 0.7).to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g) * 0.03).to(torch.float32)
    bias = torch.randn((n,), generator=g).to(out_dtype)
    layer = W4A4Linear.from_float(w.to(DEV), bias.to(DEV), out_dtype)
    assert (layer.in_features, layer.out_features) == (k, n) and "bias=True" in repr(layer)
    y = layer(x.to(DEV))
    torch.cuda.synchronize()
    assert y.shape == (3, 5, n) and y.dtype == out_dtype
    oxq, oxs = oracle_mod.quantize_pack(x.reshape(-1, k).float().numpy())
    owq, ows = oracle_mod.quantize_pack(w.numpy())
    out = oracle_mod.OUT_F16 if out_dtype == torch.float16 else oracle_mod.OUT_BF16
    d = oracle_mod.scale_round16(oracle_mod.gemm_i4(oxq, owq), oxs, ows, out)
    want = torch.from_numpy(d.view(np.int16)).view(out_dtype) + bias   # one rounded add in the output type
    assert torch.equal(y.reshape(-1, n).cpu().view(torch.int16), want.view(torch.int16))
    # the state dict round-trips through the constructor's arguments
    again = W4A4Linear(layer.weight_packed, layer.weight_scale, layer.bias, out_dtype)
    assert torch.equal(again(x.to(DEV)), y)
    assert layer(torch.empty((0, k), dtype=torch.float16, device=DEV)).shape == (0, n)
    with pytest.raises(qm.QuadmulError):
        layer(torch.zeros((2, k + 2), dtype=torch.float16, device=DEV))


def test_w4a4_linear_forms_taken_and_refused():
    """The one native call behind the module: every form of input it takes gives the bits of the 2-D contiguous
    one, what does not fit is refused before anything is launched."""
    from quadmul_amd.linear import W4A4Linear

    n, k = 96, 320
    g = torch.Generator().manual_seed(SEED_BASE + 8700)
    w, x = torch.randn((n, k), generator=g).half().to(DEV), torch.randn((6, k), generator=g).half().to(DEV)
    layer = W4A4Linear.from_float(w)
    y = layer(x)
    xq, xs = qm.quantize_pack(x)
    want = torch.empty((6, n), dtype=torch.float16, device=DEV)
    qm.gemm_scaled(xq, layer.weight_packed, want, 6, n, k, xs, layer.weight_scale)
    assert torch.equal(y, want)
    assert torch.equal(layer(x[0]), y[0]) and torch.equal(layer(x.view(2, 3, k)), y.view(2, 3, n))
    assert torch.equal(layer(x.t().contiguous().t()), y) and torch.equal(layer(x[::2]), y[::2])
    assert torch.equal(layer(x.clone().requires_grad_()), y) and not layer(x.clone().requires_grad_()).requires_grad
    assert torch.equal(layer(x.float()), y)
    assert layer(x[:0].view(2, 0, k)).shape == (2, 0, n)
    assert torch.equal(W4A4Linear(layer.weight_packed.view(torch.uint8), layer.weight_scale)(x), y)
    assert torch.equal(torch.compile(layer, backend="aot_eager")(x), y)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        again = layer(x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(again, y)
    for bad in (x.double(), x.to(torch.int8), x.cpu()):
        with pytest.raises(qm.QuadmulError):
            layer(bad)
    halved = W4A4Linear.from_float(w).half()   # the scales are no float32 any more
    with pytest.raises(qm.QuadmulError):
        halved(x)


@pytest.mark.parametrize("found", [None, "foreign"], ids=["no-module", "foreign-module"])
def test_without_the_extension_module(monkeypatch, found):
    """A build of the library alone, and another module of the extension's name on the path: the same kernels
    through ctypes, the same bits."""
    import sys
    import types

    from quadmul_amd.linear import W4A4Linear

    g = torch.Generator().manual_seed(SEED_BASE + 8800)
    w, x = torch.randn((96, 320), generator=g).half().to(DEV), torch.randn((6, 320), generator=g).half().to(DEV)
    v = torch.randint(-8, 8, (5, 34), dtype=torch.int8, generator=g).to(DEV)
    layers = [W4A4Linear.from_float(w, b) for b in (None, torch.randn(96, generator=g).to(DEV))]
    calls = [lambda: qm.quantize_pack(x), lambda: (qm.pack_int4(v), qm.unpack_int4(qm.pack_int4(v))), lambda: [f(x) for f in layers]]
    want = [t for c in calls for t in c()]
    monkeypatch.setattr(qm, "_ext", None)
    monkeypatch.setitem(sys.modules, "quadmul", None if found is None else types.ModuleType("quadmul"))
    got = [t for c in calls for t in c()]
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
    with pytest.raises(qm.QuadmulError):
        layers[0](x.double())


def test_linear_chain_through_dispatcher_ops_traced(oracle_mod):
    """quantize_pack and gemm_scaled as dispatcher ops: the whole linear chain stays in one
    traced graph (aot_eager: fake tensors go through the Meta implementations) and gives the
    oracle's bits."""
    import quadmul  # noqa: F401

    m, n, k = 48, 96, 512
    g = torch.Generator().manual_seed(SEED_BASE + 8400)
    x = (torch.randn((m, k), generator=g) * 0.5).to(torch.float16)
    w = (torch.randn((n, k), generator=g) * 0.05).to(torch.float16)
    wq, ws = torch.ops.quadmul.quantize_pack(w.to(DEV))

    def fn(x_, wq_, ws_):
        xq, xs = torch.ops.quadmul.quantize_pack(x_)
        y = torch.empty((m, n), dtype=torch.float16, device=x_.device)
        torch.ops.quadmul.gemm_scaled(xq, wq_, y, m, n, k, xs, ws_)
        return y

    y = torch.compile(fn, backend="aot_eager", fullgraph=True)(x.to(DEV), wq, ws)
    torch.cuda.synchronize()
    oxq, oxs = oracle_mod.quantize_pack(x.float().numpy())
    owq, ows = oracle_mod.quantize_pack(w.float().numpy())
    want = oracle_mod.scale_round16(oracle_mod.gemm_i4(oxq, owq), oxs, ows, oracle_mod.OUT_F16)
    assert (y.view(torch.int16).cpu().numpy().view(np.uint16) == want).all()
