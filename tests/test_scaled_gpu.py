"""GPU parity of the GEMM with the fused dequantising epilogue (scaled fp16 / bf16 output),
called through the C ABI, against the CPU oracle -- bit-exact on the 16-bit patterns."""
import numpy as np
import pytest
import torch

import quadmul_amd as qm
from util import SEED_BASE, make_operands, pack_cpu

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [(torch.float16, 1), (torch.bfloat16, 2)]


def make_scales(m, n, seed):
    g = torch.Generator().manual_seed(seed)
    rs = torch.rand(m, generator=g) * 0.02 + 1e-3   # per-token activation scales
    cs = torch.rand(n, generator=g) * 0.05 + 1e-4   # per-channel weight scales
    return rs.float(), cs.float()


def bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def poisoned_d(m, n, dtype):
    return torch.full((m, n), float("nan"), dtype=dtype, device=DEV)


SHAPES = [(1, 1, 128), (15, 17, 128), (17, 63, 256), (65, 255, 384), (128, 256, 4096), (200, 300, 1152), (257, 511, 256),
          (300, 70, 2048), (3, 5, 30), (70, 33, 162), (64, 64, 96)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_every_scaled_config_matches_oracle(oracle_mod, shape):
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 7000 + m + 3 * n + k)
    ap, bp = pack_cpu(a), pack_cpu(b)
    rs, cs = make_scales(m, n, SEED_BASE + 7100 + m)
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy())
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    ran = 0
    for dtype, out in DTYPES:
        want = oracle_mod.scale_round16(c, rs.numpy(), cs.numpy(), out)
        for cfg, name in enumerate(qm.config_names()):
            if not (qm.config_has_scaled(cfg) and qm.config_supports(cfg, m, n, k)):
                continue
            for gm, spread in [(1, 0), (3, 1)]:
                d = poisoned_d(m, n, dtype)
                qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d, cfg | (gm << 16) | (spread << 30))
                torch.cuda.synchronize()
                got = bits(d)
                bad = np.flatnonzero(got != want)
                assert bad.size == 0, f"{name} {dtype} group_m={gm}: {bad.size} mismatches, first at {bad[0]}: got {got.flat[bad[0]]:#06x} want {want.flat[bad[0]]:#06x}"
            ran += 1
        d = poisoned_d(m, n, dtype)
        qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d)
        torch.cuda.synchronize()
        assert (bits(d) == want).all()
    assert ran >= 2


def test_missing_scales_and_k_zero(oracle_mod):
    m, n, k = 130, 260, 512
    a, b = make_operands(m, n, k, SEED_BASE + 7200)
    ap, bp = pack_cpu(a), pack_cpu(b)
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy())
    rs, cs = make_scales(m, n, SEED_BASE + 7201)
    a_d, b_d = ap.to(DEV), bp.to(DEV)
    for dtype, out in DTYPES:
        for r_, c_ in [(None, None), (rs, None), (None, cs)]:
            d = poisoned_d(m, n, dtype)
            qm.gemm_scaled(a_d, b_d, d, m, n, k, None if r_ is None else r_.to(DEV), None if c_ is None else c_.to(DEV))
            torch.cuda.synchronize()
            want = oracle_mod.scale_round16(c, None if r_ is None else r_.numpy(), None if c_ is None else c_.numpy(), out)
            assert (bits(d) == want).all()
        d = poisoned_d(5, 7, dtype)
        e = torch.empty((5, 0), dtype=torch.int8, device=DEV)
        qm.gemm_scaled(e, torch.empty((7, 0), dtype=torch.int8, device=DEV), d, 5, 7, 0)
        torch.cuda.synchronize()
        assert (bits(d) == 0).all()


def test_rejections():
    m, n, k = 64, 64, 512
    a = torch.zeros((m, k // 2), dtype=torch.int8, device=DEV)
    d = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    names = qm.config_names()
    with pytest.raises(qm.QuadmulError):  # the 256 x 128 tile two to a CU has no scaled output (its registers do not hold the scales)
        qm.gemm_scaled(a, a, d, m, n, k, None, None, names.index("q256x128_w2x2_s3o2"))
    with pytest.raises(qm.QuadmulError):  # partial sums cannot meet in a rounded output: a K split needs a workspace
        qm.gemm_scaled(a, a, d, m, n, k, None, None, names.index("q128x128_w2x2_s7o1") | (2 << 24), workspace=None)
    with pytest.raises(qm.QuadmulError):
        qm.gemm_scaled(a, a, d, m, n, k, None, None, names.index("q128x128_w2x2_s7o1") | (2 << 24),
                       workspace=torch.empty(1024, dtype=torch.uint8, device=DEV))
    with pytest.raises(qm.QuadmulError):  # only the pipelined kernel splits K
        qm.gemm_scaled(a, a, d, m, n, k, None, None, names.index("s4x1_w8_u2") | (2 << 24))
    with pytest.raises(qm.QuadmulError):
        qm.gemm_scaled(a, a, torch.zeros((m, n), dtype=torch.int32, device=DEV), m, n, k)
    with pytest.raises(qm.QuadmulError):
        qm.gemm_scaled(a, a, d, m, n, k, torch.ones(m, dtype=torch.float16, device=DEV))
    lib = qm.library()
    assert lib.qm_gemm_i4_scaled(a.data_ptr(), a.data_ptr(), d.data_ptr(), m, n, k, None, None, 3, None) == -6
    assert lib.qm_gemm_i4_scaled(a.data_ptr(), a.data_ptr(), d.data_ptr() + 1, m, n, k, None, None, 1, None) == -5


BIG = [(4096, 4096, 4096), (2048, 11008, 4096), (16, 4096, 4096), (8000, 4200, 1024), (512, 6144, 4096), (100, 4096, 200)]


@pytest.mark.parametrize("shape", BIG, ids=lambda s: "x".join(map(str, s)))
def test_scaled_large_shapes_every_element(oracle_mod, shape):
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 7300 + m)
    ap, bp = pack_cpu(a), pack_cpu(b)
    rs, cs = make_scales(m, n, SEED_BASE + 7301)
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    c_d = torch.empty((m, n), dtype=torch.int32, device=DEV)
    qm.gemm(a_d, b_d, c_d, m, n, k)  # the int32 path has its own parity tests
    rows = np.unique(np.concatenate([np.arange(0, m, max(1, m // 23)), [m - 1]])).astype(np.int32)
    c_rows = oracle_mod.gemm_i4_rows(ap.numpy(), bp.numpy(), rows)
    assert (c_d.cpu().numpy()[rows] == c_rows).all()
    for dtype, out in DTYPES:
        d = poisoned_d(m, n, dtype)
        qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d)
        torch.cuda.synchronize()
        # every element: the same two float32 multiplications and the same rounding, by torch on the GPU
        want_d = ((c_d.to(torch.float32) * rs_d[:, None]) * cs_d[None, :]).to(dtype)
        assert torch.equal(d.view(torch.int16), want_d.view(torch.int16))
        # sampled rows against the oracle
        want = oracle_mod.scale_round16(c_rows, rs.numpy()[rows], cs.numpy(), out)
        assert (bits(d)[rows] == want).all()


def test_extension_module_and_dispatcher_op(oracle_mod):
    import quadmul

    m, n, k = 200, 264, 640
    a, b = make_operands(m, n, k, SEED_BASE + 7400)
    ap, bp = pack_cpu(a), pack_cpu(b)
    rs, cs = make_scales(m, n, SEED_BASE + 7401)
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy())
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    for dtype, out in DTYPES:
        want = oracle_mod.scale_round16(c, rs.numpy(), cs.numpy(), out)
        d = poisoned_d(m, n, dtype)
        quadmul.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d)
        torch.cuda.synchronize()
        assert (bits(d) == want).all()
        d2 = poisoned_d(m, n, dtype)
        torch.ops.quadmul.gemm_scaled(a_d, b_d, d2, m, n, k, rs_d, cs_d)

        def fn(x, y, r, s_):
            o = torch.full((m, n), float("nan"), dtype=dtype, device=x.device)
            torch.ops.quadmul.gemm_scaled(x, y, o, m, n, k, r, s_)
            return o

        d3 = torch.compile(fn, backend="aot_eager", fullgraph=True)(a_d, b_d, rs_d, cs_d)
        torch.cuda.synchronize()
        assert (bits(d2) == want).all() and (bits(d3) == want).all()
        # captured and replayed, every replay checked
        d4 = poisoned_d(m, n, dtype)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            quadmul.gemm_scaled(a_d, b_d, d4, m, n, k, rs_d, cs_d)
        for _ in range(3):
            d4.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert (bits(d4) == want).all()
    with pytest.raises(RuntimeError):
        quadmul.gemm_scaled(a_d, b_d, torch.zeros((m, n), dtype=torch.float32, device=DEV), m, n, k)


@pytest.mark.parametrize("shape", [(128, 1024, 14336), (200, 300, 2048), (257, 511, 1280)], ids=lambda s: "x".join(map(str, s)))
def test_scaled_with_k_split_through_a_workspace(oracle_mod, shape):
    """With a workspace the scaled form takes K splits on every pipelined configuration: the
    int32 partial tiles are added up, scaled and rounded by the second kernel."""
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 7300 + m)
    ap, bp = pack_cpu(a), pack_cpu(b)
    rs, cs = make_scales(m, n, SEED_BASE + 7400 + m)
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy())
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    ran = 0
    for dtype, out in DTYPES:
        want = oracle_mod.scale_round16(c, rs.numpy(), cs.numpy(), out)
        want_rows_only = oracle_mod.scale_round16(c, rs.numpy(), None, out)
        for cfg, name in enumerate(qm.config_names()):
            if not name.startswith("q") or not qm.config_supports(cfg, m, n, k):
                continue
            for gm, ks in [(1, 2), (3, 5)]:
                code = cfg | (gm << 16) | (ks << 24)
                assert qm.workspace_bytes(m, n, k, code, scaled=True) > 0
                d = poisoned_d(m, n, dtype)
                qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d, code)
                torch.cuda.synchronize()
                got = bits(d)
                bad = np.flatnonzero(got != want)
                assert bad.size == 0, f"{name} {dtype} group_m={gm} ksplit={ks}: {bad.size} mismatches, first at {bad[0]}"
            d = poisoned_d(m, n, dtype)
            qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, None, cfg | (4 << 24))
            torch.cuda.synchronize()
            assert (bits(d) == want_rows_only).all(), name
            ran += 1
    assert ran >= 8


def test_scaled_random_shapes_through_the_automatic_choice():
    """The same sweep for the scaled output, against torch's float32 arithmetic on the exact
    int32 product (two separate float32 multiplications, then torch's rounding to 16 bits)."""
    rng = np.random.default_rng(SEED_BASE + 7500)
    for i in range(80):
        m = int(np.exp(rng.uniform(0, np.log(1200)))) if i % 3 else int(rng.integers(1, 140))
        n = int(np.exp(rng.uniform(0, np.log(5000))))
        k = int(np.exp(rng.uniform(np.log(2), np.log(12000))))
        k = max(2, [k // 128 * 128, k // 32 * 32, k // 2 * 2, k // 128 * 128][i % 4])
        if i % 8 == 0:
            m, k = int(rng.integers(65, 129)), int(rng.integers(16, 96)) * 128
        a = torch.randint(-8, 8, (m, k), dtype=torch.int8, generator=torch.Generator().manual_seed(3000 + i))
        b = torch.randint(-8, 8, (n, k), dtype=torch.int8, generator=torch.Generator().manual_seed(4000 + i))
        rs, cs = make_scales(m, n, 5000 + i)
        a_d, b_d, rs_d, cs_d = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV), rs.to(DEV), cs.to(DEV)
        c32 = (a.to(DEV).float() @ b.to(DEV).float().t())   # exact integers in fp32
        dtype = torch.float16 if i % 2 else torch.bfloat16
        want = ((c32 * rs_d[:, None]) * cs_d[None, :]).to(dtype)
        d = poisoned_d(m, n, dtype)
        qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d)
        torch.cuda.synchronize()
        assert torch.equal(d.view(torch.int16), want.view(torch.int16)), f"{m}x{n}x{k} {dtype}"


def test_scaled_k_padded_through_the_workspace():
    m, n, k = 3000, 3000, 1058
    a = torch.randint(-8, 8, (m, k), dtype=torch.int8, generator=torch.Generator().manual_seed(SEED_BASE + 7600))
    b = torch.randint(-8, 8, (n, k), dtype=torch.int8, generator=torch.Generator().manual_seed(SEED_BASE + 7700))
    rs, cs = make_scales(m, n, SEED_BASE + 7800)
    a_d, b_d, rs_d, cs_d = pack_cpu(a).to(DEV), pack_cpu(b).to(DEV), rs.to(DEV), cs.to(DEV)
    c32 = a.to(DEV).float() @ b.to(DEV).float().t()
    assert qm.workspace_bytes(m, n, k, scaled=True) > 0
    for dtype in (torch.float16, torch.bfloat16):
        want = ((c32 * rs_d[:, None]) * cs_d[None, :]).to(dtype)
        for ws in (True, None):
            d = poisoned_d(m, n, dtype)
            qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d, workspace=ws)
            torch.cuda.synchronize()
            assert torch.equal(d.view(torch.int16), want.view(torch.int16)), (dtype, ws)


@pytest.mark.parametrize("shape", [(700, 1300, 512), (1290, 520, 384), (2100, 2052, 256 + 32), (300, 4100, 1024)], ids=lambda s: "x".join(map(str, s)))
def test_tiles_that_stick_out_of_c_on_every_pipelined_configuration(oracle_mod, shape):
    """N % 4 == 0 and an aligned C: whole tiles and tiles that stick out of the matrix (a
    ragged bottom row, a ragged right column, the corner) in one launch, several items per
    workgroup -- the write-out inside the last K-step with its stores under lane masks --
    for the int32 output and both 16-bit ones, with and without the one-item-per-workgroup
    launch, against the oracle; and the memory around C and D stays as it was."""
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 7600 + m)
    ap, bp = pack_cpu(a), pack_cpu(b)
    rs, cs = make_scales(m, n, SEED_BASE + 7700 + m)
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy())
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    want16 = {out: oracle_mod.scale_round16(c, rs.numpy(), cs.numpy(), out) for _, out in DTYPES}
    pad = 4096    # elements either side of the output that must not change
    ran = 0
    for cfg, name in enumerate(qm.config_names()):
        if not name.startswith("q") or not qm.config_supports(cfg, m, n, k):
            continue
        bm, bn = (int(x) for x in name[1:].split("_")[0].split("x"))
        assert m % bm or n % bn, (name, shape)          # (some tile sticks out)
        for gm, spread in [(1, 0), (4, 0), (2, 1)]:
            code = cfg | (gm << 16) | (spread << 30)
            buf = torch.full((m * n + 2 * pad,), 0x7F7F7F7F, dtype=torch.int32, device=DEV)
            c_d = buf[pad:pad + m * n].view(m, n)
            qm.gemm_cfg(a_d, b_d, c_d, m, n, k, code)
            torch.cuda.synchronize()
            bad = oracle_mod.compare(c_d.cpu().numpy(), c)
            assert bad == -1, f"{name} group_m={gm} spread={spread}: first mismatch at flat index {bad} (row {bad // n}, column {bad % n})"
            assert (buf[:pad] == 0x7F7F7F7F).all() and (buf[pad + m * n:] == 0x7F7F7F7F).all(), name
            if not qm.config_has_scaled(cfg):
                continue
            for dtype, out in DTYPES:
                buf16 = torch.full((m * n + 2 * pad,), float("nan"), dtype=dtype, device=DEV)
                d_d = buf16[pad:pad + m * n].view(m, n)
                qm.gemm_scaled(a_d, b_d, d_d, m, n, k, rs_d, cs_d, code)
                torch.cuda.synchronize()
                assert (bits(d_d) == want16[out]).all(), f"{name} {dtype} group_m={gm} spread={spread}"
                assert torch.isnan(buf16[:pad]).all() and torch.isnan(buf16[pad + m * n:]).all(), name
        ran += 1
    assert ran >= 8


# N % 4 = 1, 2, 3, and N % 4 == 0 with C itself off; N a multiple of no tile, one column more than one, less than one
UNALIGNED_C = [((700, 1301, 512), 0), ((512, 1026, 384), 0), ((1290, 519, 256 + 32), 3), ((300, 4097, 1024), 1), ((257, 130, 640), 0), ((520, 65, 256), 0),
               ((200, 63, 384), 0), ((512, 512, 384), 1)]


@pytest.mark.parametrize("shape,off", UNALIGNED_C, ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else f"off{s}")
def test_unaligned_rows_of_c_on_every_pipelined_configuration(oracle_mod, shape, off):
    """The right column of tiles moved left to end where C does, int32 and both 16-bit outputs, these with and
    without a bias, against the oracle; and the memory around the output stays as it was."""
    m, n, k = shape
    a, b = make_operands(m, n, k, SEED_BASE + 8600 + m + n)
    ap, bp = pack_cpu(a), pack_cpu(b)
    rs, cs = make_scales(m, n, SEED_BASE + 8700 + m)
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy())
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    pad = 4096
    ran = 0
    for cfg, name in enumerate(qm.config_names()):
        if not name.startswith("q") or not qm.config_supports(cfg, m, n, k):
            continue
        for gm, spread in [(4, 0), (2, 1)]:
            code = cfg | (gm << 16) | (spread << 30)
            buf = torch.full((m * n + 2 * pad,), 0x7F7F7F7F, dtype=torch.int32, device=DEV)
            at = pad + off
            qm.gemm_cfg(a_d, b_d, buf[at:at + m * n].view(m, n), m, n, k, code)
            torch.cuda.synchronize()
            bad = oracle_mod.compare(buf[at:at + m * n].view(m, n).cpu().numpy(), c)
            assert bad == -1, f"{name} group_m={gm} spread={spread}: first mismatch at row {bad // n}, column {bad % n}"
            assert (buf[:at] == 0x7F7F7F7F).all() and (buf[at + m * n:] == 0x7F7F7F7F).all(), name
            if not qm.config_has_scaled(cfg):
                continue
            for dtype, out in DTYPES:
                want = torch.from_numpy(oracle_mod.scale_round16(c, rs.numpy(), cs.numpy(), out).view(np.int16)).view(dtype)
                bias = torch.randn(n, generator=torch.Generator().manual_seed(SEED_BASE + n)).to(dtype)
                for bias_d, w in ((None, want), (bias.to(DEV), want + bias)):
                    buf16 = torch.full((m * n + 2 * pad,), float("nan"), dtype=dtype, device=DEV)
                    d_d = buf16[at:at + m * n].view(m, n)
                    qm.gemm_scaled(a_d, b_d, d_d, m, n, k, rs_d, cs_d, code, bias=bias_d)
                    torch.cuda.synchronize()
                    assert torch.equal(d_d.cpu().view(torch.int16), w.view(torch.int16)), f"{name} {dtype} group_m={gm} spread={spread} bias={bias_d is not None}"
                    assert torch.isnan(buf16[:at]).all() and torch.isnan(buf16[at + m * n:]).all(), name
        ran += 1
    assert ran >= 8


# every epilogue: the dot, wave-level and persistent kernels (1 to 64 rows), the kernels for any address and
# one thread per element (K % 32), each tile through its own way of writing whole tiles,
# tiles that stick out of C, odd N, a short last K-step, a K split added up out of a workspace, k = 0,
# several blocks of columns per workgroup of the persistent kernel with the last one cut short
BIAS_SHAPES = [(1, 33, 256), (2, 64, 4096), (9, 130, 8192), (40, 96, 1152), (70, 33, 162), (2048, 520, 130), (256, 512, 256), (520, 780, 384),
               (300, 1021, 416), (257, 258, 640), (6, 10, 0), (5, 8263, 384)]
# ... and zero-padded copies, the second time where the configuration that int32 takes on them has no scaled output
COPIED_SHAPES = [(300, 1021, 4100), (1518, 4099, 506)]
BIAS_SHAPES += COPIED_SHAPES


@pytest.mark.parametrize("shape", BIAS_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_bias_in_every_epilogue(oracle_mod, shape):
    """The bias added in the epilogue gives, bit for bit, the rounded value plus the bias rounded
    once more; without one, a zero with a negative scale stays -0."""
    m, n, k = shape
    if shape in COPIED_SHAPES:
        kp = (k + 127) // 128 * 128
        assert qm.workspace_bytes(m, n, k, scaled=True) >= (m + n) * kp // 2
        alike = qm.library().qm_select_config_ex(m, n, kp, 256, 0, 0) & 0xFFFF
        assert qm.config_has_scaled(alike) == (shape == COPIED_SHAPES[0]), qm.config_name(alike)
    a, b = make_operands(m, n, max(k, 2), SEED_BASE + 7600 + m + n + k)
    ap, bp = pack_cpu(a), pack_cpu(b)
    if k == 0:
        ap, bp = ap[:, :0].contiguous(), bp[:, :0].contiguous()
    ap[0] = 0                                        # zero products: -0 under the negative scales
    rs, cs = make_scales(m, n, SEED_BASE + 7601 + m)
    cs[::3] *= -1
    c = oracle_mod.gemm_i4(ap.numpy(), bp.numpy()) if k else np.zeros((m, n), np.int32)
    a_d, b_d, rs_d, cs_d = ap.to(DEV), bp.to(DEV), rs.to(DEV), cs.to(DEV)
    for dtype, out in DTYPES:
        bias = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(dtype)
        bias[1::5] = 0.0
        bias[2::5] = -0.0
        plain = torch.from_numpy(oracle_mod.scale_round16(c, rs.numpy(), cs.numpy(), out).view(np.int16)).view(dtype) if k else torch.zeros((m, n), dtype=dtype)
        want = plain + bias
        codes = [qm.CFG_AUTO]
        if k:
            for cfg in range(qm.num_configs()):
                if qm.config_supports(cfg, m, n, k) and qm.config_has_scaled(cfg):
                    codes.append(cfg | (2 << 16))
                    if k >= 640 and qm.config_name(cfg).startswith("q"):
                        codes.append(cfg | (2 << 16) | (2 << 24))
        for code in codes:
            name = "auto" if code < 0 else qm.config_name(code & 0xFFFF)
            for b_, w_ in ((bias.to(DEV), want), (None, plain)):
                d = poisoned_d(m, n, dtype)
                qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d, code, bias=b_)
                torch.cuda.synchronize()
                assert (bits(d) == bits(w_)).all(), (name, code >> 16, dtype, b_ is None)
    with pytest.raises(qm.QuadmulError):
        qm.gemm_scaled(a_d, b_d, d, m, n, k, rs_d, cs_d, bias=torch.zeros(n + 1, dtype=d.dtype, device=DEV))


def test_bf16_rounding_of_every_float():
    """What the pipelined kernel's write-out makes of each of the 2^32 floats (a product of 1, the float its row's scale):
    round to nearest even by the integer rule, a NaN its upper half with the quiet bit."""
    rows, cfg = 1 << 22, qm.config_id("q64x64_w2x2_s8o2")
    a, b = torch.zeros((rows, 64), dtype=torch.int8, device=DEV), torch.zeros((4, 64), dtype=torch.int8, device=DEV)
    a[:, 0] = b[:, 0] = 1
    d = torch.empty((rows, 4), dtype=torch.bfloat16, device=DEV)
    for first in range(-(1 << 31), 1 << 31, rows):
        x = torch.arange(first, first + rows, dtype=torch.int64, device=DEV)
        qm.gemm_scaled(a, b, d, rows, 4, 128, x.to(torch.int32).view(torch.float32), None, cfg)
        u = x & 0xFFFFFFFF
        want = torch.where((u & 0x7FFFFFFF) > 0x7F800000, (u >> 16) | 0x40, (u + 0x7FFF + ((u >> 16) & 1)) >> 16)
        assert torch.equal(d.view(torch.int16).long() & 0xFFFF, want[:, None].expand(rows, 4)), hex(first & 0xFFFFFFFF)


def test_linear_bias_that_the_kernel_cannot_take(oracle_mod):
    """A bias that autograd follows, or of another type than the output, is added apart as ever."""
    from quadmul_amd.linear import W4A4Linear

    n, k = 64, 256
    g = torch.Generator().manual_seed(SEED_BASE + 7700)
    w, x = torch.randn((n, k), generator=g).to(DEV), torch.randn((3, k), generator=g).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    layer = W4A4Linear.from_float(w, bias)
    y = layer(x)
    layer.bias = layer.bias.clone().requires_grad_(True)
    z = layer(x)
    assert z.requires_grad and torch.equal(z.detach(), y)
    z.float().sum().backward()
    assert torch.equal(layer.bias.grad, torch.full((n,), 3.0, dtype=torch.float16, device=DEV))
    layer.bias = bias                                # float32 beside a float16 output
    bare = W4A4Linear(layer.weight_packed, layer.weight_scale)(x)
    bare += bias
    assert torch.equal(layer(x), bare)
