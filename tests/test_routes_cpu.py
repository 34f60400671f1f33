"""Which way a call goes where two kernels take it: sizes that were measured on both sides of each rule."""
import pytest

import quadmul_amd as qm

F16, BF16, F32 = 1, 2, 3


def one_launch(m, n, k, dtype):
    return qm.library().qm_linear_workspace_bytes(m, n, k, dtype, 256) == 0


@pytest.mark.parametrize("m,n,k,dtype,one", [
    # time in one launch over that in two, inside a graph with the weights from HBM (; eager, where the host decides)
    (1, 4096, 4096, F32, True), (1, 28672, 4096, BF16, True), (1, 4096, 14336, BF16, True),           # 0.80, 0.92, 0.87
    (1, 8192, 8192, F16, True), (1, 8192, 8192, BF16, False), (1, 10240, 8192, F16, False),           # 0.89, 1.10, 1.07
    (1, 57344, 8192, F16, False), (1, 15610, 8096, F32, False), (1, 25984, 768, F16, False),          # 1.20, 1.23, 1.18
    (1, 11448, 1600, F32, True), (1, 20480, 1024, BF16, True), (1, 65444, 480, F16, False),           # 0.85, 1.09; 0.79, 2
    (2, 4096, 11008, F32, True), (2, 6144, 4096, BF16, True), (2, 6816, 4480, F32, False),            # 0.96, 0.91, 1.31
    (2, 12288, 4096, F16, True), (2, 12288, 4096, BF16, False), (2, 174481, 64, BF16, False),         # 0.97, 1.11, 3.45
    (2, 8000, 896, BF16, True), (2, 11821, 1056, BF16, True), (2, 16384, 1024, BF16, False),          # 0.98, 1.17; 0.80, 1.4
    (2, 12000, 512, F16, False), (3, 64, 64, F16, False)], ids=str)
def test_linear_layers_of_one_or_two_rows(m, n, k, dtype, one):
    assert one_launch(m, n, k, dtype) == one


def recoded(m, n, k, align=256):
    return qm.recode_bytes(m, n, k, ptr_align=align) > 0


@pytest.mark.parametrize("m,n,k,codes", [
    # time on 6-bit operands over that on the int8 choice, B from HBM.  A re-coded from packed rows
    (8192, 8192, 8192, True), (1753, 8192, 8192, True), (3584, 4096, 4096, True), (5601, 2627, 13376, True),       # 0.83, 0.82, 0.94, 0.86
    (2816, 2635, 2112, False), (6912, 5099, 1536, False), (5502, 1139, 4544, False), (964, 7321, 3456, False),   # 1.19, 1.15, 1.14, 1.13
    (830, 5611, 3904, False), (4352, 1472, 17696, False), (2304, 3040, 8224, False), (1280, 4096, 11008, False),   # 1.09, 1.05, 1.05, 1.03
    # both operands copied with padded rows
    (1531, 3307, 4100, True), (2148, 27456, 1370, True), (6954, 1045, 604, False), (5386, 938, 1066, False),        # 0.91, 0.88, 1.27, 1.25
    (1392, 11198, 682, False), (5096, 922, 1388, False), (2375, 3234, 2402, False)], ids=str)                      # 1.23, 1.21, 1.14
def test_large_products_on_6_bit_operands(m, n, k, codes):
    assert recoded(m, n, k) == codes


@pytest.mark.parametrize("m,n,k,codes", [(2048, 11008, 4096, True), (3078, 2368, 4544, True), (4381, 951, 15232, False),          # 0.85, 0.94, 1.18
                                         (3456, 1184, 11488, False), (6168, 1125, 5792, False), (2587, 1792, 13952, False)], ids=str)   # 1.11, 1.07, 1.07
def test_large_layers_on_6_bit_operands(m, n, k, codes):
    """... quantised straight to codes, or by way of packed rows."""
    got = qm.library().qm_linear_workspace_bytes(m, n, k, BF16, 256) - (4 * m + 255) // 256 * 256
    steps = -(-k // 128) + (-(-k // 128) & 1)
    packed = (m * (k // 2) + 255) // 256 * 256
    layout = (m + 31) // 32 * (steps * 3072 + -(-steps // 32) * 32 * 4)
    assert got == (layout if codes else packed + max(qm.workspace_bytes(m, n, k, scaled=True), qm.recode_bytes(m, n, k, True)))


def block(m, n, k):
    """Rows and columns of a block of the wave-level kernel that the call runs on, or None: tiles of the pipelined one."""
    name = qm.config_name(qm.select_config(m, n, k) & 0xFFFF)
    return tuple(16 * int(x) for x in name[1:].split("_")[0].split("x")) if name[0] == "d" else None


@pytest.mark.parametrize("m,n,k,between", [
    (144, 8192, 28672, True), (82, 8192, 28672, True), (105, 4889, 32000, True), (79, 9088, 19168, True),              # 0.65, 0.98, 0.99, 1.02
    (77, 15034, 30944, False), (80, 16074, 28704, False), (95, 8786, 24160, False), (377, 1787, 31040, False),         # 1.23, 1.22, 1.19, 1.09
    (213, 4352, 24928, False), (248, 2445, 25120, False), (93, 8501, 21888, False)], ids=str)                          # 1.09, 1.07, 1.07
def test_blocks_between_32_and_96_rows_on_a_very_long_k(m, n, k, between):
    got = block(m, n, k)
    assert (got is not None and got[0] > 32 and (got[0] % 64 != 0 or got[1] == 48)) == between


@pytest.mark.parametrize("m,k,dtype,esz", [(1, 4096, F16, 2), (2, 2048, BF16, 2), (2, 2048, F32, 4), (4, 4096, F16, 2), (8, 4096, BF16, 2), (16, 2048, F16, 2)], ids=str)
def test_a_layer_that_overwrites_its_rows_is_never_one_launch(m, k, dtype, esz):
    """One launch reads x while it writes D.  (Without the workspace of two launches such a call is refused, whatever part of x it is that D overlaps;
    nothing is enqueued.)"""
    assert one_launch(m, k, k, dtype)
    lib, x, size, out = qm.library(), 1 << 30, m * k * esz, 2 * m * k
    call = lambda d, ws, ws_bytes: lib.qm_linear_i4(x, dtype, 2 << 30, d, m, k, k, None, None, 1, None, ws, ws_bytes)
    need = (4 * m + 255) // 256 * 256 + (m * k // 2 + 255) // 256 * 256
    for d in (x, x + 2, x + size - 2, x - out + 2):
        assert call(d, None, 0) == -7 and call(d, 3 << 30, need - 1) == -7, hex(d)
