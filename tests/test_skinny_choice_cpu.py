"""The kernel of 3 to 64 rows on both sides of each line of its rules."""
import pytest

import quadmul_amd as qm


@pytest.mark.parametrize("m,n,k,int32,scaled", [
    (10, 4448, 6720, "p1x1_w16_r2k2", None), (10, 4096, 6720, "d1x1_w16_r1", None), (10, 5120, 6112, "d1x1_w16_r1", None), (10, 5120, 6144, "p1x1_w16_r2k2", None),
    (16, 4096, 16416, "d1x1_w16_r1", None), (16, 4097, 16416, "d1x2_w8_r2", None), (3, 8193, 20000, "d1x1_w16_r1", None), (3, 12289, 20000, "d1x2_w8_r2", None),
    (17, 2048, 1024, "d1x1_w16_r1", None), (17, 2048, 992, "p2x1_w16_r2k1", None), (17, 2049, 1024, "d1x2_w8_r2", None), (32, 4096, 2016, "d1x2_w8_r2", None),
    (32, 4097, 2016, "p2x1_w16_r2k1", None),
    (32, 16384, 3584, "p2x1_w8_r2k2", None), (32, 16385, 3584, "p2x1_w16_r2k1", None), (32, 20480, 3616, "p2x1_w8_r2k2", None), (32, 20481, 3616, "p2x1_w8_r2k2", "p2x1_w16_r2k1"),
    (17, 22016, 4096, "p2x1_w8_r2k2", "p2x1_w16_r2k1"),
    (32, 8192, 5120, "d2x2_w8_r1", None), (32, 8193, 5120, "d3x3_w8_r1", None), (17, 12288, 5120, "d3x3_w8_r1", None), (17, 12289, 5120, "d2x4_w8_r1", None),
    (32, 16384, 8192, "d2x4_w8_r1", None), (32, 16385, 8192, "d2x2_w8_r1", None),
    (48, 16385, 2048, "d3x3_w8_r1", None), (48, 22529, 2048, "d4x4_w4_r1", None), (59, 12288, 2048, "d4x3_w8_r1", None), (60, 12288, 2048, "d4x4_w8_r1", None)], ids=str)
def test_kernel_by_size(m, n, k, int32, scaled):
    name = lambda as_scaled: qm.config_name(qm.select_config_ex(m, n, k, scaled=as_scaled) & 0xFFFF)
    assert (name(False), name(True)) == (int32, scaled or int32)
