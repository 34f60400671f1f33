"""The kernel of 3 to 64 rows on both sides of each line of its rules."""
import subprocess

import pytest

import quadmul_amd as qm
from quadmul_amd import build


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


def test_sizes_whose_workgroups_go_round(tmp_path):
    """Sizes of the same kernels that were measured with workgroups that begin at different places of K over all at the same, B from HBM and in the caches."""
    sizes = {
        # 0.88, 0.99; 0.97, 1.02; 0.90, 0.99; 0.85, 0.92; 0.91, 0.97; 0.97, 0.96; 0.99, 1.00; 0.91, 0.71; 0.97, 0.91; 0.99, 0.99; many sizes: 0.96, 0.97; 0.96, 0.99
        True: [(2, 4096, 8192), (1, 2048, 8192), (2, 3584, 8192), (1, 2304, 32768), (16, 4096, 8192), (32, 2048, 8192), (24, 2304, 8192), (56, 4096, 32768), (80, 3072, 32768), (160, 4096, 16384),
               (256, 4096, 8192), (8, 2560, 57344), (64, 3584, 57344)],
        # 1.24, 1.49; 1.15, 1.35; 1.12, 1.21; 1.13, 1.13; 1.04, 1.05; 1.04, 1.06; 1.01, 1.08; many sizes: 0.99, 1.09; 1.00, 1.00; rows that are no whole 4096 bytes
        False: [(233, 7945, 32768), (201, 9667, 32768), (216, 2117, 24576), (149, 3260, 24576), (46, 9903, 32768), (50, 12039, 32768), (47, 9203, 49152), (48, 4097, 57344), (257, 4096, 8192),
                (161, 8200, 16384), (16, 4096, 12288), (16, 4096, 11008)]}
    source = tmp_path / "round.hip"
    source.write_text('#include "qm_common.hpp"\n' + "".join(f"static_assert({'' if yes else '!'}qm::goes_round({m}, {n}, {k}));\n" for yes, of in sizes.items() for m, n, k in of))
    r = subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-host-only", "-fsyntax-only", str(source)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
