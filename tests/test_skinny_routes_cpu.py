"""Layers of 3 to 16 rows: in one launch or in two, by sizes that were measured on both sides of the rule."""
import subprocess

import pytest

from quadmul_amd import build
from test_routes_cpu import BF16, F16, F32, one_launch


@pytest.mark.parametrize("m,n,k,dtype,one", [
    # time in one launch over that in two, inside a graph with the weights from HBM
    (3, 4096, 4096, F16, True), (4, 12288, 4096, BF16, True), (4, 2144, 6688, BF16, True), (3, 4096, 4096, F32, False),      # 0.73, 0.94, 0.94
    (4, 28640, 864, F16, False), (4, 11264, 8832, F16, False), (4, 4096, 11008, BF16, False),                                 # 1.11; no kernel holds the other two
    (8, 6144, 4096, F16, True), (5, 1120, 2528, BF16, True), (8, 20896, 3968, BF16, False), (7, 2464, 6080, F16, False),      # 0.86, 0.86, 1.08; no kernel
    (16, 2048, 2048, F16, True), (9, 3104, 1056, BF16, True), (13, 4096, 4096, F16, False), (13, 28640, 864, BF16, False),    # 0.92, 0.80; no kernel; 1.34
    (17, 2048, 2048, F16, False), (16, 1000, 2048, F16, False)], ids=str)
def test_linear_layers_of_up_to_sixteen_rows(m, n, k, dtype, one):
    assert one_launch(m, n, k, dtype) == one


# the longest K that the kernels' registers hold
PROGRAM = r"""
#include "qm_skinny_linear.hpp"
using namespace qm;
static_assert(skinny_linear_fits(16, 2048, QM_IN_F16) && !skinny_linear_fits(16, 2080, QM_IN_F16) && !skinny_linear_fits(9, 2080, QM_IN_BF16));
static_assert(skinny_linear_fits(8, 4096, QM_IN_F16) && !skinny_linear_fits(8, 4128, QM_IN_F16) && !skinny_linear_fits(5, 4128, QM_IN_BF16));
static_assert(skinny_linear_fits(4, 8192, QM_IN_F16) && !skinny_linear_fits(4, 8224, QM_IN_F16) && !skinny_linear_fits(17, 32, QM_IN_F16) && !skinny_linear_fits(4, 32, QM_IN_F32));
constexpr bool whatever_pays_fits()
{
    for (int in : {QM_IN_F16, QM_IN_BF16, QM_IN_F32})
        for (int m = 1; m <= 20; ++m)
            for (int n : {1024, 4096, 8192, 12288, 16384})
                for (int k = 32; k <= 16384; k += 32)
                    if (skinny_linear_pays(m, n, k, in) && !skinny_linear_fits(m, k, in)) return false;
    return true;
}
static_assert(whatever_pays_fits());
"""


def test_layers_that_pay_are_layers_that_fit(tmp_path):
    source = tmp_path / "fits.hip"
    source.write_text(PROGRAM)
    flags = [f for f in build.HIP_FLAGS if f != "-O3"]
    r = subprocess.run([build.HIPCC, *flags, "--cuda-host-only", "-fsyntax-only", "-fconstexpr-steps=100000000", str(source)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
