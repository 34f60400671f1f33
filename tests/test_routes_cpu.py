"""Which way a call goes where two kernels take it: sizes that were measured on both sides of each rule."""
import pytest

import quadmul_amd as qm

F16, BF16, F32 = 1, 2, 3


def one_launch(m, n, k, dtype):
    return qm.library().qm_linear_workspace_bytes(m, n, k, dtype, 256) == 0


@pytest.mark.parametrize("m,n,k,dtype,one", [
    # time in one launch over that in two, inside a graph with the weights from HBM
    (1, 4096, 4096, F32, True), (1, 28672, 4096, BF16, True), (1, 4096, 14336, BF16, True),           # 0.80, 0.92, 0.87
    (1, 8192, 8192, F16, True), (1, 8192, 8192, BF16, False), (1, 10240, 8192, F16, False),           # 0.89, 1.10, 1.07
    (1, 57344, 8192, F16, False), (1, 15610, 8096, F32, False), (1, 25984, 768, F16, False),          # 1.20, 1.23, 1.18
    (1, 11448, 1600, F32, True), (1, 15264, 1024, F32, False), (1, 16352, 1024, F16, True),           # 0.85, 1.05, 0.96
    (2, 4096, 11008, F32, True), (2, 6144, 4096, BF16, True), (2, 6816, 4480, F32, False),            # 0.96, 0.91, 1.31
    (2, 12288, 4096, F16, True), (2, 12288, 4096, BF16, False), (2, 174481, 64, BF16, False),         # 0.97, 1.11, 3.45
    (2, 8000, 896, BF16, True), (2, 11821, 1056, BF16, False), (3, 64, 64, F16, False)], ids=str)     # 0.98, 1.17
def test_linear_layers_of_one_or_two_rows(m, n, k, dtype, one):
    assert one_launch(m, n, k, dtype) == one
