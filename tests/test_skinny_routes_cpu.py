"""Layers of 3 to 16 rows: in one launch or in two, by sizes that were measured on both sides of the rule."""
import pytest

from test_routes_cpu import BF16, F16, F32, one_launch


@pytest.mark.parametrize("m,n,k,dtype,one", [
    # time in one launch over that in two, inside a graph with the weights from HBM
    (3, 4096, 4096, F16, True), (4, 12288, 4096, BF16, True), (4, 2144, 6688, BF16, True), (3, 4096, 4096, F32, False),      # 0.73, 0.94, 0.94
    (4, 28640, 864, F16, False), (4, 11264, 8832, F16, False), (4, 4096, 11008, BF16, False),                                 # 1.11, 1.10, 1.15
    (8, 6144, 4096, F16, True), (5, 1120, 2528, BF16, True), (8, 20896, 3968, BF16, False), (7, 2464, 6080, F16, False),      # 0.86, 0.86, 1.08, 1.17
    (16, 2048, 2048, F16, True), (9, 3104, 1056, BF16, True), (13, 4096, 4096, F16, False), (13, 28640, 864, BF16, False),    # 0.92, 0.80, 1.11, 1.34
    (17, 2048, 2048, F16, False), (16, 1000, 2048, F16, False)], ids=str)
def test_linear_layers_of_up_to_sixteen_rows(m, n, k, dtype, one):
    assert one_launch(m, n, k, dtype) == one
