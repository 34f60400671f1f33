"""Products whose rows lie off the multiples of four bytes: on the kernel for any address or on padded copies, by sizes that were
measured both ways."""
import pytest

import quadmul_amd as qm


@pytest.mark.parametrize("m,n,k,copied", [
    # time on the kernel for any address over that on the copies
    (17, 3307, 4100, False), (143, 1003, 1788, False), (99, 577, 5058, False), (395, 743, 1266, False), (551, 660, 1210, False),   # 0.58, 0.59, 0.63, 0.77, 0.77
    (89, 622, 8652, True), (133, 413, 8098, True), (122, 435, 7554, True), (87, 2280, 3596, True), (129, 11230, 362, True),                       # 1.20, 1.20, 1.15, 1.10, 1.11
    (216, 8669, 332, True), (85, 2222, 3382, True), (197, 819, 6190, True),                                                     # 1.16, 1.05, 1.07
    # ... and on a B of 40 MB and more
    (7, 44701, 3582, False), (26, 25086, 4630, False), (36, 49813, 9482, False), (59, 22887, 7090, False),                               # 0.59, 0.71, 0.72, 0.90
    (117, 28679, 4998, True), (152, 16876, 6878, True),                                                                                  # 1.25, 1.29
    (470, 33870, 2452, True), (225, 13824, 6110, True),                                                                                 # 1.97, 1.52
    # the last rows that the rule was fitted on, and one more, which would gain as much (B in the caches)
    (1500, 552, 1126, False), (1501, 552, 1126, True)], ids=str)                                                                        # 0.74, 0.73
def test_rows_off_the_multiples_of_four(m, n, k, copied):
    assert (qm.workspace_bytes(m, n, k) > 0) == copied
