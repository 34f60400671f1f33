"""fp16 rows, which are quantised by an arithmetic of their own where they hold no NaN and no infinity (quant8_plain in csrc/qm_aux.hpp)."""
import pytest
import torch

import quadmul

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# every fp16 pattern as an element of rows with a maximum above it, the shorter arithmetic, and of rows with infinities and NaN, the longer
# (k: rows that take the shorter arithmetic only, and rows too short for it)
@pytest.mark.parametrize("k", [8192, 2048])
def test_every_fp16_value_is_quantised_as_the_same_value_in_fp32_is(k):
    for top in (1.0, 7.0, 65504.0, 6.1e-5):
        x = torch.arange(65536, dtype=torch.int32, device=DEV).to(torch.int16).view(torch.float16).view(-1, k).clone()
        special = ~(x.float().abs() <= top)
        finite = torch.where(special, torch.zeros_like(x), x)
        finite[:, 0] = top
        for rows in (finite, x):
            q16, s16 = quadmul.quantize_pack(rows)
            q32, s32 = quadmul.quantize_pack(rows.float())   # (the same values, by the other arithmetic)
            assert torch.equal(q16, q32) and torch.equal(s16.view(torch.int32), s32.view(torch.int32)), top


@pytest.mark.parametrize("rows,k", [(1024, 2048), (1025, 2048), (1025, 510), (256, 4096), (257, 4096), (1025, 2050), (1, 4098), (3, 16384), (2, 16386)], ids=str)
def test_both_sides_of_the_choice_between_the_arithmetics(rows, k):
    x = torch.randn(rows, k, device=DEV, generator=torch.Generator(device=DEV).manual_seed(rows + k)).half()
    x[0, 1], x[rows // 2, k - 1], x[rows - 1, 0] = float("inf"), float("nan"), -0.0
    q16, s16 = quadmul.quantize_pack(x)
    q32, s32 = quadmul.quantize_pack(x.float())
    assert torch.equal(q16, q32) and torch.equal(s16.view(torch.int32), s32.view(torch.int32))
