"""The layer's weight, scales and bias as whatever they are by the time of a call: buffers, a parameter in their place, a
parametrization, a plain attribute, other tensors for one call."""
import pytest
import torch

from quadmul_amd.linear import W4A4Linear
from util import SEED_BASE

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def test_what_is_in_place_of_a_buffer_is_used():
    gen = torch.Generator(device=DEV).manual_seed(SEED_BASE + 44000)
    n, k = 64, 256
    w = torch.randn(n, k, device=DEV, generator=gen, dtype=torch.float16)
    x = torch.randn(3, k, device=DEV, generator=gen, dtype=torch.float16)
    b = torch.randn(n, device=DEV, generator=gen, dtype=torch.float16)
    plain, biased = W4A4Linear.from_float(w), W4A4Linear.from_float(w, b)
    y, yb = plain(x), biased(x)
    assert not torch.equal(y, yb)
    plain.bias = b                                                       # another tensor in the same buffer
    assert torch.equal(plain(x), yb)
    plain.bias = torch.nn.Parameter(b.clone(), requires_grad=False)      # a parameter
    assert torch.equal(plain(x), yb)
    del plain.bias
    object.__setattr__(plain, "bias", None)                              # a plain attribute
    assert torch.equal(plain(x), y)

    class Doubled(torch.nn.Module):
        def forward(self, scale):
            return scale * 2

    torch.nn.utils.parametrize.register_parametrization(biased, "weight_scale", Doubled())
    assert torch.equal(biased(x), (y * 2) + b)                           # (twice a scale: no other rounding)
    other = W4A4Linear.from_float(w)
    got = torch.func.functional_call(other, {"bias": b}, (x,))           # for one call
    assert torch.equal(got, yb) and torch.equal(other(x), y)
