"""A W4A4 linear layer on top of the packed-int4 GEMM: the caller the reference's README
(README.md:7, "easy to fuse with quantisation") has in mind and does not ship.

    y[t, n] = round16((sum_k xq[t, k] * wq[n, k]) * x_scale[t] * w_scale[n]) (+ bias[n])

with ``xq, x_scale = quantize_pack(x)`` (per-token symmetric int4, scale = amax / 7) and
``wq, w_scale`` the same quantisation of the weight rows, done once.  One or two launches out of one native
call: quantise + pack the activations, and the GEMM with the dequantising epilogue, which adds
the bias too; the int32 product never reaches memory.
"""
from __future__ import annotations

from typing import Optional

import torch
from torch.autograd import forward_ad

from . import QuadmulError, _native, gemm_scaled, quantize_pack


def _fusable(bias: torch.Tensor, x: torch.Tensor, out_dtype: torch.dtype, n: int) -> bool:
    return (type(bias) in (torch.Tensor, torch.nn.Parameter) and bias.layout is torch.strided and not bias.requires_grad and not bias.is_neg()
            and bias.dtype == out_dtype and bias.device == x.device and bias.shape == (n,) and bias.is_contiguous()
            and forward_ad._current_level < 0)


class W4A4Linear(torch.nn.Module):
    """``forward(x)``: ``x`` [..., in_features] float16 / bfloat16 / float32 on the GPU ->
    [..., out_features] in ``out_dtype`` (float16 or bfloat16)."""

    def __init__(self, weight_packed: torch.Tensor, weight_scale: torch.Tensor, bias: Optional[torch.Tensor] = None,
                 out_dtype: torch.dtype = torch.float16):
        super().__init__()
        if weight_packed.dim() != 2 or weight_packed.dtype not in (torch.int8, torch.uint8):
            raise QuadmulError("W4A4Linear: weight_packed must be [out_features, in_features / 2] int8 or uint8")
        if out_dtype not in (torch.float16, torch.bfloat16):
            raise QuadmulError("W4A4Linear: out_dtype must be float16 or bfloat16")
        n = weight_packed.shape[0]
        if weight_scale.shape != (n,) or weight_scale.dtype != torch.float32:
            raise QuadmulError("W4A4Linear: weight_scale must be float32 [out_features]")
        if bias is not None and bias.shape != (n,):
            raise QuadmulError("W4A4Linear: bias must be [out_features]")
        self.out_features = n
        self.in_features = weight_packed.shape[1] * 2
        self.out_dtype = out_dtype
        self.register_buffer("weight_packed", weight_packed.contiguous())
        self.register_buffer("weight_scale", weight_scale.contiguous())
        self.register_buffer("bias", None if bias is None else bias.to(out_dtype).contiguous())

    @classmethod
    def from_float(cls, weight: torch.Tensor, bias: Optional[torch.Tensor] = None, out_dtype: torch.dtype = torch.float16):
        """Quantise a float [out_features, in_features] weight (on the GPU) row by row with the
        library's own kernel: the same rule as for the activations."""
        wq, ws = quantize_pack(weight.contiguous())
        return cls(wq, ws, bias, out_dtype)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        in_features = self.in_features
        if x.shape[-1] != in_features:
            raise QuadmulError(f"W4A4Linear: last dimension of x must be {in_features}")
        flat = x.dim() == 2 and in_features > 0
        x2 = x if flat else x.reshape(-1, in_features)
        if not x2.is_contiguous():
            x2 = x2.contiguous()
        if x2.shape[0]:
            out_dtype = self.out_dtype
            bf16 = out_dtype is torch.bfloat16
            if not bf16 and out_dtype is not torch.float16:
                raise QuadmulError("W4A4Linear: out_dtype must be float16 or bfloat16")
            # (out of the dictionary: an attribute that is a buffer is found after everything else has been looked through, 0.28 us each of the
            # 6.2 of a small call.  Only where nothing would be found ahead of it -- not in a subclass, nor with an attribute of that
            # name beside the buffer, on the layer or on the class.  One that is no buffer any more -- replaced by a parameter,
            # parametrized -- is looked up as ever)
            own = self.__dict__
            shadowed = (type(self) is not W4A4Linear or "weight_packed" in own or "weight_scale" in own or "bias" in own
                        or "weight_packed" in _CLASS or "weight_scale" in _CLASS or "bias" in _CLASS)
            held = {} if shadowed else own["_buffers"]
            try:
                weight, weight_scale, bias = held["weight_packed"], held["weight_scale"], held["bias"]
            except KeyError:
                weight, weight_scale, bias = self.weight_packed, self.weight_scale, self.bias
            # in the GEMM's epilogue: a separate addition reads and writes all of y once more
            # (2048 x 11008: 21 us beside a GEMM of 73).  A bias that the kernel cannot take as
            # it is -- moved or cast after construction -- or that autograd follows is added apart.
            fused = bias is not None and _fusable(bias, x2, out_dtype, self.out_features)
            y = _native("linear", x2, weight, self.out_features, weight_scale, bias if fused else None, bf16)
            if y is None:
                y = torch.empty((x2.shape[0], self.out_features), dtype=out_dtype, device=x.device)
                xq, xs = quantize_pack(x2)
                gemm_scaled(xq, weight, y, x2.shape[0], self.out_features, self.in_features, xs, weight_scale,
                            bias=bias if fused else None)
            if bias is not None and not fused:
                y += bias
        else:
            y = torch.empty((0, self.out_features), dtype=self.out_dtype, device=x.device)
        return y if flat else y.reshape(*x.shape[:-1], self.out_features)

    def extra_repr(self) -> str:
        return f"in_features={self.in_features}, out_features={self.out_features}, bias={self.bias is not None}, out_dtype={self.out_dtype}"


_CLASS = W4A4Linear.__dict__  # (as it is at the time of a call)
