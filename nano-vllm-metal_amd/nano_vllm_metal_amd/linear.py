"""Quantised weight carrier and the dense W4A16 matmul.

Mirrors layers/linear.py of nano-vllm-metal (reference paths relative to
``src/nano_vllm_metal``): ``QuantizedWeights`` (linear.py:47-70),
``quantized_matmul`` (linear.py:73-89 -> metal/bindings.cpp:16-32) and
``quantized_linear`` (linear.py:92-126), on torch tensors resident on the GPU.

The MLX affine int4 layout is kept as is (no repacking at load time):
``weight`` uint32 ``[..., out, in/8]`` with code j of each word in bits
[4j, 4j+4), ``scales``/``biases`` in the activation dtype ``[..., out, in/group]``,
``w = q * scale + bias``.

``quantize``/``dequantize`` restate MLX's ``mx.quantize``/``mx.dequantize`` in
torch so that synthetic weights can be produced directly on the device (the
reference obtains its weights from MLX); they are layout utilities, not part of
the MoE hot path.
"""

from __future__ import annotations

from typing import Any

import torch

from . import _lib


class QuantizedWeights:
    """The five fields of the reference's ``QuantizedWeights`` (linear.py:47-60)."""

    def __init__(self, scales: torch.Tensor, biases: torch.Tensor, group_size: int, bits: int,
                 weight: torch.Tensor):
        self.scales = scales
        self.biases = biases
        self.group_size = group_size
        self.bits = bits
        self.weight = weight

    @staticmethod
    def from_mlx_layer(layer: Any) -> "QuantizedWeights":
        """Wrap any object with ``scales/biases/group_size/bits/weight`` fields
        (linear.py:62-70); the tensors are referenced, not copied."""
        return QuantizedWeights(scales=layer.scales, biases=layer.biases,
                                group_size=layer.group_size, bits=layer.bits,
                                weight=layer.weight)

    @property
    def in_features(self) -> int:
        return self.weight.shape[-1] * (32 // self.bits)

    @property
    def out_features(self) -> int:
        return self.weight.shape[-2]

    def to(self, device) -> "QuantizedWeights":
        return QuantizedWeights(self.scales.to(device), self.biases.to(device), self.group_size,
                                self.bits, self.weight.to(device))


def _u32_view_as_i32(t: torch.Tensor) -> torch.Tensor:
    return t if t.dtype == torch.int32 else t.view(torch.int32)


def quantize(w: torch.Tensor, group_size: int = 64, bits: int = 4):
    """MLX affine quantisation of ``w[..., n]`` -> ``(wq, scales, biases)``.

    Restates MLX 0.29's affine quantizer: per group the larger-magnitude edge
    is kept exact, the scale is signed so codes stay in [0, 15] and is
    adjusted so zero is representable.  Scales/biases take ``w.dtype``; codes
    are computed against the rounded scale/bias.  ``wq`` is int32 holding the
    uint32 bit patterns (torch has no full uint32 support).
    """
    if bits != 4:
        raise ValueError("only 4-bit quantisation is supported")
    n = w.shape[-1]
    if n % group_size:
        raise ValueError(f"last dim {n} not divisible by group_size {group_size}")
    act = w.dtype
    g = w.float().reshape(*w.shape[:-1], n // group_size, group_size)
    n_bins = float((1 << bits) - 1)
    w_max = g.amax(dim=-1)
    w_min = g.amin(dim=-1)
    mask = w_min.abs() > w_max.abs()
    scales = torch.clamp((w_max - w_min) / n_bins, min=1e-7)
    scales = torch.where(mask, scales, -scales)
    edge = torch.where(mask, w_min, w_max)
    q0 = torch.round(edge / scales)
    nz = q0 != 0
    scales = torch.where(nz, edge / torch.where(nz, q0, torch.ones_like(q0)), scales)
    biases = torch.where(nz, edge, torch.zeros_like(edge))
    scales = scales.to(act)
    scales = torch.where(scales == 0, torch.full_like(scales, 1e-7), scales)
    biases = biases.to(act)
    q = torch.round((g - biases.float()[..., None]) / scales.float()[..., None])
    q = q.clamp_(0, n_bins).to(torch.int64).reshape(*w.shape[:-1], n // 8, 8)
    shifts = torch.arange(0, 32, 4, device=w.device, dtype=torch.int64)
    wq = (q << shifts).sum(dim=-1)
    wq = torch.where(wq >= 2 ** 31, wq - 2 ** 32, wq).to(torch.int32)
    return wq, scales, biases


def dequantize(wq: torch.Tensor, scales: torch.Tensor, biases: torch.Tensor, group_size: int,
               bits: int = 4) -> torch.Tensor:
    """``q * scale + bias`` in float32 (exact), shape ``[..., in]``."""
    if bits != 4:
        raise ValueError("only 4-bit quantisation is supported")
    w = _u32_view_as_i32(wq).to(torch.int64) & 0xFFFFFFFF
    shifts = torch.arange(0, 32, 4, device=w.device, dtype=torch.int64)
    q = ((w[..., None] >> shifts) & 0xF).reshape(*w.shape[:-1], w.shape[-1] * 8).float()
    n = q.shape[-1]
    qg = q.reshape(*q.shape[:-1], n // group_size, group_size)
    out = qg * scales.float()[..., None] + biases.float()[..., None]
    return out.reshape(q.shape)


def quantized_matmul(scales: torch.Tensor, biases: torch.Tensor, group_size: int, bits: int,
                     a: torch.Tensor, b: torch.Tensor, transpose_b: bool = False) -> torch.Tensor:
    """``a[..., N] . dequant(b[K, N/8])^T -> [..., K]`` on the GPU.

    Mirrors linear.py:73-89 / ``_ext.quantized_matmul``: ``transpose_b`` must
    be True (quantized_matmul.cpp:56-58), ``a``, ``scales`` and ``biases`` share
    the f16/bf16 dtype (:26-37).  Router-sized products (up to 512 outputs
    over up to 64 rows) accumulate in float64 and round once to ``a.dtype``;
    the rest run on the expert GEMV or GEMM as a single expert, accumulating
    in float32 like the reference's kernels (quantized_matmul.metal:25-44).
    """
    lib = _lib.load()
    if a.dtype != scales.dtype or scales.dtype != biases.dtype:
        raise ValueError("quantized_matmul: a, scales and biases must share a dtype")
    dev = _lib.require_device(a, b, scales, biases)
    *lead, N = a.shape
    a2 = (a if len(lead) == 1 else a.reshape(-1, N)).contiguous()
    b = _u32_view_as_i32(b).contiguous()
    scales = scales.contiguous()
    biases = biases.contiguous()
    if b.dim() != 2:
        raise ValueError("quantized_matmul: b must be 2-D")
    K = b.shape[0]
    if b.shape[1] * 8 != N or scales.shape != (K, N // group_size) or biases.shape != scales.shape:
        raise ValueError("quantized_matmul: shapes of a, b, scales, biases do not agree")
    out = torch.empty((a2.shape[0], K), dtype=a.dtype, device=dev)
    _lib.check(lib.nvm_quantized_matmul(
        scales.data_ptr(), biases.data_ptr(), group_size, bits, a2.data_ptr(), b.data_ptr(),
        int(bool(transpose_b)), out.data_ptr(), a2.shape[0], N, K, _lib.dtype_code(a.dtype),
        _lib.stream_of(dev)))
    return out if len(lead) == 1 else out.reshape(*lead, K)


def swiglu_supports(x: torch.Tensor, w_gate: QuantizedWeights, w_up: QuantizedWeights) -> bool:
    """Whether ``quantized_swiglu`` takes these operands: one shape, group
    size and dtype for both weights, 32-bit words, and a product that
    ``quantized_matmul`` does not run on its exact float64 path."""
    shape, gs, act, N = w_gate.weight.shape, w_gate.group_size, x.dtype, x.shape[-1]
    if len(shape) != 2 or w_up.weight.shape != shape or w_up.group_size != gs \
            or gs not in (64, 128) or not w_gate.bits == w_up.bits == 4:
        return False
    if not w_gate.weight.element_size() == w_up.weight.element_size() == 4:
        return False  # (the shape below counts 32-bit words)
    K = shape[0]
    if shape[1] * 8 != N or not 0 < N <= 8192 or N % gs or K % 16 or act not in _lib.DTYPE_CODES:
        return False
    per_row = (K, N // gs)
    for t in (w_gate.scales, w_gate.biases, w_up.scales, w_up.biases):
        if t.dtype != act or t.shape != per_row:
            return False
    M = x.numel() // N
    return M > 0 and (K > 512 or M > 64)


def quantized_swiglu(x: torch.Tensor, w_gate: QuantizedWeights, w_up: QuantizedWeights
                     ) -> torch.Tensor:
    """``silu(x . gate^T) * (x . up^T)`` in one launch, each op rounded to
    ``x.dtype`` as the separate products and ``silu`` round it
    (models/qwen3.py:176-184); operands as ``swiglu_supports``."""
    lib = _lib.load()
    if not swiglu_supports(x, w_gate, w_up):
        raise ValueError("quantized_swiglu: operands take two separate products")
    dev = _lib.require_device(x, w_gate.weight, w_gate.scales, w_gate.biases, w_up.weight,
                              w_up.scales, w_up.biases)
    *lead, N = x.shape
    a = x.reshape(-1, N).contiguous()
    gw, uw = _u32_view_as_i32(w_gate.weight).contiguous(), _u32_view_as_i32(w_up.weight).contiguous()
    gsc, gbi = w_gate.scales.contiguous(), w_gate.biases.contiguous()
    usc, ubi = w_up.scales.contiguous(), w_up.biases.contiguous()
    K = gw.shape[0]
    out = torch.empty((a.shape[0], K), dtype=x.dtype, device=dev)
    _lib.check(lib.nvm_quantized_swiglu(
        gsc.data_ptr(), gbi.data_ptr(), gw.data_ptr(), usc.data_ptr(), ubi.data_ptr(),
        uw.data_ptr(), w_gate.group_size, w_gate.bits, a.data_ptr(), out.data_ptr(), a.shape[0],
        N, K, _lib.dtype_code(x.dtype), _lib.stream_of(dev)))
    return out if len(lead) == 1 else out.reshape(*lead, K)


def quantized_linear(x: torch.Tensor, w: QuantizedWeights,
                     bias: torch.Tensor | None = None) -> torch.Tensor:
    """``x . dequant(w)^T (+ bias)`` (linear.py:92-126) through the HIP matmul."""
    out = quantized_matmul(w.scales, w.biases, w.group_size, w.bits, x, w.weight, True)
    if bias is not None:
        out = out + bias
    return out
