"""``ARCQPackedLinearOnTheFly``: the packed on-the-fly layer (the path the reference's README
benchmarks), constructor and buffers as FQ/arcq_packed_on_the_fly.py:93-135.

Reference forward (:137-161): fp16 copy of x -> Triton quantize+reconstruct in place -> Triton
unpack of the whole weight into an fp16 buffer in HBM -> cuBLAS ``F.linear``.  Here the layer is one
or two HIP launches: ``arcq_linear_otf_ws`` / ``arcq_linear_otf_ex``, or ``arcq_prepare`` (stage 1 and the
weights in one launch) and ``arcq_linear_prepared`` (the product), whichever is faster for the sizes
(the rule and its figures: ``prepare_pays`` in csrc_host/arcq_host.cpp).  x_hat (fp16) lies in a workspace or
in LDS, and so do the dense fp16 weights:
  * below 512 rows and 768 inputs they are rebuilt tile by tile in LDS and never exist in memory;
  * else they are reconstructed in the layer's first (or only) launch and pass through memory (L2-resident, a
    few MB) -- the reference's unpack-then-GEMM order without a launch of its own -- in ``_weight_buffer`` where
    that is set (the flat fp16 scratch the reference's benchmark shares between all layers,
    scripts/benchmark_arcq_on_the_fly.py:182-191, read at :148-158; ``packed_convert.share_buffers`` sets it),
    otherwise in scratch of the call's own.  The one-launch kernels from 512 rows on run only with it.
The result is bit-identical either way.

Differences from the reference module that a caller can observe (all on the side of more accuracy;
for these cases "same indices as the reference" is not pinned by any test):
  * the input tensor is never overwritten (the reference overwrites a contiguous fp16 input);
  * group statistics are taken in fp32 even for fp16 input (the Triton kernel reduces in fp16);
  * an fp32 input is quantized from its fp32 values (the reference first casts x to fp16, :139);
  * the bias is added in fp32 before the one output rounding (the reference rounds the bias to fp16);
  * ``model.half()`` leaves the fp32 metadata (codebooks, thresholds, center/scale/code_sum, bias)
    at their fp32 values (the reference's half chain leaves them rounded to fp16).
"""
from __future__ import annotations

from typing import Optional

import torch
import torch.nn as nn

from . import _lib, ops


def clear_workspaces() -> None:
    """Kept for callers of earlier versions: scratch tensors come from torch's caching allocator call by call, so there is
    nothing to drop (``torch.cuda.empty_cache()`` returns the memory)."""


class ARCQPackedLinearOnTheFly(nn.Module):
    """Stores packed codes + codebooks + per-group metadata + bias only (no dense weight)."""

    def __init__(self, in_features: int, out_features: int, bias: bool,
                 packed_weight_codes: torch.Tensor, weight_codebook: torch.Tensor,
                 weight_center: torch.Tensor, weight_scale: torch.Tensor, weight_code_sum: torch.Tensor,
                 activation_codebook: torch.Tensor, activation_thresholds: torch.Tensor,
                 bits: int, group_size: int, bias_tensor: Optional[torch.Tensor]):
        super().__init__()
        self.in_features = int(in_features)
        self.out_features = int(out_features)
        self.bits = int(bits)
        self.group_size = int(group_size)
        self.groups = self.in_features // self.group_size
        if self.bits not in (2, 3, 4):
            raise ValueError(f"packed kernel supports bits 2/3/4, got {self.bits}")
        if self.in_features % self.group_size != 0:
            raise ValueError(f"in_features={self.in_features} must be divisible by group_size={self.group_size}")
        if tuple(packed_weight_codes.shape) != (self.out_features, (self.in_features * self.bits + 7) // 8):
            raise ValueError(f"packed_weight_codes has shape {tuple(packed_weight_codes.shape)}, expected "
                             f"{(self.out_features, (self.in_features * self.bits + 7) // 8)}")
        self.register_buffer("packed_weight_codes", packed_weight_codes)
        self.register_buffer("weight_codebook", weight_codebook)
        self.register_buffer("weight_center", weight_center)
        self.register_buffer("weight_scale", weight_scale)
        self.register_buffer("weight_code_sum", weight_code_sum)
        self.register_buffer("activation_codebook", activation_codebook)
        self.register_buffer("activation_thresholds", activation_thresholds)
        if bias and bias_tensor is not None and bias_tensor.numel() > 0:
            self.register_buffer("bias_tensor", bias_tensor)
        else:
            self.register_buffer("bias_tensor", torch.empty(0))
        self.out_dtype = torch.float16
        self._host_plan = None      # the host extension's view of the buffers above, made by the first forward
        self._fp8_mult = None       # what _fp8_multiplier keeps (without the extension)
        # Opt-in: operands rounded to FP8 and the product on FP8 matrix units (ops.linear_otf_fp8).  Faster on the
        # large models, not the reference's numerics; see set_fp8_operands in packed_convert.
        self.fp8_operands = False

    @classmethod
    def from_packed(cls, packed_layer: nn.Module) -> "ARCQPackedLinearOnTheFly":
        """From an ``ARCQPackedLinear`` (what scripts/benchmark_arcq_on_the_fly.py:151-170 does)."""
        b = packed_layer.bias if packed_layer.bias.numel() > 0 else None
        return cls(packed_layer.in_features, packed_layer.out_features, b is not None,
                   packed_layer.packed_weight_codes, packed_layer.weight_codebook, packed_layer.weight_center,
                   packed_layer.weight_scale, packed_layer.weight_code_sum, packed_layer.activation_codebook,
                   packed_layer.activation_thresholds, packed_layer.bits, packed_layer.group_size, b)

    _FP32_BUFFERS = ("weight_codebook", "weight_center", "weight_scale", "weight_code_sum",
                     "activation_codebook", "activation_thresholds", "bias_tensor")

    def _apply(self, fn, *args, **kwargs):
        # model.half() must not narrow the fp32 metadata.  (The reference casts the whole model and
        # then widens these buffers again, scripts/benchmark_arcq_on_the_fly.py:63-85, which leaves
        # them rounded to fp16.)  Device moves still apply; dtype changes of these buffers do not.
        keep = {n: self._buffers[n] for n in self._FP32_BUFFERS if self._buffers.get(n) is not None}
        self._host_plan = self._fp8_mult = None         # and with them what they hold where the layer was
        super()._apply(fn, *args, **kwargs)
        for name, orig in keep.items():
            new = self._buffers[name]
            if new.dtype != orig.dtype:
                self._buffers[name] = orig.to(device=new.device)
        return self

    def _load_from_state_dict(self, *args, **kwargs):
        self._host_plan = self._fp8_mult = None
        return super()._load_from_state_dict(*args, **kwargs)

    def can_quantize_for(self, consumer: nn.Module, rows: int) -> bool:
        """Whether ``forward(..., quantize_for=consumer)`` is available: this layer's launch then ends with the
        consumer's stage 1 (the consumer is called with ``input_is_xhat=True``).  From 512 rows on it needs the shared
        weight buffer (``_weight_buffer``)."""
        if not (isinstance(consumer, ARCQPackedLinearOnTheFly) and not self.fp8_operands and not consumer.fp8_operands
                and rows > 0 and self.group_size == 64 and consumer.group_size == 64 and self.bits == consumer.bits
                and consumer.in_features == self.out_features and self.out_features % 64 == 0
                and self.in_features % 64 == 0 and self.out_dtype == torch.float16):
            return False
        if rows < 512:                       # the small-M kernel's epilogue
            return self.in_features <= 1536
        # The block-layout GEMM kernels' epilogue: needs the weight workspace.  Not taken where this layer would run as
        # one launch with stage 1 inside (short rows: DeiT-S at batch 64): the consumer's stage 1 is then already hidden
        # under its own product and the chained pair measured slower (DeiT-S forward 1.86 -> 2.08 ms; DeiT-B 4.88 ->
        # 4.76, ViT-L 49.7 -> 48.5).
        if getattr(self, "_weight_buffer", None) is None or rows * self.in_features * 2 >= 2 ** 32:
            return False
        kernel = _lib.load().arcq_linear_otf_ws_kernel(rows, self.out_features, self.in_features, 1)
        return not kernel.startswith(b"otf_rows")

    def forward(self, x: torch.Tensor, layernorm: Optional[nn.LayerNorm] = None, activation: Optional[str] = None,
                residual: Optional[torch.Tensor] = None, quantize_for: Optional[nn.Module] = None,
                input_is_xhat: bool = False) -> torch.Tensor:
        """``residual + activation(linear(stage1(layernorm(x))))``.  The three optional parts (the LayerNorm in front
        of the layer, ``activation="gelu"`` and the skip connection behind it, as they surround the block linears in
        timm's ``Block``, FQ/timm_quant_models.py:63-121) are fused into the layer's launches where the library can
        (group size 64; for the LayerNorm K <= 1024 from 512 rows on and K <= 1536 below) and run as separate torch
        operations otherwise; without them this is the reference module's forward.  ``quantize_for=consumer`` (see
        ``can_quantize_for``): the result is the consumer's ``x_hat`` instead of this layer's output, to be passed to
        ``consumer(..., input_is_xhat=True)``, which skips its own stage 1."""
        host = _lib._host or _lib.host()
        y = host.layer_forward(self, x, layernorm, activation == "gelu", residual, quantize_for, input_is_xhat) \
            if activation is None or activation == "gelu" else None
        if y is not None:
            return y
        return self._forward_general(x, layernorm, activation, residual, quantize_for, input_is_xhat)

    def _forward_general(self, x, layernorm, activation, residual, quantize_for, input_is_xhat) -> torch.Tensor:
        """Calls the host extension does not take as they are: arguments are checked, converted to what it takes
        (contiguous fp16 / fp32 tensors, the tensor's device current), and parts that do not fuse run as torch operations."""
        original_shape = x.shape
        if original_shape[-1] != self.in_features:
            raise ValueError(f"expected last dim {self.in_features}, got {original_shape[-1]}")
        if not x.is_cuda or not self.packed_weight_codes.is_cuda:
            raise RuntimeError("x and the layer's buffers must be CUDA tensors (there is no CPU forward)")
        if activation not in (None, "gelu"):
            raise ValueError(f"activation must be None or 'gelu', got {activation!r}")
        x2 = x.reshape(-1, self.in_features)
        if x2.dtype not in (torch.float16, torch.float32):
            x2 = x2.to(torch.float16)
        x2 = x2.contiguous()
        m = x2.shape[0]
        chain = quantize_for is not None or input_is_xhat
        if quantize_for is not None and not self.can_quantize_for(quantize_for, m):
            raise ValueError("quantize_for: not available for this pair of layers / number of rows (see can_quantize_for)")
        if input_is_xhat and (x2.dtype != torch.float16 or layernorm is not None or self.fp8_operands):
            raise ValueError("input_is_xhat: x must be the float16 x_hat a producer made for this layer")
        ln_fusable = layernorm is None or (self.in_features <= (1024 if m >= 512 else 1536) and layernorm.elementwise_affine
                                           and type(layernorm) is nn.LayerNorm
                                           and tuple(layernorm.normalized_shape) == (self.in_features,))
        if chain and not ln_fusable:     # (a chained call cannot fall back as a whole: only the LayerNorm runs apart)
            x2, layernorm, ln_fusable = layernorm(x2).contiguous(), None, True
        extras = layernorm is not None or activation is not None or residual is not None or chain
        fuse = (extras and not self.fp8_operands and m > 0 and self.group_size == 64 and self.in_features % 64 == 0
                and ln_fusable)
        if extras and not fuse:          # separate operations around the plain layer
            if layernorm is not None:
                x2 = layernorm(x2)
            y = self.forward(x2)
            if activation == "gelu":
                y = torch.nn.functional.gelu(y)
            if residual is not None:
                y = y + residual.reshape(-1, self.out_features)
            return y.reshape(*original_shape[:-1], self.out_features)
        if self.packed_weight_codes.device != x2.device:
            raise RuntimeError("x and the layer's buffers must be on the same device")
        if m == 0:
            return torch.empty((*original_shape[:-1], self.out_features), dtype=self.out_dtype, device=x2.device)
        w_ws = getattr(self, "_weight_buffer", None)
        if w_ws is not None and (not w_ws.is_cuda or w_ws.dtype != torch.float16 or not w_ws.is_contiguous()
                                 or w_ws.numel() < self.out_features * self.in_features or w_ws.device != x2.device):
            raise ValueError("_weight_buffer must be a contiguous float16 CUDA tensor of at least "
                             "out_features * in_features elements")
        if residual is not None:
            r2 = residual.reshape(-1, self.out_features)
            if r2.dtype != self.out_dtype or tuple(r2.shape) != (m, self.out_features) or r2.device != x2.device:
                raise ValueError("residual must have the output's shape, dtype and device")
            residual = r2.contiguous()
        if self.fp8_operands and self.group_size != 64:
            raise ValueError("fp8_operands needs group_size 64")
        with torch.cuda.device(x2.device):
            y = _lib.host().layer_forward(self, x2, layernorm, activation == "gelu", residual, quantize_for, input_is_xhat)
        if y is None:
            y = self._forward_ops(x2, layernorm, activation, residual, quantize_for, input_is_xhat)
        return y.reshape(*original_shape[:-1], self.out_features)

    def _forward_ops(self, x2, layernorm, activation, residual, quantize_for, input_is_xhat) -> torch.Tensor:
        """The same layer through the operators: without the host extension, and for what it does not take (which the operators
        refuse, saying why)."""
        if tuple(self.packed_weight_codes.shape) != (self.out_features, (self.in_features * self.bits + 7) // 8):
            raise RuntimeError(f"packed_weight_codes has shape {tuple(self.packed_weight_codes.shape)}, which is not the layer's")
        if any(b.numel() > 0 and b.device != x2.device for b in self._buffers.values()):
            raise RuntimeError("x and the layer's buffers must be on the same device")
        args = (x2, self.activation_thresholds, self.activation_codebook, self.packed_weight_codes, self.weight_codebook,
                self.weight_center, self.weight_scale, self.weight_code_sum, self.bias_tensor, self.bits)
        if self.fp8_operands:
            return ops.linear_otf_fp8(*args, out_dtype=self.out_dtype, w_mult=self._fp8_multiplier())
        xh_ws, w_ws = getattr(self, "_x_hat_buffer", None), getattr(self, "_weight_buffer", None)
        if (xh_ws is not None and (xh_ws.dtype != torch.float16 or not xh_ws.is_contiguous() or xh_ws.numel() < x2.numel()
                                   or xh_ws.device != x2.device)):
            xh_ws = None
        common = dict(out_dtype=self.out_dtype, x_hat_ws=xh_ws, w_hat_ws=w_ws)
        if layernorm is None and activation is None and residual is None and quantize_for is None and not input_is_xhat:
            return ops.linear_otf(*args, self.group_size, scratch=True, **common)
        ln = None
        if layernorm is not None:
            bias = torch.zeros_like(layernorm.weight) if layernorm.bias is None else layernorm.bias
            ln = (layernorm.weight.detach(), bias.detach(), layernorm.eps)
        following = None if quantize_for is None else (quantize_for.activation_thresholds, quantize_for.activation_codebook)
        return ops.linear_otf_ex(*args, self.group_size, layernorm=ln, gelu=activation == "gelu", residual=residual,
                                 next_quant=following, x_is_xhat=bool(input_is_xhat), **common)

    def _fp8_multiplier(self) -> float:
        """``ops.fp8_weight_multiplier`` of the layer, read back once per set of buffers (they are held, so that their addresses
        name them); at every call where they are inference tensors, whose changes in place leave no trace."""
        meta = (self.weight_codebook, self.weight_center, self.weight_scale, self.weight_code_sum)
        if any(t.is_inference() for t in meta):
            return ops.fp8_weight_multiplier(*meta)
        key = tuple((t.data_ptr(), t._version) for t in meta)
        kept = self.__dict__.get("_fp8_mult")
        if kept is None or kept[0] != key:
            kept = self._fp8_mult = (key, ops.fp8_weight_multiplier(*meta), tuple(t.detach() for t in meta))
        return kept[1]

    def estimated_persistent_mb(self) -> float:
        """MiB held by this layer's buffers (FQ/arcq_packed_on_the_fly.py:163-169)."""
        return sum(b.numel() * b.element_size() for b in self.buffers()) / 1024 / 1024
