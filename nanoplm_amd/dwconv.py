"""Varlen depthwise 1-D convolution over packed sequences: autograd Function and nn.Module.

Drop-in surface for the conv on the packed path of the encoder layer
(reference call site: src/nanoplm/pretraining/models/modern_bert/modeling.py:421-439, which passes
``x:[total_tokens, hidden]`` and int32 ``cu_seqlens`` (collator.py:322-325) to its sub-modules):

    y = VarlenDWConv1dFunction.apply(x, cu_seqlens, weight, bias)
    conv = VarlenDWConv1d(channels=C, kernel_size=K);  y = conv(x, cu_seqlens)

``residual=True`` (function argument / module option) fuses the residual connection a caller would
write as ``x = x + conv(x, cu_seqlens)``: the kernels compute ``x + conv(x)`` and ``dy + conv^T(dy)``
directly, which saves the elementwise add's three passes over [T, C] in each direction.

All arithmetic runs in hand-written HIP kernels reached through the C ABI of libnplm_dwconv.so.
There is deliberately no CPU or pure-PyTorch implementation here: tensors that are not on a ROCm
device, or a missing shared library, raise.
"""
from __future__ import annotations

import math
from typing import Optional

import torch
from torch import nn

from . import _lib

_DTYPES = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16}


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)   # fast path; public API otherwise


class _launch_on:
    """Context for one library call: makes the tensor's device current (nothing to do when it already is, the
    usual case) and holds the raw handle of that device's current stream in ``.stream``."""
    __slots__ = ("idx", "prev", "stream")

    def __init__(self, t: torch.Tensor):
        self.prev = torch.cuda.current_device()
        self.idx = self.prev if t.device.index is None else t.device.index
        self.stream = None

    def __enter__(self):
        if self.idx != self.prev:
            torch.cuda.set_device(self.idx)
        self.stream = (_raw_stream(self.idx) if _raw_stream is not None
                       else torch.cuda.current_stream(self.idx).cuda_stream)
        return self

    def __exit__(self, *exc):
        if self.idx != self.prev:
            torch.cuda.set_device(self.prev)
        return False


def _validate(x, cu_seqlens, weight, bias):
    """Shape/dtype/device checks shared by forward and backward. Returns (T, C, K, S)."""
    if not isinstance(x, torch.Tensor) or x.dim() != 2:
        raise ValueError("x must be a 2-D tensor [T, C] of packed tokens")
    if x.dtype not in _DTYPES:
        raise TypeError(f"x must be float32 or bfloat16, got {x.dtype}")
    if not x.is_cuda:
        raise RuntimeError("varlen_dwconv runs only on a ROCm device (x is on "
                           f"{x.device}); there is no CPU implementation")
    T, C = x.shape
    if weight.dim() != 2 or weight.shape[0] != C:
        raise ValueError(f"weight must be [C={C}, K], got {tuple(weight.shape)}")
    K = weight.shape[1]
    if K % 2 == 0:
        raise ValueError(f"kernel size must be odd for centred 'same' padding, got K={K}")
    if weight.dtype not in _DTYPES:
        raise TypeError(f"weight must be float32 or bfloat16, got {weight.dtype}")
    if bias is not None and tuple(bias.shape) != (C,):
        raise ValueError(f"bias must be [C={C}], got {tuple(bias.shape)}")
    if cu_seqlens.dtype != torch.int32 or cu_seqlens.dim() != 1 or cu_seqlens.numel() < 1:
        raise TypeError("cu_seqlens must be a 1-D int32 tensor with at least one entry")
    for name, t in (("cu_seqlens", cu_seqlens), ("weight", weight), ("bias", bias)):
        if t is not None and t.device != x.device:
            raise RuntimeError(f"{name} is on {t.device}, x is on {x.device}")
    return T, C, K, cu_seqlens.numel() - 1


def _with_flags(tuning: _lib.Tuning, flags: int) -> _lib.Tuning:
    t = _lib.Tuning.from_buffer_copy(tuning)
    t.flags = flags
    return t


def varlen_dwconv_fwd(x, cu_seqlens, weight, bias=None, *, residual: bool = False,
                      tuning: Optional[_lib.Tuning] = None):
    """y = conv(x), or x + conv(x) with ``residual`` (same dtype as x). Raw forward without autograd."""
    T, C, K, S = _validate(x, cu_seqlens, weight, bias)
    lib = _lib.load()
    x = x.contiguous()
    weight = weight.contiguous()
    cu_seqlens = cu_seqlens.contiguous()
    if bias is not None:
        bias = bias.to(weight.dtype).contiguous()
    y = torch.empty_like(x)
    with _launch_on(x) as dev:
        stream = dev.stream
        flags = _lib.RESIDUAL if residual else 0
        args = (_ptr(x), _ptr(cu_seqlens), _ptr(weight), _ptr(bias), _ptr(y), T, C, K, S,
                _DTYPES[x.dtype], _DTYPES[weight.dtype])
        if tuning is None:
            rc = lib.nplm_dwconv_fwd_ex(*args, flags, stream)
        else:
            rc = lib.nplm_dwconv_fwd_tuned(*args, stream, _with_flags(tuning, flags))
    _lib.check(rc, "nplm_dwconv_fwd")
    return y


def bwd_workspace_bytes(T: int, C: int, K: int, dtype: torch.dtype) -> int:
    """Bytes of workspace the backward needs for these sizes (host arithmetic only)."""
    return int(_lib.load().nplm_dwconv_bwd_workspace_bytes(T, C, K, _DTYPES[dtype]))


def exec_kernel_size(K: int) -> int:
    """The kernel size a plain conv of K taps is planned as, and its workspace made for: an odd K <= 31 that has no
    kernels of its own takes the next size that has, with zero taps on either side (K = 11 and 17 .. 21 with fewer of
    them on the LDS-staged and role-split kernels, whose slabs then fill part of their place)."""
    return int(_lib.load().nplm_dwconv_exec_kernel_size(K))


def varlen_dwconv_bwd(x, dy, cu_seqlens, weight, *, need_dx=True, need_dw=True, residual: bool = False,
                      tuning: Optional[_lib.Tuning] = None, workspace: Optional[torch.Tensor] = None,
                      grads_bf16: bool = False):
    """(dx, dw, db): dx in x's dtype (or None), dw [C,K] and db [C] in fp32 (or None, None).

    With ``residual`` dx is the gradient of x + conv(x), i.e. dy + conv^T(dy); dw and db do not change.
    With ``grads_bf16`` dw and db come back in bf16: the same fp32 sums, rounded once by the kernel that forms them
    (what ``dw.to(torch.bfloat16)`` would give, without the two cast kernels)."""
    T, C, K, S = _validate(x, cu_seqlens, weight, None)
    if dy.shape != x.shape or dy.dtype != x.dtype or dy.device != x.device:
        raise ValueError("dy must match x in shape, dtype and device")
    lib = _lib.load()
    x = x.contiguous()
    dy = dy.contiguous()
    weight = weight.contiguous()
    cu_seqlens = cu_seqlens.contiguous()
    act = _DTYPES[x.dtype]
    dx = torch.empty_like(x) if need_dx else None
    gdt = torch.bfloat16 if grads_bf16 else torch.float32
    dw = torch.empty((C, K), dtype=gdt, device=x.device) if need_dw else None
    db = torch.empty((C,), dtype=gdt, device=x.device) if need_dw else None
    with _launch_on(x) as dev:
        if need_dw and workspace is None:
            if tuning is None:
                nbytes = int(lib.nplm_dwconv_bwd_workspace_bytes(T, C, K, act))
            else:
                nbytes = int(lib.nplm_dwconv_bwd_slabs(T, C, K, act, tuning)) * (exec_kernel_size(K) + 1) * C * 4
            workspace = torch.empty((max(nbytes, 256),), dtype=torch.uint8, device=x.device)
        stream = dev.stream
        flags = (_lib.RESIDUAL if residual else 0) | (_lib.GRADS_BF16 if grads_bf16 else 0)
        args = (_ptr(x), _ptr(dy), _ptr(cu_seqlens), _ptr(weight), _ptr(dx), _ptr(dw), _ptr(db),
                _ptr(workspace), 0 if workspace is None else workspace.numel() * workspace.element_size(),
                T, C, K, S, act, _DTYPES[weight.dtype])
        if tuning is None:
            rc = lib.nplm_dwconv_bwd_ex(*args, flags, stream)
        else:
            rc = lib.nplm_dwconv_bwd_tuned(*args, stream, _with_flags(tuning, flags))
    _lib.check(rc, "nplm_dwconv_bwd")
    return dx, dw, db


def check_cu_seqlens(cu_seqlens: torch.Tensor, T: int) -> None:
    """Debug helper: verify cu[0] == 0, non-decreasing, cu[-1] == T (synchronises the stream)."""
    if not cu_seqlens.is_cuda or cu_seqlens.dtype != torch.int32:
        raise TypeError("cu_seqlens must be an int32 tensor on a ROCm device")
    lib = _lib.load()
    with _launch_on(cu_seqlens) as dev:
        rc = lib.nplm_dwconv_check_cu(_ptr(cu_seqlens.contiguous()), cu_seqlens.numel() - 1, T, dev.stream)
    _lib.check(rc, "nplm_dwconv_check_cu")


class VarlenDWConv1dFunction(torch.autograd.Function):
    """``apply(x, cu_seqlens, weight, bias[, residual]) -> y``; backward returns ``(dx, None, dw, db[, None])``.

    dw and db are reduced and produced in fp32 by the kernels and cast to the parameters' dtypes
    only here. Under ``torch.autocast`` the op takes its inputs as they come (bf16 activations
    with fp32 parameters is a supported combination), so no cast kernels are inserted.
    """

    @staticmethod
    def forward(ctx, x, cu_seqlens, weight, bias=None, residual=False):
        y = varlen_dwconv_fwd(x, cu_seqlens, weight, bias, residual=bool(residual))
        ctx.save_for_backward(x, cu_seqlens, weight)
        ctx.bias_dtype = None if bias is None else bias.dtype
        ctx.residual = bool(residual)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, cu_seqlens, weight = ctx.saved_tensors
        need_dx = ctx.needs_input_grad[0]
        need_dw = ctx.needs_input_grad[2] or (ctx.bias_dtype is not None and ctx.needs_input_grad[3])
        if dy.dtype != x.dtype:
            dy = dy.to(x.dtype)
        # bf16 parameters take their gradients in bf16 straight from the reduction kernel (no cast kernels)
        grads_bf16 = weight.dtype == torch.bfloat16 and ctx.bias_dtype in (None, torch.bfloat16)
        dx, dw, db = varlen_dwconv_bwd(x, dy, cu_seqlens, weight, need_dx=need_dx, need_dw=need_dw,
                                       residual=ctx.residual, grads_bf16=grads_bf16)
        if dw is not None:
            dw = dw.to(weight.dtype) if ctx.needs_input_grad[2] else None
            db = db.to(ctx.bias_dtype) if (ctx.bias_dtype is not None and ctx.needs_input_grad[3]) else None
        return dx, None, dw, db, None


def varlen_dwconv(x, cu_seqlens, weight, bias=None, residual: bool = False):
    """Functional form of :class:`VarlenDWConv1dFunction`. While ``torch.compile`` is tracing, the call goes
    through the registered custom ops instead (same kernels), so that callers of this function (the padded-batch
    door among them) never break the graph. Otherwise the native node takes the call (same kernels, same gradients, no Python in
    either direction) or, for a call that is not of its form, leaves it to the Function."""
    if torch.compiler.is_compiling():
        return varlen_dwconv_fwd_op(x, cu_seqlens, weight, bias, residual)
    y = _lib.load_node().dwconv(x, cu_seqlens, weight, bias, residual)
    return VarlenDWConv1dFunction.apply(x, cu_seqlens, weight, bias, residual) if y is None else y


class VarlenDWConv1d(nn.Module):
    """Depthwise conv over packed sequences: ``forward(x:[T,C], cu_seqlens:int32[S+1]) -> [T,C]``.

    ``weight`` is ``[C, K]`` (tap k multiplies row ``t + k - (K-1)//2``), ``bias`` is ``[C]``.
    Rows outside a sequence read as zero; nothing crosses a sequence boundary.
    ``residual=True`` makes the module return ``x + conv(x)`` from the same single pass.

    How the parameters meet the reference's training loop:

    * ``flat_weight=True`` registers the taps as a 1-D parameter ``weight_flat`` of ``C*K`` elements
      (``.weight`` stays available as its ``[C, K]`` view). A 2-D ``[C, K]`` parameter would be routed
      to Muon by ``build_muon_optimizer`` (src/nanoplm/pretraining/optim.py:43-51 sends every
      ``ndim == 2`` hidden parameter there; orthogonalising a C x 7 tap table is meaningless) and
      weight-decayed by ``_use_weight_decay`` (src/nanoplm/pretraining/pure_pipeline.py:68-76);
      a 1-D parameter lands in the AdamW no-decay group of both, with no change to the reference.
    * ``init``: ``"normal"`` = N(0, 1/K) taps and N(0, 0.02^2) bias (the benchmark's distributions);
      ``"zero"`` = all zeros, so a ``residual=True`` block starts as the identity, matching the
      reference's zero-initialised output projections (modeling.py:602-605); ``"identity"`` = centre
      tap 1, for the non-residual form. The reference's ``init_weights`` (modeling.py:581-623) has no
      branch that would touch this module, so the module initialises itself.
    """

    def __init__(self, channels: int, kernel_size: int, bias: bool = True, residual: bool = False,
                 flat_weight: bool = False, init: str = "normal", device=None, dtype=None):
        super().__init__()
        if kernel_size < 1 or kernel_size % 2 == 0:
            raise ValueError(f"kernel_size must be odd and positive, got {kernel_size}")
        if init not in ("normal", "zero", "identity"):
            raise ValueError(f"init must be 'normal', 'zero' or 'identity', got {init!r}")
        self.channels = channels
        self.kernel_size = kernel_size
        self.residual = bool(residual)
        self.flat_weight = bool(flat_weight)
        self.init = init
        if self.flat_weight:
            self.weight_flat = nn.Parameter(torch.empty((channels * kernel_size,), device=device, dtype=dtype))
        else:
            self.weight = nn.Parameter(torch.empty((channels, kernel_size), device=device, dtype=dtype))
        self.bias = nn.Parameter(torch.empty((channels,), device=device, dtype=dtype)) if bias else None
        self.reset_parameters()

    def __getattr__(self, name):
        # .weight of a flat_weight module: the [C, K] view of the 1-D parameter (autograd flows through it)
        if name == "weight" and "weight_flat" in self.__dict__.get("_parameters", {}):
            return self._parameters["weight_flat"].view(self.channels, self.kernel_size)
        return super().__getattr__(name)

    @torch.no_grad()
    def reset_parameters(self) -> None:
        w = self.weight
        if self.init == "normal":
            nn.init.normal_(w, mean=0.0, std=1.0 / math.sqrt(self.kernel_size))
        else:
            w.zero_()
            if self.init == "identity":
                w[:, (self.kernel_size - 1) // 2] = 1.0
        if self.bias is not None:
            if self.init == "normal":
                nn.init.normal_(self.bias, mean=0.0, std=0.02)
            else:
                self.bias.zero_()

    def forward_padded(self, x: torch.Tensor, attention_mask: torch.Tensor,
                       assume_right_padded: bool = True) -> torch.Tensor:
        """Padded-batch door: ``x:[B, L, C]``, ``attention_mask:[B, L]`` (see nanoplm_amd.padded)."""
        from .padded import padded_dwconv
        return padded_dwconv(x, attention_mask, self.weight, self.bias, self.residual, assume_right_padded)

    def forward(self, x: torch.Tensor, cu_seqlens: torch.Tensor) -> torch.Tensor:
        return varlen_dwconv(x, cu_seqlens, self.weight, self.bias, self.residual)

    def forward_gated(self, z: torch.Tensor, cu_seqlens: torch.Tensor) -> torch.Tensor:
        """SwiGLU door: ``z = Wi(x)`` of width ``2 * channels`` (x_proj columns, then gate columns);
        returns ``conv(x_proj * silu(gate))`` with the gate product fused into the kernels (see nanoplm_amd.gated)."""
        from .gated import gated_varlen_dwconv
        return gated_varlen_dwconv(z, cu_seqlens, self.weight, self.bias, self.residual)

    def forward_prenorm(self, x: torch.Tensor, cu_seqlens: torch.Tensor, norm: nn.LayerNorm) -> torch.Tensor:
        """Pre-norm door: ``conv(norm(x))`` (``+ x`` with ``residual=True``: the identity is the raw x, as in the
        reference's ``x + sub_module(norm(x))``, modeling.py:430-438) with ``norm`` — a ``torch.nn.LayerNorm`` over the
        channels (modeling.py:408-414) — evaluated inside the conv's kernels (see nanoplm_amd.lnconv)."""
        from .lnconv import ln_varlen_dwconv_compilable
        if tuple(norm.normalized_shape) != (self.channels,):
            raise ValueError(f"norm must normalise over the {self.channels} channels, got {tuple(norm.normalized_shape)}")
        ln_weight = norm.weight if norm.weight is not None else torch.ones(self.channels, device=x.device, dtype=self.weight.dtype)
        return ln_varlen_dwconv_compilable(x, cu_seqlens, ln_weight, norm.bias, self.weight, self.bias, eps=norm.eps,
                                           residual=self.residual)

    def extra_repr(self) -> str:
        return (f"channels={self.channels}, kernel_size={self.kernel_size}, bias={self.bias is not None}, "
                f"residual={self.residual}, flat_weight={self.flat_weight}, init={self.init}")


# ---------------------------------------------------------------------------------------------
# torch.library registration: the same two kernels as opaque custom ops, so that
# torch.compile(model, dynamic=False) (src/nanoplm/pretraining/pure_pipeline.py:519-524) traces
# through a model that contains the conv without a graph break. Neither op synchronises the host;
# cu_seqlens may be the static collator's fixed-length tensor (collator.py:430-450).
# ---------------------------------------------------------------------------------------------
@torch.library.custom_op("nanoplm_amd::varlen_dwconv_fwd", mutates_args=(), device_types="cuda")
def varlen_dwconv_fwd_op(x: torch.Tensor, cu_seqlens: torch.Tensor, weight: torch.Tensor,
                         bias: Optional[torch.Tensor], residual: bool = False) -> torch.Tensor:
    return varlen_dwconv_fwd(x, cu_seqlens, weight, bias, residual=residual)


@varlen_dwconv_fwd_op.register_fake
def _(x, cu_seqlens, weight, bias, residual=False):
    return torch.empty_like(x, memory_format=torch.contiguous_format)


@torch.library.custom_op("nanoplm_amd::varlen_dwconv_bwd", mutates_args=(), device_types="cuda")
def varlen_dwconv_bwd_op(x: torch.Tensor, dy: torch.Tensor, cu_seqlens: torch.Tensor, weight: torch.Tensor,
                         residual: bool = False, grads_bf16: bool = False) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(dx, dw, db) with dw [C,K] and db [C] in fp32 (bf16 with ``grads_bf16``)."""
    dx, dw, db = varlen_dwconv_bwd(x, dy, cu_seqlens, weight, residual=residual, grads_bf16=grads_bf16)
    return dx, dw, db


@varlen_dwconv_bwd_op.register_fake
def _(x, dy, cu_seqlens, weight, residual=False, grads_bf16=False):
    C, K = weight.shape
    gdt = torch.bfloat16 if grads_bf16 else torch.float32
    return (torch.empty_like(x, memory_format=torch.contiguous_format),
            x.new_empty((C, K), dtype=gdt), x.new_empty((C,), dtype=gdt))


def _op_setup_context(ctx, inputs, output):
    x, cu_seqlens, weight, bias, residual = inputs
    ctx.save_for_backward(x, cu_seqlens, weight)
    ctx.bias_dtype = None if bias is None else bias.dtype
    ctx.residual = bool(residual)


def _op_backward(ctx, dy):
    x, cu_seqlens, weight = ctx.saved_tensors
    if dy.dtype != x.dtype:
        dy = dy.to(x.dtype)
    grads_bf16 = weight.dtype == torch.bfloat16 and ctx.bias_dtype in (None, torch.bfloat16)
    dx, dw, db = varlen_dwconv_bwd_op(x, dy.contiguous(), cu_seqlens, weight, ctx.residual, grads_bf16)
    return dx, None, dw.to(weight.dtype), (None if ctx.bias_dtype is None else db.to(ctx.bias_dtype)), None


varlen_dwconv_fwd_op.register_autograd(_op_backward, setup_context=_op_setup_context)


def varlen_dwconv_compilable(x, cu_seqlens, weight, bias=None, residual: bool = False):
    """Same result as :func:`varlen_dwconv`, routed through the registered custom ops (traceable)."""
    return varlen_dwconv_fwd_op(x, cu_seqlens, weight, bias, residual)
