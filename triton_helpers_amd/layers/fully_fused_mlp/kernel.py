"""Fully fused small MLP on MI355X.

Drop-in for ``triton_helpers/layers/fully_fused_mlp/kernel.py`` of the reference:
same ``fully_fused_mlp(...)`` functional and ``_fully_fused_mlp`` autograd Function
(argument order, 9-tuple returned by ``backward``), same assertions and the same
weight layout (``w_hid`` = hidden layers stacked along rows, ``b_hid [depth-1, H]``).
The Triton launches are replaced by ``nf_mlp_fwd`` / ``nf_mlp_bwd`` of ``libnf_cdna4.so``.

Supersets / differences:
  * any bias may be ``None`` (the reference always has biases);
  * weight gradients are accumulated in float32 inside the kernel and rounded once
    (the reference sums per-program partials in the storage dtype, kernel.py:599-633);
  * ``fp16_acc`` is accepted and ignored: accumulation is always float32 (MFMA);
  * float16 and bfloat16 storage (what autocast produces) runs on the 16-bit matrix instructions: the fast path.
    float32 tensors (the reference feeds them to ``tl.dot``, which multiplies in TF32: float32 range, 10-bit
    mantissa) run on the float32 matrix instruction: float32 range and mantissa, about a sixth of the 16-bit rate, and
    a backward scratch of ``depth * rows * d_hidden * 4`` bytes.  ``set_float32_operands("float16")`` trades the
    range for speed: float32 tensors are then multiplied with float16 operands (the same 10-bit mantissa as TF32,
    float32 accumulation and results; operands beyond +-65504 overflow).
"""
from __future__ import annotations

from typing import Final, Optional

import torch
import torch.nn.functional as F
from torch import Tensor
from torch.autograd import Function

from ... import _lib

# Above this size the weights do not stay on chip (reference kernel.py:13-14)
FULLY_FUSED_MAX_DIM: Final = 64

_ACTIVATIONS = ("relu", "relu2", "silu", "none")

_FLOAT32_OPERANDS = "float32"


def set_float32_operands(kind: str) -> str:
    """How float32 tensors are multiplied: ``"float32"`` (default: float32 range and mantissa) or ``"float16"``
    (float16 operands, float32 accumulation: several times faster, operands limited to +-65504).  Returns the
    previous setting.  (The counterpart of ``allow_tf32`` for ``tl.dot`` in the reference, kernel.py:17-47.)"""
    global _FLOAT32_OPERANDS
    assert kind in ("float32", "float16"), f"float32 operands are 'float32' or 'float16', got {kind!r}"
    previous, _FLOAT32_OPERANDS = _FLOAT32_OPERANDS, kind
    return previous


def get_float32_operands() -> str:
    return _FLOAT32_OPERANDS


# ---------------------------------------------------------------------------
# Per-layer math with the reference's names (kernel.py:17-74).  In the reference these
# are Triton device functions; here they are plain torch functions for users' tests.
# No operator of this package calls them.
# ---------------------------------------------------------------------------
def _activate(z: Tensor, activation: str) -> Tensor:
    if activation == "relu":
        return torch.where(z < 0, torch.zeros_like(z), z)
    if activation == "silu":
        return z * torch.sigmoid(z)
    if activation == "relu2":
        return torch.clamp_min(z, 0) * z
    if activation == "none":
        return z
    raise ValueError(f"Invalid activation function: {activation}")


def feedforward(x: Tensor, w: Tensor, b: Optional[Tensor], HAS_BIAS: bool = True, ACTIVATION: str = "relu",
                DTYPE: torch.dtype = torch.float32) -> Tensor:
    z = x.to(DTYPE) @ w.to(DTYPE).t()
    if HAS_BIAS and b is not None:
        z = z + b.to(DTYPE)
    return _activate(z, ACTIVATION).to(x.dtype)


def feedforward_bwd_dz(z: Tensor, do: Tensor, ACTIVATION: str) -> Tensor:
    zf, g = z.float(), do.float()
    if ACTIVATION == "relu":
        dz = torch.where(zf > 0, g, torch.zeros_like(g))
    elif ACTIVATION == "silu":
        s = torch.sigmoid(zf)
        dz = g * s * (zf * (1 - s) + 1)
    elif ACTIVATION == "relu2":
        dz = torch.where(zf > 0, g * (2 * zf), torch.zeros_like(g))
    elif ACTIVATION == "none":
        dz = g
    else:
        raise ValueError(f"Invalid activation function: {ACTIVATION}")
    return dz.to(do.dtype)


def feedforward_bwd_dw(x: Tensor, dz: Tensor, DTYPE: torch.dtype = torch.float32) -> Tensor:
    return (dz.to(DTYPE).t() @ x.to(DTYPE)).to(dz.dtype)


def feedforward_bwd_dx(w: Tensor, dz: Tensor, DTYPE: torch.dtype = torch.float32) -> Tensor:
    return (dz.to(DTYPE) @ w.to(DTYPE)).to(dz.dtype)


# ---------------------------------------------------------------------------
def _check_storage(x: Tensor, w_in: Tensor, *others: Optional[Tensor]) -> None:
    """Parameters share one dtype.  With 16-bit parameters ``x`` may be in the other 16-bit dtype (an fp16 encoder
    output in front of bf16 weights): the kernels convert it while loading, exactly as a cast in front would.
    float32 runs as a whole (``x`` and parameters)."""
    if w_in.dtype == torch.float32:
        assert x.dtype == torch.float32, f"float32 parameters take a float32 input, got {x.dtype}"
    else:
        for t in (x, w_in):
            if t.dtype not in (torch.float16, torch.bfloat16):
                raise NotImplementedError(
                    f"fully_fused_mlp runs on float16 / bfloat16 / float32 storage, got {t.dtype}; cast the tensors or use autocast"
                )
    for t in others:
        assert t is None or t.dtype == w_in.dtype, f"All parameters must share one dtype, got {w_in.dtype} and {t.dtype}"
    for t in (w_in, *others):
        assert t is None or t.device == x.device, "All tensors must be on the same device"
    assert x.device.type == "cuda", "All tensors must be on a GPU device"


_rows2d = _lib.rows2d


def _half(t: Optional[Tensor]) -> Optional[Tensor]:
    return None if t is None else t.to(torch.float16)


class _fully_fused_mlp(Function):
    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda", cast_inputs=torch.float16)
    def forward(
        ctx,
        x: Tensor,
        w_in: Tensor, b_in: Optional[Tensor],
        w_out: Tensor, b_out: Optional[Tensor],
        w_hid: Optional[Tensor], b_hid: Optional[Tensor],
        activation: str = "relu",
        fp16_acc: bool = False,
    ) -> Tensor:
        B, L, D = x.shape
        D_hidden, D_in = w_in.shape
        D_out, _ = w_out.shape
        assert D_in == D, "Input dimension mismatch"
        assert D_hidden == w_out.shape[-1], "Hidden dimension mismatch"

        assert D_in <= FULLY_FUSED_MAX_DIM, f"Input dimension {D_in} too large for full fusion"
        assert D_hidden <= FULLY_FUSED_MAX_DIM, f"Hidden dimension {D_hidden} too large for full fusion"
        assert D_out <= FULLY_FUSED_MAX_DIM, f"Output dimension {D_out} too large for full fusion"

        assert D_hidden & (D_hidden - 1) == 0, "Hidden dimension must be a power of 2"
        assert D_hidden >= 16, "Hidden dimension must be at least 16"

        if w_hid is not None and w_hid.numel() > 0:
            n_hid = w_hid.shape[0] // D_hidden
            assert w_hid.shape == (n_hid * D_hidden, D_hidden), "Hidden weight shape mismatch"
            assert b_hid is None or b_hid.shape == (n_hid, D_hidden), "Hidden bias shape mismatch"
            depth = n_hid + 1
        else:
            depth = 1
            w_hid = b_hid = None
        assert b_in is None or b_in.shape == (D_hidden,), "Input bias shape mismatch"
        assert b_out is None or b_out.shape == (D_out,), "Output bias shape mismatch"

        assert activation in _ACTIVATIONS, f"Invalid activation function: {activation}"
        _check_storage(x, w_in, b_in, w_out, b_out, w_hid, b_hid)

        ctx.save_for_backward(x, w_in, b_in, w_out, b_out, w_hid, b_hid)
        ctx.activation = activation
        ctx.fp16_acc = fp16_acc
        ctx.wide = wide = w_in.dtype == torch.float32 and _FLOAT32_OPERANDS == "float16"
        if wide:  # float16 operands, float32 accumulation and results
            x, w_in, b_in, w_out, b_out, w_hid, b_hid = (_half(t) for t in (x, w_in, b_in, w_out, b_out, w_hid, b_hid))
        o = _lib.native().mlp_launch_forward(x, w_in, b_in, w_out, b_out, w_hid, b_hid, _lib.NF_ACT[activation])
        return o.float() if wide else o

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, do: Tensor):
        tensors = ctx.saved_tensors
        if ctx.wide:
            tensors = tuple(_half(t) for t in tensors)
        dx, *grads = _lib.native().mlp_launch_backward(*tensors, _lib.NF_ACT[ctx.activation], do, ctx.needs_input_grad[0], ctx.wide)
        if ctx.wide and dx is not None:
            dx = dx.float()
        return dx, *grads, None, None


def fully_fused_mlp(
    x: Tensor,
    w_in: Tensor, b_in: Optional[Tensor],
    w_out: Tensor, b_out: Optional[Tensor],
    w_hid: Optional[Tensor] = None, b_hid: Optional[Tensor] = None,
    activation: str = "relu",
    fp16_acc: bool = False,
) -> Tensor:
    r"""Fully fused forward pass of a small MLP (reference kernel.py:640-686).

    Shapes:
        - x: :math:`(B, L, D_{in})`
        - w_in: :math:`(D_{hidden}, D_{in})`, b_in: :math:`(D_{hidden},)` or ``None``
        - w_out: :math:`(D_{out}, D_{hidden})`, b_out: :math:`(D_{out},)` or ``None``
        - w_hid: :math:`((depth-1) \cdot D_{hidden}, D_{hidden})`, b_hid: :math:`(depth-1, D_{hidden})` or ``None``
        - Output: :math:`(B, L, D_{out})`

    ``activation`` is one of ``"relu"``, ``"relu2"``, ``"silu"``, ``"none"`` and is applied after every
    layer but the last.
    """
    if _FLOAT32_OPERANDS == "float32":
        y = _lib.native().mlp(x, w_in, b_in, w_out, b_out, w_hid, b_hid, activation)
        if y is not None:
            return y
    # float16 operands for float32 tensors, or arguments to be refused
    return _fully_fused_mlp.apply(x, w_in, b_in, w_out, b_out, w_hid, b_hid, activation, fp16_acc)
