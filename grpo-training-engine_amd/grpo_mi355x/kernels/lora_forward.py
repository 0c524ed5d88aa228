"""``lora_fused_forward`` -- the NF4 + LoRA linear on the HIP kernel.

Same call surface and dispatch as the reference's
``src/triton_kernels/lora_forward.py:933-1037``:

* ``lora_layer`` (a ``ManualLoRALayer``-like object) or explicit
  ``base_layer/lora_A/lora_B/scaling/dropout``;
* dropout p > 0 -> ``ValueError`` (``:958-960``);
* a base weight with ``quant_state`` and ``prefer_base_layer=False`` -> the
  fused kernel (``FusedLoRAFunction``, ``:966-984``); otherwise the adapter
  branch ``base_layer(x) + B(A(x)) * scaling`` (``:986-1037``);
* shape/dtype/device problems -> ``ValueError`` (``_validate_inputs``,
  ``:435-487``); rank <= 0 -> ``ValueError`` (``:670-671``).

The fused forward is ``grpo_nf4_lora_linear`` for few rows (the weight decoded
as it is multiplied: the split-K kernel up to 64 rows, the NF4 GEMM beyond) and
``grpo_nf4_lora_train_forward`` where ``train_forward_pays`` (the weight brought to
16 bits in the call, then an MFMA GEMM with the epilogue in it).  float16 x
with float16 adapters (the reference's float16 X_DTYPE / LORA_DTYPE, ``:141-143,
745-749``) has every rounding point float16; mixed dtypes raise ``ValueError``
(the caller's torch branch then serves them, as for any shape the kernels do not
take).  The backward (``:761-930``) is ``grpo_nf4_lora_train_backward``: the
reference's gradients and rounding points, grad_x as one GEMM over the weight
transposed in 16 bits, everything of rank r straight from x and grad_out.
Tensors the training kernels do not take (``_train_workspace``), a forward of many
rows whose product is too long for its tiles (``train_forward_pays``) and a
backward that is itself differentiated run the same products as torch ops.
"""

from __future__ import annotations

from typing import Optional

import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F

from ..core.nf4 import float_absmax
from . import ops


_HALF = (torch.bfloat16, torch.float16)


def _validate_inputs(x: torch.Tensor, weight_4bit: torch.Tensor, quant_state,
                     lora_A: torch.Tensor, lora_B: torch.Tensor):
    """``lora_forward.py:435-487`` (same messages, same ValueError)."""
    xs, sa, sb = x.shape, lora_A.shape, lora_B.shape
    if len(xs) == 3 and len(sa) == 2 and len(sb) == 2 and x.is_cuda and weight_4bit.is_cuda and \
            lora_A.is_cuda and lora_B.is_cuda and x.dtype in _HALF and lora_A.dtype in _HALF and \
            lora_A.dtype == lora_B.dtype:
        n, k = quant_state.shape
        if xs[2] == k == sa[1] and sb[0] == n and sb[1] == sa[0]:
            return xs[0] * xs[1], n, k, sa[0]
    return _validate_each(x, weight_4bit, quant_state, lora_A, lora_B)


def _validate_each(x, weight_4bit, quant_state, lora_A, lora_B):
    """The checks of ``_validate_inputs`` one by one, for their messages."""
    if x.ndim != 3:
        raise ValueError(f"x must be [batch, seq_len, hidden], got {x.shape}.")
    if lora_A.ndim != 2 or lora_B.ndim != 2:
        raise ValueError("lora_A and lora_B must be 2D weight matrices.")
    if not x.is_cuda:
        raise ValueError("x must be on CUDA device.")
    if not weight_4bit.is_cuda:
        raise ValueError("weight_4bit must be on CUDA device.")
    if not lora_A.is_cuda or not lora_B.is_cuda:
        raise ValueError("lora_A and lora_B must be on CUDA device.")
    if x.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError(f"x must be float16/bfloat16, got {x.dtype}.")
    if lora_A.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError(f"lora_A must be float16/bfloat16, got {lora_A.dtype}.")
    if lora_B.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError(f"lora_B must be float16/bfloat16, got {lora_B.dtype}.")
    if lora_A.dtype != lora_B.dtype:
        raise ValueError(
            f"lora_A and lora_B must have the same dtype, got {lora_A.dtype} and {lora_B.dtype}.")
    batch, seq_len, in_features = x.shape
    out_features, in_features_w = tuple(quant_state.shape)
    if in_features != in_features_w:
        raise ValueError("Input hidden size does not match quantized weight shape: "
                         f"{in_features} vs {in_features_w}.")
    rank, in_features_a = lora_A.shape
    out_features_b, rank_b = lora_B.shape
    if in_features_a != in_features:
        raise ValueError(f"lora_A input features mismatch: {in_features_a} vs {in_features}.")
    if out_features_b != out_features or rank_b != rank:
        raise ValueError("lora_B shape mismatch: expected "
                         f"[{out_features}, {rank}], got {lora_B.shape}.")
    return batch * seq_len, out_features, in_features, rank


def _extract_quant_state(weight_4bit: torch.Tensor, quant_state):
    """``lora_forward.py:527-576``: the float32 absmax, codebook and blocksize.

    A double-quantized (nested) state's absmax is expanded to float32 once
    (``lora_forward.py:187-199``, see ``core.nf4.float_absmax``) and cached on
    the state: the base weights are frozen."""
    device = weight_4bit.device
    if getattr(quant_state, "nested", False) and quant_state.absmax.device != device:
        raise ValueError("nested quant_state must be on the weight's device.")
    absmax, code = float_absmax(quant_state), quant_state.code
    if absmax.device != device or not absmax.is_contiguous():
        absmax = absmax.to(device=device).contiguous()
    if code.device != device or code.dtype != torch.float32 or not code.is_contiguous():
        code = code.to(device=device, dtype=torch.float32).contiguous()
    if absmax.dtype != torch.float32:
        raise ValueError(f"absmax must be float32 for a non-nested state, got {absmax.dtype}.")
    if code.numel() != 16:
        raise ValueError("quant_state.code must have 16 entries (a 4-bit codebook).")
    return absmax, code, int(quant_state.blocksize)


def _scalar_as(v: float, dtype: torch.dtype) -> float:
    """``v`` rounded to ``dtype`` (bf16 or float16), as a Python float:
    ``t * _scalar_as(v, t.dtype)`` is dtype(float(t) * dtype(v)), the
    reference's product with a 0-dim tensor of the LoRA dtype
    (lora_forward.py:836-837), without a host-to-device copy."""
    return float(torch.tensor(float(v), dtype=dtype))


def _bf16_scalar(v: float) -> float:
    """``_scalar_as(v, torch.bfloat16)``."""
    return _scalar_as(v, torch.bfloat16)


# Where the torch ops run (see _train_workspace): rows of grad_out from which
# grad_x's NF4 product is dequantize + bf16 GEMM instead of the fused nf4_grad_x
# kernel.  Measured on MI355X at M = 4096
# over the Qwen2-1.5B projection shapes: the GEMM path is 1.8x (q, o) to 4.2x
# (gate, up) faster.  Below 1024 rows the fused kernel avoids writing and
# re-reading the whole dequantized weight for few rows.
GRAD_X_GEMM_MIN_ROWS = 1024


def fused_forward_rows(k: int) -> int:
    """Where the training linear does not apply: most rows for which the forward
    runs the fused NF4 GEMM rather than the dequantized weight + hipBLASLt.  Measured on MI355X over the Qwen2-1.5B
    projection shapes (r = 16): the fused GEMM is faster up to 4096 rows for
    K = 1536 (e.g. gate at 4096 rows: 217 us against 257 us) and up to 1024
    rows for down_proj's K = 8960 (96 against 84 us at 1024 rows with LoRA, 73
    against 84 without); from 8192 rows hipBLASLt's GEMM wins for every shape.
    """
    return 4096 if k <= 4096 else 1024


def train_forward_pays(m: int, n: int, k: int, r: int, blocksize: int,
                       dtype: torch.dtype) -> bool:
    """Whether the forward runs the training linear (the weight brought to 16 bits in
    the call, then an MFMA GEMM) rather than the kernels that decode the weight as they
    multiply.  Decoding costs the NF4 GEMM a share of every tile, so what counts is M N.
    Measured on MI355X (us, those against this, N x K at M rows, r = 16, bf16, the NF4
    GEMM's ring kernel): 1536 x 1536 26.5 / 30.4 at 2048, 44.9 / 38.8 at 4096; 3584 x
    3584 49.2 / 52.3 at 1024, 91.4 / 79.8 at 2048; 8960 x 1536 41.7 / 45.1 at 512, 65.2 /
    54.8 at 1024; 256 x 1536 15.5 / 19.1 at 4096.  Shapes its older kernel takes cross
    earlier: 24.2 / 19.2 at 512 rows of 1536 x 1536, 136.6 / 106.3 at 2048 of 1536 x
    8960.  In float16 the decoding kernel does not split K: 32.9 / 17.2 (1536 x 1536) and
    33.2 / 30.1 (8960 x 1536) at 16 rows; it wins where N is wide enough to fill the chip
    at few rows over a short K (8960 x 1536 34.5 / 38.3 at 256, 48.2 / 45.5 at 512; 8960 x
    1024 26.2 / 30.2 at 384).

    Beyond ``fused_forward_rows`` the other route is the dequantized weight + library
    GEMMs, which cut a long K over the CUs that the 256 x 256 tiles leave idle: K = 8960,
    r = 16, that against this, 135 / 176 at 3072 rows of N 1536 (72 tiles), 177 / 208 at
    4096 of 2048 (128), 389 / 479 at 8192 of 2560 (320: two rounds), but 249 / 243 at 8192 of
    2048 (256) and 616 / 454 at 2048 of 8960.  At K = 18944 the library's time is uneven and
    this one is mostly faster (3584 columns: 458 / 387 at 2048 rows, 357 / 370 at 1536).
    Rank 32 costs the preparation more, which decides at few columns: 55.7 / 66.2 at 6144
    rows of 512 x 3584."""
    rows = fused_forward_rows(k)
    if m > rows:
        if 4096 < k <= 10240 and n <= 4096:
            tiles = -(-m // 256) * -(-n // 256)
            return tiles >= (0.73 if r <= 16 else 0.88) * 256 * -(-tiles // 256)
        return not (r > 16 and n <= 1024 and 3072 <= k <= 4096)
    if dtype == torch.float16:
        return not (128 <= m <= 384 and k <= 1536 and n >= 4 * k)
    if k % 128 == 0 and r <= 16 and blocksize >= 64:
        return m * n >= 5_000_000
    return m >= (512 if k <= 4096 else 1024)


def _train_workspace(w: torch.Tensor, blocksize: int, lora_A: torch.Tensor,
                     lora_B: torch.Tensor, *rows: torch.Tensor) -> int:
    """Workspace bytes of the training linear for these tensors, 0 if its kernels do
    not take them: one dtype, N and K multiples of 32, rank <= 32, a power-of-two
    blocksize >= 32, 16-byte aligned (tensors without a storage, as under a vmapped
    backward, are left to the torch ops)."""
    x = rows[0]
    if lora_A.dtype != x.dtype or lora_B.dtype != x.dtype:
        return 0
    r, k = lora_A.shape
    nbytes = ops.nf4_lora_train_workspace_bytes(x.shape[0], lora_B.shape[0], k, r, blocksize)
    if not nbytes:
        return 0
    try:
        low = w.data_ptr() | lora_A.data_ptr()
        for t in rows:
            low |= t.data_ptr()
    except RuntimeError:
        return 0
    return nbytes if low % 16 == 0 else 0


def _run_forward(x, weight_4bit, quant_state, lora_A, lora_B, scaling, bias):
    """The fused linear: (output, what its backward needs)."""
    m, n, k, r = _validate_inputs(x, weight_4bit, quant_state, lora_A, lora_B)
    if r <= 0:
        raise ValueError(f"LoRA rank must be > 0, got {r}.")
    dt = x.dtype
    if lora_A.dtype != dt:
        raise ValueError("the HIP NF4+LoRA kernels take x and the adapters in one dtype "
                         f"(bfloat16 or float16); got x {dt}, lora {lora_A.dtype}.")
    absmax, code, blocksize = _extract_quant_state(weight_4bit, quant_state)
    w = weight_4bit if weight_4bit.is_contiguous() else weight_4bit.contiguous()
    if w.dtype != torch.uint8:
        w = w.view(-1).view(torch.uint8)
    x_flat = (x if x.is_contiguous() else x.contiguous()).view(m, k)
    if w.numel() * 2 < n * k or absmax.numel() * blocksize < n * k:
        raise ValueError("packed weight or absmax too short for the quant_state's shape.")
    if bias is not None and (not bias.is_cuda or bias.numel() != n):
        raise ValueError(f"bias must have {n} elements on the ROCm/HIP device.")
    nbytes = (_train_workspace(w, blocksize, lora_A, lora_B, x_flat)
              if train_forward_pays(m, n, k, r, blocksize, dt) else 0)
    if nbytes:
        if bias is not None and (bias.dtype != dt or not bias.is_contiguous()):
            bias = bias.to(dt).contiguous()
        out = ops.train_forward(x_flat, w, absmax, code, blocksize, lora_A.contiguous(),
                                lora_B.contiguous(), scaling, bias, nbytes)
    else:
        out = _forward_any(x_flat, w, absmax, code, blocksize, n, lora_A, lora_B, scaling, bias)
    return out.view(x.shape[:-1] + (n,)), (x_flat, lora_A, lora_B, w, absmax, code), blocksize


def _forward_any(x_flat, w, absmax, code, blocksize, n, lora_A, lora_B, scaling, bias):
    """Few rows, and what the training linear does not take."""
    (m, k), r, dt = x_flat.shape, lora_A.shape[0], x_flat.dtype
    out = torch.empty((m, n), device=x_flat.device, dtype=dt)
    if m == 0 or n == 0:
        return out
    gemm_ok = m <= fused_forward_rows(k) and ops.nf4_gemm_supported(m, n, k, r, blocksize)
    if gemm_ok or (dt == torch.bfloat16
                   and ops.nf4_linear_plan(m, n, k, r, 1, blocksize) is not None):
        return ops.nf4_lora_linear(x_flat, w, absmax, code, blocksize, n, bias=bias,
                                   lora_a=lora_A, lora_b=lora_B, scaling=scaling, out=out)
    # W dequantized once (bit-exact), then GEMMs with the kernel's rounding
    # points (lora_forward.py:246-257): dt(x W^T), + bias, t = dt(x A^T),
    # u = dt(dt(t B^T) * dt(scaling)), y = dt(acc + u), dt = bf16 or float16
    wb = ops.nf4_dequant(w, absmax, code, n * k, blocksize, dtype=dt).view(n, k)
    acc = F.linear(x_flat, wb)
    if bias is not None:
        acc = acc + bias.to(acc.dtype)
    u = F.linear(F.linear(x_flat, lora_A), lora_B)
    return torch.add(acc, u * _scalar_as(scaling, dt))


class FusedLoRAFunction(torch.autograd.Function):
    """Forward = one fused NF4+LoRA kernel launch (``lora_forward.py:653-759``);
    backward = the reference's gradients (``:761-930``), float32 accumulation
    and one rounding per result or intermediate."""

    @staticmethod
    def forward(ctx, x, weight_4bit, quant_state, lora_A, lora_B, scaling, bias):
        scaling = float(scaling)
        out, saved, blocksize = _run_forward(x, weight_4bit, quant_state, lora_A, lora_B, scaling,
                                             bias)
        ctx.save_for_backward(*saved)
        ctx.blocksize, ctx.scaling, ctx.has_bias = blocksize, scaling, bias is not None
        ctx.x_shape = x.shape
        return out

    @staticmethod
    def backward(ctx, grad_out):
        x_flat, lora_A, lora_B, w, absmax, code = ctx.saved_tensors
        m, k = x_flat.shape
        n = lora_B.shape[0]
        dt = x_flat.dtype  # the adapters' dtype too (checked in forward)
        g = grad_out.contiguous().view(m, n)
        if g.dtype != dt:
            g = g.to(dt)
        grad_bias = (g.sum(dim=0) if ctx.has_bias and ctx.needs_input_grad[6]
                     else None)  # lora_forward.py:790
        nbytes = (_train_workspace(w, ctx.blocksize, lora_A, lora_B, x_flat, g)
                  if m > 0 and not torch.is_grad_enabled() else 0)
        if nbytes:
            need = ctx.needs_input_grad
            grad_x, grad_A, grad_B = ops.train_backward(
                x_flat, g, w, absmax, code, ctx.blocksize, lora_A.contiguous(),
                lora_B.contiguous(), ctx.scaling, need[0], need[3], need[4], nbytes)
            return (None if grad_x is None else grad_x.view(ctx.x_shape), None, None, grad_A,
                    grad_B, None, grad_bias)
        # scaled_grad = dt(g * dt(scaling)) (:836-837); grad_intermediate,
        # grad_x_lora, xA, grad_B, grad_A: dt GEMMs, float32 accumulation (:839-928)
        sg = g * _scalar_as(ctx.scaling, dt)
        gi = torch.matmul(sg, lora_B)
        gxl = torch.matmul(gi, lora_A)
        if (dt != torch.bfloat16 or m >= GRAD_X_GEMM_MIN_ROWS
                or not ops.nf4_grad_x_supported(n, k, ctx.blocksize)):
            # float16, many rows, or a shape the fused bf16 kernel does not
            # tile (the reference's masked kernel takes any shape, :262-348): W
            # dequantized once to the gradient's dtype (bit-exact HIP kernel,
            # the reference's cast of W to grad_block.dtype, :343), then a
            # plain GEMM -- the same rounding points as the fused kernel
            wb = ops.nf4_dequant(w, absmax, code, n * k, ctx.blocksize, dtype=dt).view(n, k)
            grad_x = torch.add(torch.matmul(g, wb), gxl)
        else:
            grad_x = ops.nf4_grad_x(g, w, absmax, code, ctx.blocksize, n, k, addend=gxl)
        xa = torch.matmul(x_flat, lora_A.t().contiguous())
        grad_B = torch.matmul(sg.t().contiguous(), xa)
        grad_A = torch.matmul(gi.t().contiguous(), x_flat)
        return grad_x.view(ctx.x_shape), None, None, grad_A, grad_B, None, grad_bias


def lora_fused_forward(x: torch.Tensor, base_layer=None, lora_A=None, lora_B=None,
                       scaling: Optional[float] = None, dropout=None, lora_layer=None,
                       prefer_base_layer: bool = False) -> torch.Tensor:
    """Drop-in for ``src.triton_kernels.lora_forward.lora_fused_forward``."""
    if lora_layer is not None:
        base_layer = getattr(lora_layer, "base_layer", None)
        lora_A = getattr(lora_layer, "lora_A", None)
        lora_B = getattr(lora_layer, "lora_B", None)
        scaling = getattr(lora_layer, "scaling", None)
        dropout = getattr(lora_layer, "lora_dropout", None)
    if base_layer is None or lora_A is None or lora_B is None or scaling is None:
        raise ValueError("Provide lora_layer or base_layer/lora_A/lora_B/scaling for fused LoRA.")
    dropout_p = (0.0 if dropout is None or type(dropout) is torch.nn.Identity
                 else getattr(dropout, "p", 0.0))
    if dropout_p and dropout_p > 0.0:
        raise ValueError("Dropout is not supported in lora_fused_forward.")

    weight_4bit = getattr(base_layer, "weight", None)
    lora_A_weight = getattr(lora_A, "weight", lora_A)
    lora_B_weight = getattr(lora_B, "weight", lora_B)

    if (not prefer_base_layer and weight_4bit is not None
            and getattr(weight_4bit, "quant_state", None) is not None):
        args = (x, weight_4bit, weight_4bit.quant_state, lora_A_weight, lora_B_weight,
                float(scaling), getattr(base_layer, "bias", None))
        # With nothing to record (no grad mode, no forward-mode level, no transform)
        # the autograd function's own bookkeeping, 5 us of a decode call's 25, is left out.
        if not torch.is_grad_enabled() and fwAD._current_level < 0 and \
                not torch._C._are_functorch_transforms_active():
            return _run_forward(*args)[0]
        return FusedLoRAFunction.apply(*args)

    # Adapter branch (lora_forward.py:986-1037): base layer + the two adapter
    # products, each rounded to the adapter dtype, scaled, cast, added.
    if x.ndim != 3:
        raise ValueError(f"x must be [batch, seq_len, hidden], got {x.shape}.")
    if lora_A_weight.ndim != 2 or lora_B_weight.ndim != 2:
        raise ValueError("lora_A and lora_B must be 2D weight matrices.")
    if not x.is_cuda or not lora_A_weight.is_cuda or not lora_B_weight.is_cuda:
        raise ValueError("x, lora_A and lora_B must be on CUDA device.")
    r = lora_A_weight.shape[0]
    if r <= 0:
        raise ValueError(f"LoRA rank must be > 0, got {r}.")
    if lora_A_weight.shape[1] != x.shape[-1] or lora_B_weight.shape[1] != r:
        raise ValueError("lora_A/lora_B shape mismatch.")
    base_output = base_layer(x.contiguous())
    if getattr(base_output, "requires_grad", False):
        base_output = base_output.clone()
    x_lora = x.reshape(-1, x.shape[-1]).to(lora_A_weight.dtype)
    t = (x_lora.float() @ lora_A_weight.float().t()).to(lora_A_weight.dtype)
    u = (t.float() @ lora_B_weight.float().t()).to(lora_A_weight.dtype)
    u = u * float(scaling)
    if u.dtype != base_output.dtype:
        u = u.to(base_output.dtype)
    return base_output + u.view(base_output.shape)


__all__ = ["lora_fused_forward", "FusedLoRAFunction"]
