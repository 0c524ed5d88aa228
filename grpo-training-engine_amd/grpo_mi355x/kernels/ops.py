"""Tensor-level wrappers of the C ABI (one call = one or two kernel launches).

These validate shapes/dtypes on the host (``ValueError``, like the reference's
``_validate_inputs``), pass raw device pointers and torch's current stream to
``libgrpo_hip.so``, and manage the per-device workspaces the kernels need.
"""

from __future__ import annotations

import functools

import torch

from .. import _lib

# ----------------------------------------------------------- workspaces --

_workspaces: dict[tuple[str, int], torch.Tensor] = {}


def workspace(kind: str, nbytes: int, device: torch.device) -> torch.Tensor | None:
    """A zero-initialised uint8 scratch tensor of at least ``nbytes`` per (kind, device).

    Used for the attention's split-context partials and the NF4 linear's
    split-K partial sums (no initialisation needed).  Calls on different
    streams must not run concurrently with the same workspace.
    """
    if nbytes <= 0:
        return None
    idx = device.index if device.index is not None else torch.cuda.current_device()
    key = (kind, idx)
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < nbytes:
        size = max(nbytes, 1 << 20)
        ws = torch.zeros(size, dtype=torch.uint8, device=device)
        _workspaces[key] = ws
    return ws


def reserve_workspace(kind: str, nbytes: int, device: torch.device) -> None:
    """Pre-size a workspace (call before HIP-graph capture)."""
    workspace(kind, nbytes, device)


# ------------------------------------------------------------- helpers --

def _need_cuda(*ts: torch.Tensor | None) -> None:
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("all tensors must be on the ROCm/HIP device.")


def _need_dtype(t: torch.Tensor, dtype: torch.dtype, name: str) -> None:
    if t.dtype != dtype:
        raise ValueError(f"{name} must be {dtype}, got {t.dtype}.")


def _need_nf4(packed: torch.Tensor, absmax: torch.Tensor, code: torch.Tensor) -> None:
    """The device and types of a packed weight, its float32 absmax and its codebook."""
    if not (packed.is_cuda and absmax.is_cuda and code.is_cuda and packed.dtype == torch.uint8
            and absmax.dtype == torch.float32 and code.dtype == torch.float32):
        _need_cuda(packed, absmax, code)
        _need_dtype(packed, torch.uint8, "packed weight")
        _need_dtype(absmax, torch.float32, "absmax")
        _need_dtype(code, torch.float32, "code")


# --------------------------------------------------------------- NF4 ---

def nf4_absmax_expand(absmax_q: torch.Tensor, code2: torch.Tensor, absmax2: torch.Tensor,
                      blocksize2: int, offset: float) -> torch.Tensor:
    """Float32 absmax of a double-quantized NF4 state (``lora_forward.py:187-199``):
    ``fma(code2[absmax_q[i]], absmax2[i // blocksize2], offset)`` per block."""
    lib = _lib.device_library()
    _need_cuda(absmax_q, code2, absmax2)
    _need_dtype(absmax_q, torch.uint8, "nested absmax")
    _need_dtype(code2, torch.float32, "state2 code")
    _need_dtype(absmax2, torch.float32, "state2 absmax")
    n = absmax_q.numel()
    if code2.numel() != 256:
        raise ValueError("state2 code must have 256 entries.")
    if absmax2.numel() * blocksize2 < n:
        raise ValueError("state2 absmax too short for the nested absmax.")
    q, c2, a2 = absmax_q.contiguous(), code2.contiguous(), absmax2.contiguous()
    out = torch.empty(n, dtype=torch.float32, device=absmax_q.device)
    rc = lib.grpo_nf4_absmax_expand(q.data_ptr(), c2.data_ptr(), a2.data_ptr(), int(blocksize2),
                                    float(offset), n, out.data_ptr(),
                                    _lib.stream_handle(absmax_q.device))
    _lib.check(rc, "grpo_nf4_absmax_expand")
    return out


def nf4_dequant(packed: torch.Tensor, absmax: torch.Tensor, code: torch.Tensor, numel: int,
                blocksize: int, out: torch.Tensor | None = None,
                dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """Bit-exact NF4 dequantization to a flat tensor of ``numel`` elements:
    ``dtype(code[q] * absmax)``, bf16 or float16 (round to nearest even)."""
    if dtype not in (torch.bfloat16, torch.float16):
        raise ValueError(f"dequantization to bfloat16 or float16, got {dtype}.")
    lib = _lib.device_library()
    _need_nf4(packed, absmax, code)
    if packed.numel() * 2 < numel:
        raise ValueError(f"packed weight holds {packed.numel() * 2} nibbles, need {numel}.")
    if absmax.numel() * blocksize < numel:
        raise ValueError("absmax too short for numel/blocksize.")
    if code.numel() != 16:
        raise ValueError("code must have 16 entries.")
    packed, absmax, code = packed.contiguous(), absmax.contiguous(), code.contiguous()
    if out is None:
        out = torch.empty(numel, dtype=dtype, device=packed.device)
    elif out.dtype != dtype:
        raise ValueError(f"out must be {dtype}.")
    fn = lib.grpo_nf4_dequant_f16 if dtype == torch.float16 else lib.grpo_nf4_dequant
    rc = fn(packed.data_ptr(), absmax.data_ptr(), code.data_ptr(), out.data_ptr(), numel,
            blocksize, _lib.stream_handle(packed.device))
    _lib.check(rc, "grpo_nf4_dequant")
    return out


def nf4_dequant_t_supported(packed: torch.Tensor, n: int, k: int, blocksize: int) -> bool:
    """Weights ``nf4_dequant_t`` takes."""
    return (blocksize >= 32 and blocksize & (blocksize - 1) == 0 and k % 32 == 0 and n % 8 == 0
            and packed.data_ptr() % 16 == 0)


def nf4_dequant_t(packed: torch.Tensor, absmax: torch.Tensor, code: torch.Tensor, n: int, k: int,
                  blocksize: int, dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """``nf4_dequant`` of W [n, k], stored transposed: a contiguous [k, n] tensor."""
    if dtype not in (torch.bfloat16, torch.float16):
        raise ValueError(f"dequantization to bfloat16 or float16, got {dtype}.")
    lib = _lib.device_library()
    _need_nf4(packed, absmax, code)
    if packed.numel() * 2 < n * k or absmax.numel() * blocksize < n * k:
        raise ValueError("packed weight or absmax too short for [n, k].")
    if code.numel() != 16:
        raise ValueError("code must have 16 entries.")
    packed, absmax, code = packed.contiguous(), absmax.contiguous(), code.contiguous()
    out = torch.empty((k, n), dtype=dtype, device=packed.device)
    _lib.check(lib.grpo_nf4_dequant_t(
        packed.data_ptr(), absmax.data_ptr(), code.data_ptr(), out.data_ptr(), n, k, blocksize,
        int(dtype == torch.float16), _lib.stream_handle(packed.device)), "grpo_nf4_dequant_t")
    return out


def nf4_lora_train_workspace_bytes(m: int, n: int, k: int, r: int, blocksize: int) -> int:
    """Workspace of ``nf4_lora_train_forward`` / ``_backward`` (0: unsupported shape)."""
    return _lib.library().grpo_nf4_lora_train_workspace_bytes(m, n, k, r, blocksize)


def _check_train(x, packed, absmax, code, blocksize, lora_a, lora_b, others) -> int:
    """Shape and dtype checks of the training linear; its workspace bytes."""
    _need_cuda(x, packed, absmax, code, lora_a, lora_b, *others)
    m, k = x.shape
    n, r = lora_b.shape
    if lora_a.shape != (r, k):
        raise ValueError("lora_A must be [r, K] and lora_B [N, r].")
    if x.dtype not in (torch.bfloat16, torch.float16):
        raise ValueError(f"bfloat16 or float16 tensors required, got {x.dtype}.")
    for t in (x, lora_a, lora_b, *others):
        if t is not None and (t.dtype != x.dtype or not t.is_contiguous()):
            raise ValueError("all tensors must be contiguous and of one dtype.")
    _need_dtype(packed, torch.uint8, "packed weight")
    _need_dtype(absmax, torch.float32, "absmax")
    if packed.numel() * 2 < n * k or absmax.numel() * blocksize < n * k or code.numel() != 16:
        raise ValueError("packed weight or absmax too short for [N, K], or not a 4-bit codebook.")
    return nf4_lora_train_workspace_bytes(m, n, k, r, int(blocksize))


def train_forward(x, packed, absmax, code, blocksize, lora_a, lora_b, scaling, bias, nbytes):
    """``nf4_lora_train_forward`` of checked arguments (``nbytes``: their workspace)."""
    (m, k), (n, r), dev = x.shape, lora_b.shape, x.device
    y = torch.empty((m, n), dtype=x.dtype, device=dev)
    ws = torch.empty(nbytes or 16, dtype=torch.uint8, device=dev)
    rc = _lib.device_library().grpo_nf4_lora_train_forward(
        x.data_ptr(), k, packed.data_ptr(), absmax.data_ptr(), code.data_ptr(), blocksize,
        None if bias is None else bias.data_ptr(), lora_a.data_ptr(), lora_b.data_ptr(), r,
        scaling, y.data_ptr(), n, m, n, k, x.dtype == torch.float16, ws.data_ptr(), nbytes,
        _lib.stream_handle(dev))
    if rc:
        _lib.check(rc, "grpo_nf4_lora_train_forward")
    return y


def train_backward(x, grad, packed, absmax, code, blocksize, lora_a, lora_b, scaling, want_x,
                   want_a, want_b, nbytes):
    """``nf4_lora_train_backward`` of checked arguments (``nbytes``: their workspace)."""
    (m, k), (n, r), dev = x.shape, lora_b.shape, x.device
    gx = torch.empty_like(x) if want_x else None
    ga = torch.empty_like(lora_a) if want_a else None
    gb = torch.empty_like(lora_b) if want_b else None
    ws = torch.empty(nbytes or 16, dtype=torch.uint8, device=dev)
    rc = _lib.device_library().grpo_nf4_lora_train_backward(
        x.data_ptr(), k, grad.data_ptr(), n, packed.data_ptr(), absmax.data_ptr(),
        code.data_ptr(), blocksize, lora_a.data_ptr(), lora_b.data_ptr(), r, scaling, m, n, k,
        x.dtype == torch.float16, None if gx is None else gx.data_ptr(), k,
        None if ga is None else ga.data_ptr(), None if gb is None else gb.data_ptr(),
        ws.data_ptr(), nbytes, _lib.stream_handle(dev))
    if rc:
        _lib.check(rc, "grpo_nf4_lora_train_backward")
    return gx, ga, gb


def nf4_lora_train_forward(x: torch.Tensor, packed: torch.Tensor, absmax: torch.Tensor,
                           code: torch.Tensor, blocksize: int, lora_a: torch.Tensor,
                           lora_b: torch.Tensor, scaling: float,
                           bias: torch.Tensor | None = None) -> torch.Tensor:
    """``y [M, N]`` of the NF4 + LoRA linear for training batches (bf16 or float16)."""
    _lib.device_library()
    nbytes = _check_train(x, packed, absmax, code, blocksize, lora_a, lora_b, (bias,))
    if bias is not None and bias.numel() != lora_b.shape[0]:
        raise ValueError(f"bias must have {lora_b.shape[0]} elements.")
    return train_forward(x, packed, absmax, code, int(blocksize), lora_a, lora_b, float(scaling),
                         bias, nbytes)


def nf4_lora_train_backward(x: torch.Tensor, grad: torch.Tensor, packed: torch.Tensor,
                            absmax: torch.Tensor, code: torch.Tensor, blocksize: int,
                            lora_a: torch.Tensor, lora_b: torch.Tensor, scaling: float,
                            want_x: bool = True, want_a: bool = True, want_b: bool = True):
    """(grad_x, grad_A, grad_B) of the NF4 + LoRA linear (None where not wanted)."""
    _lib.device_library()
    nbytes = _check_train(x, packed, absmax, code, blocksize, lora_a, lora_b, (grad,))
    if grad.shape != (x.shape[0], lora_b.shape[0]):
        raise ValueError(f"grad must be [{x.shape[0]}, {lora_b.shape[0]}], got "
                         f"{tuple(grad.shape)}.")
    return train_backward(x, grad, packed, absmax, code, int(blocksize), lora_a, lora_b,
                          float(scaling), want_x, want_a, want_b, nbytes)


def nf4_grad_x_supported(n: int, k: int, blocksize: int) -> bool:
    """Shapes ``grpo_nf4_grad_x`` takes: N a multiple of 32, K of 128, blocksize of 8."""
    return n > 0 and k > 0 and n % 32 == 0 and k % 128 == 0 and blocksize > 0 \
        and blocksize % 8 == 0


def nf4_grad_x(grad: torch.Tensor, packed: torch.Tensor, absmax: torch.Tensor,
               code: torch.Tensor, blocksize: int, n: int, k: int,
               addend: torch.Tensor | None = None) -> torch.Tensor:
    """``bf16(grad [M, n] @ W_nf4 [n, k])`` (+ ``addend`` [M, k], rounded once more)."""
    lib = _lib.device_library()
    _need_cuda(grad, packed, absmax, code, addend)
    _need_dtype(grad, torch.bfloat16, "grad")
    _need_dtype(packed, torch.uint8, "packed weight")
    _need_dtype(absmax, torch.float32, "absmax")
    if grad.ndim != 2 or grad.shape[1] != n:
        raise ValueError(f"grad must be [M, {n}], got {tuple(grad.shape)}.")
    if packed.numel() * 2 < n * k or absmax.numel() * blocksize < n * k:
        raise ValueError("packed weight or absmax too short for [n, k].")
    if code.numel() != 16:
        raise ValueError("code must have 16 entries.")
    m = grad.shape[0]
    grad = grad.contiguous()
    if addend is not None:
        _need_dtype(addend, torch.bfloat16, "addend")
        if tuple(addend.shape) != (m, k):
            raise ValueError(f"addend must be [{m}, {k}], got {tuple(addend.shape)}.")
        addend = addend.contiguous()
    out = torch.empty((m, k), dtype=torch.bfloat16, device=grad.device)
    rc = lib.grpo_nf4_grad_x(grad.data_ptr(), n, packed.data_ptr(), absmax.data_ptr(),
                             code.contiguous().data_ptr(), blocksize, m, n, k,
                             None if addend is None else addend.data_ptr(), k, out.data_ptr(), k,
                             _lib.stream_handle(grad.device))
    _lib.check(rc, "grpo_nf4_grad_x")
    return out


def nf4_lora_linear(x2d: torch.Tensor, packed: torch.Tensor, absmax: torch.Tensor,
                    code: torch.Tensor, blocksize: int, n: int, bias: torch.Tensor | None = None,
                    lora_a: torch.Tensor | None = None, lora_b: torch.Tensor | None = None,
                    scaling: float = 1.0, out: torch.Tensor | None = None) -> torch.Tensor:
    """``y[M, N] = W_nf4(x) + bias + B(A(x)) * scaling`` (bf16).

    Up to 32 rows: the one-launch tile kernel (``grpo_nf4_tile_linear``, LoRA A
    packed once per tensor version); up to 64 rows split-K partial sums +
    finish (two launches); beyond, the NF4 GEMM (one launch, or K slices +
    finish when the tiles are few); one generic launch for other shapes.
    float16 x (with float16 LoRA and bias) runs the NF4 GEMM's float16 form for
    any M (``y`` float16).
    """
    lib = _lib.device_library()
    if not (x2d.is_cuda and packed.is_cuda and absmax.is_cuda and code.is_cuda):
        raise ValueError("all tensors must be on the ROCm/HIP device.")
    _need_cuda(bias, lora_a, lora_b)
    if x2d.ndim != 2:
        raise ValueError(f"x must be 2-D [M, K], got {tuple(x2d.shape)}.")
    if x2d.dtype == torch.float16:
        return _nf4_lora_linear_f16(lib, x2d, packed, absmax, code, blocksize, n, bias, lora_a,
                                    lora_b, scaling, out)
    bf = torch.bfloat16
    _need_dtype(x2d, bf, "x")
    m, k = x2d.shape
    if x2d.stride(1) != 1:
        x2d = x2d.contiguous()
    r = 0
    if lora_a is not None:
        r = lora_a.shape[0]
        if lora_a.shape != (r, k) or lora_b is None or lora_b.shape != (n, r):
            raise ValueError("lora_A must be [r, K] and lora_B [N, r].")
        if lora_a.dtype != bf or lora_b.dtype != bf:
            _need_dtype(lora_a, bf, "lora_A")
            _need_dtype(lora_b, bf, "lora_B")
        lora_a, lora_b = lora_a.contiguous(), lora_b.contiguous()
    if bias is not None:
        if bias.numel() != n:
            raise ValueError(f"bias must have {n} elements.")
        if bias.dtype != bf or not bias.is_contiguous():
            bias = bias.to(bf).contiguous()
    if packed.numel() * 2 < n * k:
        raise ValueError("packed weight smaller than N*K/2 bytes.")
    dev, ldx, xp, wp = x2d.device, x2d.stride(0), x2d.data_ptr(), packed.data_ptr()
    if out is None:
        out = torch.empty((m, n), dtype=bf, device=dev)
    elif out.shape != (m, n) or out.stride(1) != 1 or out.dtype != bf:
        raise ValueError("out must be a bf16 [M, N] tensor with unit column stride.")
    bp, st = _lib.ptr(bias), _lib.stream_handle(dev)
    if m <= TILE_MAX_ROWS and ldx % 8 == 0 and xp % 16 == 0 and wp % 16 == 0 and \
            lib.grpo_nf4_tile_supported(m, n, k, r, 1, int(blocksize)):
        # decode batches: the one-launch tile linear (LoRA A in its packed
        # order, built once per A version)
        rc = lib.grpo_nf4_tile_linear_one(
            xp, ldx, wp, absmax.data_ptr(), code.data_ptr(), int(blocksize), bp,
            packed_lora_a(lora_a).data_ptr() if r > 0 else None, _lib.ptr(lora_b), r,
            float(scaling), out.data_ptr(), out.stride(0), m, n, k, st)
        _lib.check(rc, "grpo_nf4_tile_linear")
        return out
    nbytes = int(lib.grpo_nf4_lora_linear_workspace_bytes(m, n, k, r, 1, int(blocksize)))
    ws = workspace("nf4_linear", nbytes, dev)
    rc = lib.grpo_nf4_lora_linear(
        xp, ldx, wp, absmax.data_ptr(), code.data_ptr(), int(blocksize), bp, _lib.ptr(lora_a),
        _lib.ptr(lora_b), r, float(scaling), out.data_ptr(), out.stride(0), m, n, k, _lib.ptr(ws),
        0 if ws is None else ws.numel(), st)
    _lib.check(rc, "grpo_nf4_lora_linear")
    return out


TILE_MAX_ROWS = 32  # rows up to which nf4_lora_linear runs the one-launch tile kernel

# Packed LoRA A per live A tensor: id(A) -> (weakref to A, A._version, packed).
# An entry is valid while A is the same object at the same version (an
# optimizer step updates A in place and bumps the version) and is dropped
# when A is freed.
_packed_a: dict[int, tuple] = {}


def packed_lora_a(a: torch.Tensor) -> torch.Tensor:
    """``pack_lora_a(a)``, cached per A tensor and version."""
    import weakref

    key = id(a)
    e = _packed_a.get(key)
    if e is not None and e[0]() is a and e[1] == a._version:
        return e[2]
    p = pack_lora_a(a)
    _packed_a[key] = (weakref.ref(a, lambda _r, k=key: _packed_a.pop(k, None)), a._version, p)
    return p


def pack_lora_a(a: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """LoRA A [r, K] bf16 in the MFMA order the one-launch linear reads
    (``grpo_nf4_tile_pack_lora_a``); valid until A changes."""
    lib = _lib.device_library()
    _need_cuda(a)
    _need_dtype(a, torch.bfloat16, "lora_A")
    r, k = a.shape
    a = a.contiguous()
    nbytes = int(lib.grpo_nf4_tile_packed_lora_a_bytes(k))
    if out is None:
        out = torch.empty(nbytes // 2, dtype=torch.bfloat16, device=a.device)
    elif out.numel() * out.element_size() < nbytes:
        raise ValueError(f"packed LoRA A needs {nbytes} bytes.")
    _lib.check(lib.grpo_nf4_tile_pack_lora_a(a.data_ptr(), r, k, k, out.data_ptr(),
                                             _lib.stream_handle(a.device)), "pack_lora_a")
    return out


def tile_linear_desc(m: int, k: int, seg_rows, biases=None, lora_a=None, lora_b=None,
                     scaling: float = 1.0):
    """``grpo_tile_linear_t`` of an [M, K] x [N = sum(seg_rows), K] NF4 linear:
    per segment an optional bf16 bias and LoRA A [r, K] / B [rows, r] (device
    tensors, kept referenced by the returned descriptor)."""
    d = _lib.TileLinear()
    d.M, d.K, d.nseg = m, k, len(seg_rows)
    if not 1 <= d.nseg <= _lib.MAX_SEGMENTS:
        raise ValueError(f"1..{_lib.MAX_SEGMENTS} segments, got {d.nseg}.")
    keep = []
    end, r = 0, 0
    for i, rows in enumerate(seg_rows):
        end += int(rows)
        d.seg_end[i] = end
        if biases is not None and biases[i] is not None:
            b = biases[i].to(torch.bfloat16).contiguous()
            if b.numel() != rows:
                raise ValueError(f"bias {i} must have {rows} elements.")
            keep.append(b)
            d.bias[i] = b.data_ptr()
        if lora_a is not None:
            a, bb = lora_a[i].contiguous(), lora_b[i].contiguous()
            r = a.shape[0]
            if a.shape != (r, k) or bb.shape != (rows, r):
                raise ValueError("lora_A must be [r, K] and lora_B [rows, r] per segment.")
            _need_dtype(a, torch.bfloat16, "lora_A")
            _need_dtype(bb, torch.bfloat16, "lora_B")
            ap = pack_lora_a(a)
            keep += [ap, bb]
            d.lora_a[i], d.lora_b[i] = ap.data_ptr(), bb.data_ptr()
    d.N, d.r, d.scaling = end, r, float(scaling)
    d._keep = keep
    return d


def nf4_tile_linear(x: torch.Tensor, packed: torch.Tensor, absmax: torch.Tensor,
                    code: torch.Tensor, blocksize: int, desc, out: torch.Tensor | None = None,
                    norm: tuple | None = None, residual: torch.Tensor | None = None,
                    sumsq: torch.Tensor | None = None) -> torch.Tensor:
    """The one-launch NF4 (+ LoRA) linear (``grpo_nf4_tile_linear*``) for a
    ``tile_linear_desc`` descriptor.

    ``norm = (sumsq [M, G] float32, weight [K] bf16, eps)``: ``x`` is h and the
    kernel stages RMSNorm(h).  ``residual`` ([M, N] bf16, may be ``out``):
    ``out = bf16(residual + y)`` and ``sumsq`` ([M, G] float32, G =
    ``grpo_nf4_tile_sumsq_groups``) receives the per-group sums of ``out**2``."""
    lib = _lib.device_library()
    _need_cuda(x, packed, absmax, code, out, residual, sumsq)
    _need_dtype(x, torch.bfloat16, "x")
    m, n, k = desc.M, desc.N, desc.K
    if x.ndim != 2 or x.shape != (m, k) or x.stride(1) != 1:
        raise ValueError(f"x must be [{m}, {k}] with unit column stride.")
    if out is None:
        out = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    if out.shape != (m, n) or out.stride(1) != 1 or out.dtype != torch.bfloat16:
        raise ValueError("out must be a bf16 [M, N] tensor with unit column stride.")
    st = _lib.stream_handle(x.device)
    args = (packed.data_ptr(), absmax.data_ptr(), code.data_ptr(), int(blocksize),
            ctypes_byref(desc))
    if norm is not None:
        ss, w, eps = norm
        rc = lib.grpo_nf4_tile_linear_norm(x.data_ptr(), x.stride(0), ss.data_ptr(), ss.shape[1],
                                           w.data_ptr(), float(eps), *args, out.data_ptr(),
                                           out.stride(0), st)
    elif residual is not None:
        if sumsq is None or residual.stride() != out.stride():
            raise ValueError("residual needs sumsq and the row stride of out.")
        rc = lib.grpo_nf4_tile_linear_residual(x.data_ptr(), x.stride(0), *args,
                                               residual.data_ptr(), out.data_ptr(), out.stride(0),
                                               sumsq.data_ptr(), st)
    else:
        rc = lib.grpo_nf4_tile_linear(x.data_ptr(), x.stride(0), *args, out.data_ptr(),
                                      out.stride(0), st)
    _lib.check(rc, "grpo_nf4_tile_linear")
    return out


def ctypes_byref(obj):
    import ctypes

    return ctypes.byref(obj)


def _nf4_lora_linear_f16(lib, x2d, packed, absmax, code, blocksize, n, bias, lora_a, lora_b,
                         scaling, out):
    """float16 x and adapters: the NF4 GEMM's float16 form (``grpo_nf4_gemm_f16``,
    every rounding point float16, any M)."""
    m, k = x2d.shape
    if x2d.stride(1) != 1 or x2d.stride(0) % 8 or x2d.data_ptr() % 16:
        x2d = x2d.contiguous()
    r = 0
    if lora_a is not None:
        r = lora_a.shape[0]
        if lora_a.shape != (r, k) or lora_b is None or lora_b.shape != (n, r):
            raise ValueError("lora_A must be [r, K] and lora_B [N, r].")
        _need_dtype(lora_a, torch.float16, "lora_A")
        _need_dtype(lora_b, torch.float16, "lora_B")
        lora_a, lora_b = lora_a.contiguous(), lora_b.contiguous()
    if bias is not None:
        if bias.numel() != n:
            raise ValueError(f"bias must have {n} elements.")
        bias = bias.to(torch.float16).contiguous()
    if packed.numel() * 2 < n * k:
        raise ValueError("packed weight smaller than N*K/2 bytes.")
    if not nf4_gemm_supported(m, n, k, r, blocksize):
        raise ValueError(f"float16 NF4 linear: shape M={m} N={n} K={k} r={r} blocksize="
                         f"{blocksize} is outside the NF4 GEMM (K % 32, r <= 32).")
    if out is None:
        out = torch.empty((m, n), dtype=torch.float16, device=x2d.device)
    elif out.shape != (m, n) or out.stride(1) != 1 or out.dtype != torch.float16:
        raise ValueError("out must be a float16 [M, N] tensor with unit column stride.")
    if m == 0 or n == 0:
        return out
    rc = lib.grpo_nf4_gemm_f16(
        x2d.data_ptr(), x2d.stride(0), packed.data_ptr(), absmax.data_ptr(), code.data_ptr(),
        int(blocksize), _lib.ptr(bias), _lib.ptr(lora_a), _lib.ptr(lora_b), r, float(scaling),
        out.data_ptr(), out.stride(0), m, n, k, _lib.stream_handle(x2d.device))
    _lib.check(rc, "grpo_nf4_gemm_f16")
    return out


def nf4_gemm_supported(m: int, n: int, k: int, r: int, blocksize: int) -> bool:
    """True if the NF4 GEMM (``grpo_nf4_gemm``; more than 64 rows) takes this
    shape (alignment aside)."""
    return bool(_lib.library().grpo_nf4_gemm_supported(m, n, k, r, int(blocksize)))


def nf4_linear_plan(m: int, n: int, k: int, r: int, nseg: int,
                    blocksize: int) -> tuple[int, int, int] | None:
    """(splits, part_bytes, tpart_bytes) of the split-K path, or None if the
    shape takes the generic kernel."""
    import ctypes

    s, pb, tb = ctypes.c_int(0), ctypes.c_size_t(0), ctypes.c_size_t(0)
    rc = _lib.library().grpo_nf4_linear_plan(m, n, k, r, nseg, blocksize, ctypes.byref(s),
                                             ctypes.byref(pb), ctypes.byref(tb))
    if rc != 0:
        return None
    return s.value, pb.value, tb.value


# ----------------------------------------------------------- paged KV ---

_BF16, _I32 = torch.bfloat16, torch.int32


def _check_cache(k_cache: torch.Tensor, v_cache: torch.Tensor) -> torch.Size:
    shape = k_cache.shape
    if len(shape) != 4 or v_cache.ndim != 4:
        raise ValueError("k_cache/v_cache must be [num_blocks, heads, block, head_dim].")
    if shape != v_cache.shape:
        raise ValueError("k_cache and v_cache must have identical shapes.")
    if k_cache.dtype != _BF16 or v_cache.dtype != _BF16:
        _need_dtype(k_cache, _BF16, "k_cache")
        _need_dtype(v_cache, _BF16, "v_cache")
    if not (k_cache.is_contiguous() and v_cache.is_contiguous()):
        raise ValueError("k_cache/v_cache must be contiguous.")
    return shape


def _check_tables(block_tables: torch.Tensor, context_lens: torch.Tensor, b: int):
    """(row stride, max_blocks) of checked tables."""
    shape = block_tables.shape
    if len(shape) != 2 or shape[0] != b:
        raise ValueError("block_tables must be [batch, max_blocks].")
    if context_lens.shape != (b,):
        raise ValueError("context_lens must be [batch].")
    if block_tables.dtype != _I32 or context_lens.dtype != _I32:
        _need_dtype(block_tables, _I32, "block_tables")
        _need_dtype(context_lens, _I32, "context_lens")
    row, col = block_tables.stride()
    if col != 1 or not context_lens.is_contiguous():
        raise ValueError("block_tables rows and context_lens must be contiguous.")
    return row, shape[1]


def paged_kv_append(k_new: torch.Tensor, v_new: torch.Tensor, k_cache: torch.Tensor,
                    v_cache: torch.Tensor, block_tables: torch.Tensor,
                    context_lens: torch.Tensor) -> None:
    """Write ``k_new/v_new [B, Hkv, D]`` at slot ``context_lens[b]`` of each sequence."""
    lib = _lib.device_library()
    if not (k_new.is_cuda and v_new.is_cuda and k_cache.is_cuda and v_cache.is_cuda
            and block_tables.is_cuda and context_lens.is_cuda):
        raise ValueError("all tensors must be on the ROCm/HIP device.")
    nb, hkv, bs, d = _check_cache(k_cache, v_cache)
    shape = k_new.shape
    if shape != v_new.shape or len(shape) != 3 or shape[1:] != (hkv, d):
        raise ValueError(f"k_new/v_new must be [B, {hkv}, {d}].")
    b = shape[0]
    row, max_blocks = _check_tables(block_tables, context_lens, b)
    k_new = k_new.to(_BF16)
    v_new = v_new.to(_BF16)
    st = k_new.stride()
    if st[2] != 1 or st != v_new.stride():
        k_new, v_new = k_new.contiguous(), v_new.contiguous()
        st = k_new.stride()
    rc = lib.grpo_paged_kv_append(
        k_new.data_ptr(), v_new.data_ptr(), st[0], st[1], k_cache.data_ptr(),
        v_cache.data_ptr(), nb, block_tables.data_ptr(), row, context_lens.data_ptr(), b, hkv, d,
        bs, max_blocks, _lib.stream_handle(k_cache.device))
    _lib.check(rc, "grpo_paged_kv_append")


def paged_attention_workspace_bytes(b: int, hq: int, hkv: int, d: int, bs: int,
                                    max_blocks: int) -> int:
    return int(_lib.library().grpo_paged_attn_workspace_bytes(b, hq, hkv, d, bs, max_blocks))


# One-launch attention (grpo_paged_attn_decode_merged): per device, the int32
# arrival counters of the in-kernel merge (zero, left zero by every call) and
# the XCD error word.  Calls on one device share them, as they share the
# workspace: calls that overlap on two streams must be ordered by the caller.
_attn_merge: dict = {}
ATTN_ONE_LAUNCH = True


@functools.lru_cache(maxsize=1024)
def _attn_plan(b: int, hq: int, hkv: int, d: int, bs: int, max_blocks: int) -> tuple[int, int]:
    """(workspace bytes, merge counters) of an attention call of this shape."""
    lib = _lib.library()
    return (int(lib.grpo_paged_attn_workspace_bytes(b, hq, hkv, d, bs, max_blocks)),
            max(int(lib.grpo_paged_attn_merge_counter_bytes(b, hkv)) // 4, 1))


def _attn_merge_state(device, need: int):
    st = _attn_merge.get(device)
    if st is None or st[0].numel() < need:
        err = st[1] if st is not None else torch.zeros(1, dtype=torch.int32, device=device)
        st = (torch.zeros(need, dtype=torch.int32, device=device), err)
        _attn_merge[device] = st
    return st


def attention_handover_check(device=None) -> None:
    """Check the one-launch attention calls made so far on ``device`` (host
    sync): their in-kernel merge hands each (sequence, KV head)'s split
    partials to the last-arriving split through an L2 counter, which is
    correct only when the pair's splits ran on one XCD.  The kernel flags a
    pair that did not, and such a pair leaves its counter non-zero; either
    raises ``RuntimeError`` (those calls' outputs are not valid), clears the
    state and turns the one-launch form off (``ATTN_ONE_LAUNCH``) for later
    calls, which then take the split launch + merge launch."""
    global ATTN_ONE_LAUNCH
    keys = [torch.device(device)] if device is not None else list(_attn_merge)
    for key in keys:
        st = _attn_merge.get(key)
        if st is None:
            continue
        if int(st[1].item()) != 0 or bool((st[0] != 0).any()):
            st[0].zero_()
            st[1].zero_()
            ATTN_ONE_LAUNCH = False
            raise RuntimeError("paged attention: the context splits of a (sequence, KV head) "
                               "pair did not run on one XCD; outputs of the one-launch calls "
                               "since the last check are not valid (one-launch form now off)")


def paged_attention_decode(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                           block_tables: torch.Tensor, context_lens: torch.Tensor, scale: float,
                           out_dtype: torch.dtype = torch.float32,
                           out: torch.Tensor | None = None,
                           no_alloc: bool = False) -> torch.Tensor:
    """GQA paged decode attention; ``q [B, Hq, D]`` bf16 -> ``[B, Hq, D]`` out_dtype.

    One launch (``grpo_paged_attn_decode_merged``: the last-arriving context
    split of each (sequence, KV head) merges the pair's splits) while
    ``ATTN_ONE_LAUNCH``; ``attention_handover_check`` verifies those calls.
    ``no_alloc`` calls ``grpo_paged_attn_decode_noalloc`` (split partials in the
    library's per-GPU scratch array, no workspace, split + merge launches);
    ``out`` must then be given for the call to allocate nothing at all."""
    lib = _lib.device_library()
    if not (q.is_cuda and k_cache.is_cuda and v_cache.is_cuda and block_tables.is_cuda
            and context_lens.is_cuda):
        raise ValueError("all tensors must be on the ROCm/HIP device.")
    nb, hkv, bs, d = _check_cache(k_cache, v_cache)
    shape, dev = q.shape, q.device
    if len(shape) != 3 or shape[2] != d:
        raise ValueError(f"q must be [B, Hq, {d}].")
    b, hq, _ = shape
    if hq % hkv != 0:
        raise ValueError(f"query heads ({hq}) must be a multiple of KV heads ({hkv}).")
    row, max_blocks = _check_tables(block_tables, context_lens, b)
    q = q.to(_BF16)
    qsb, qsh, qsd = q.stride()
    if qsd != 1:
        q = q.contiguous()
        qsb, qsh, _ = q.stride()
    if out_dtype not in (torch.float32, _BF16):
        raise ValueError("out_dtype must be float32 or bfloat16.")
    if out is None:
        out = torch.empty(shape, dtype=out_dtype, device=dev)
    elif out.shape != (b, hq, d) or not out.is_contiguous() or out.dtype != out_dtype:
        raise ValueError("out must be a contiguous [B, Hq, D] tensor of out_dtype.")
    st = _lib.stream_handle(dev)
    args = (q.data_ptr(), qsb, qsh, k_cache.data_ptr(), v_cache.data_ptr(), nb,
            block_tables.data_ptr(), row, context_lens.data_ptr(), out.data_ptr(),
            1 if out_dtype == _BF16 else 0, b, hq, hkv, d, bs, max_blocks, float(scale))
    if no_alloc:
        _lib.check(lib.grpo_paged_attn_decode_noalloc(*args, st),
                   "grpo_paged_attn_decode_noalloc")
        return out
    nbytes, counters = _attn_plan(b, hq, hkv, d, bs, max_blocks)
    ws = workspace("paged_attn", nbytes, dev)
    args += (_lib.ptr(ws), 0 if ws is None else ws.numel())
    if ATTN_ONE_LAUNCH:
        cnt, err = _attn_merge_state(dev, counters)
        _lib.check(lib.grpo_paged_attn_decode_merged(*args, cnt.data_ptr(), err.data_ptr(), st),
                   "grpo_paged_attn_decode_merged")
    else:
        _lib.check(lib.grpo_paged_attn_decode(*args, st), "grpo_paged_attn_decode")
    return out
