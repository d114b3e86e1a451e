"""Sparse-mask attention: the user-facing Python API, with the reference's functions and arguments.

Mirrors ``python/sparse_attention.py`` of the reference (line numbers below refer to it):

* ``sparse_attention(q, k, v, mask)``       :120-154  autograd-aware entry point
* ``sparse_attention_func(q, k, v, mask)``  :157-177  inference-only variant (no LSE, no graph)
* ``pack_mask(mask)``                       :184-201  bool [B,H,N,N] -> int32 [B,H,N,ceil(N/32)]
* ``SparseAttentionFunction``               :49-113   what ``sparse_attention`` differentiates, with the scale given
* ``sparse_attention_ref``                  :24-42    the plain-PyTorch statement of the operator
* ``generate_random_sparse_mask``           :204-211

``q, k, v`` are ``[B, H, N, D]`` fp16 / bf16 tensors on an MI355X, D = 64 as in the reference or any other up to
128 (multiples of 8 as they are, others zero-padded to the next multiple of 8, see below); fp32 inputs are computed in
bf16 and returned as fp32, as in the reference :140-142,151-152.  ``mask`` is a bool
``[B, H, N, N]`` tensor, True = attend.  Query rows that attend to nothing give zeros.

What differs from the reference, on purpose:

* The compute path is the HIP extension ``sparse_attn_cuda`` (same module name) and nothing else.
  Where the reference silently computes with PyTorch ops when the extension is missing or the
  tensors live on the CPU (:148-149, :65-74), this module raises ``RuntimeError``: a silent
  fallback would hide a broken build.  ``sparse_attention_ref`` stays available for callers who
  want the PyTorch formulation explicitly.
* ``q, k, v`` need not be contiguous: views whose last dimension is contiguous and whose other
  strides are multiples of 8 elements (a ``[B, N, H, D]`` buffer viewed as ``[B, H, N, D]``, slices
  of a fused qkv projection) go to the kernels as they are, where the reference would read them as
  if they were contiguous; anything else is copied with ``.contiguous()`` first.
* ``mask`` may be ``[1, 1, N, N]``, ``[B, 1, N, N]`` or ``[1, H, N, N]``: it is packed once at that
  size and shared between batch entries / heads by the kernels (the reference needs the expanded
  ``[B, H, N, N]`` tensor).  A mask passed as an ``expand``-ed view is recognised by its zero
  strides and treated the same way.
* Head dims: the kernels exist for 64 (the reference's only one), 32, 80, 96 and 128.  Any multiple of 8 in
  between runs in the next larger one as it is; any other D <= 128 is computed exactly by zero-padding q, k, v (the
  scores and the first D output columns do not change; the scale stays 1/sqrt(D)) at the price of the padding copies.
* The mask is not packed in a pass of its own: where the kernel's limits allow (any q, k, v the strided kernels take,
  N >= 16) one launch reads the bool mask itself and forms the packed words tile by
  tile, which is 15-35 % faster than pack + attention; under autograd the same launch also leaves
  the packed words behind for the backward.  Otherwise the mask is packed as the reference does.
  Results are bit-identical either way; both ways count any non-zero mask byte as True, so a bool
  tensor made by ``view`` from bytes other than 0 and 1 is read the same by both.
* Block-structured masks (sliding window, block-sparse, causal): ``tile_map(mask_packed)`` says
  which 64 x 64 blocks of the mask hold a set bit; given as ``tile_map=`` together with
  ``mask_packed=`` the forward neither loads nor computes the key tiles that hold none (the
  reference skips such a tile only after loading it, ``csrc/sparse_attention.cu:211,238-252``).
  Worth it for a mask that is used many times; ``tile_map`` returns None when too few visits would
  disappear for the walk to pay.
* ``.backward()`` works.  The reference calls a ``sparse_attn_cuda.backward`` that was never
  written (:91-94); here that function exists (HIP kernels, from the saved log-sum-exp and the packed mask: dQ and
  dK/dV, or one for a whole head).  ``backward_recompute`` states the same gradients with PyTorch
  ops (the reference's own formulas, :97-111) for cross-checks.
* ``SparseAttentionFunction`` has ``apply`` and nothing else of a ``torch.autograd.Function``: its node is native.  The node
  shows ``saved_tensors``, ``scale`` and ``tile_map``.  Forward-mode AD is refused (``NotImplementedError``), and a
  ``torch.jit`` trace records each call as one operation.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG_DIR = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if _PKG_DIR not in sys.path:
    sys.path.insert(0, _PKG_DIR)

try:
    import sparse_attn_cuda  # pybind shim over libsma_hip.so, built in-tree by buildlib.py
    HAS_CUDA_EXT = True
    _EXT_ERROR = None
except ImportError as exc:  # the API stays importable; any compute call reports the cause
    sparse_attn_cuda = None
    HAS_CUDA_EXT = False
    _EXT_ERROR = exc


def _rows(t: torch.Tensor) -> torch.Tensor:
    """t itself if the kernels can address it (contiguous last dimension, the strides of the other
    dimensions multiples of 8 elements, 16-byte aligned storage), else a contiguous copy: what a call does
    with q, k and v, by the rule that it goes by."""
    return t if sparse_attn_cuda.addressable(t) else t.contiguous()


def _require_ext(t: torch.Tensor) -> None:
    if not HAS_CUDA_EXT:
        raise RuntimeError(
            "the HIP extension sparse_attn_cuda is not built or failed to load "
            f"({_EXT_ERROR}); run `python setup.py build_ext --inplace` in {_PKG_DIR}")
    if not t.is_cuda:
        raise RuntimeError("sparse attention runs on the GPU only: move q, k, v and mask to the "
                           "device (sparse_attention_ref is the PyTorch formulation for any device)")


# ----------------------------------------------------------------------------------------------
# Plain-PyTorch statement of the operator (never called by the functions below)
# ----------------------------------------------------------------------------------------------

def sparse_attention_ref(q, k, v, mask):
    """softmax(mask ? q k^T / sqrt(D) : -inf) v with PyTorch ops, in the dtype of the inputs."""
    scale = 1.0 / math.sqrt(q.shape[-1])
    logits = (q @ k.transpose(-1, -2)) * scale
    logits = logits.masked_fill(mask.logical_not(), float("-inf"))
    probs = torch.nan_to_num(torch.softmax(logits, dim=-1), nan=0.0)   # empty rows -> zeros
    return probs @ v


# ----------------------------------------------------------------------------------------------
# autograd
# ----------------------------------------------------------------------------------------------

class SparseAttentionFunction:
    """forward = fused HIP kernel (saves LSE); backward = the HIP backward kernels.

    The autograd node itself is native (csrc/binding.cpp, SparseAttentionBackward): in a small training
    step the host is what takes time, and a node written in Python made it twice as long.  Tensors are checked as
    ``sparse_attention`` checks them, and q, k and v have one type; what is wrong raises ``RuntimeError``.

    ``mask_packed`` may be None: the mask is then read as it is by the one-launch forward, which
    leaves the packed words the backward uses (and, with ``tile_map=True``, the mask's tile map) as
    by-products, or packed first where that kernel does not apply.  ``tile_map=True`` is not the
    default because a mask without empty blocks (any random one) would pay for a by-product that
    nothing can use."""

    @staticmethod
    def apply(q, k, v, mask_packed, mask_bool, scale, seq_len, tile_map=None):
        _require_ext(q)
        if torch.jit.is_tracing():
            return _TracedCall.apply(SparseAttentionFunction.apply, q, k, v, mask_packed, mask_bool, scale, seq_len, tile_map)
        return sparse_attn_cuda.attention_function(q, k, v, mask_packed, mask_bool, scale, tile_map)


class _TracedCall(torch.autograd.Function):
    """``call(q, k, v, *rest)`` as one operation of a ``torch.jit`` trace, which records operations of PyTorch and sees
    nothing of a native call.  The call itself, made with the tracer off, and its native node do the work."""

    @staticmethod
    def forward(ctx, call, q, k, v, *rest):
        state = torch._C._get_tracing_state()
        torch._C._set_tracing_state(None)
        try:
            with torch.enable_grad():
                ctx.inputs = [t.detach().requires_grad_(wanted) for t, wanted in zip((q, k, v), ctx.needs_input_grad[1:4])]
                ctx.output = call(*ctx.inputs, *rest)
            out = ctx.output.detach()
        finally:
            torch._C._set_tracing_state(state)
        ctx.others = len(rest)
        return out.clone()              # known to the tracer, and free to be changed in place

    @staticmethod
    def backward(ctx, dout):
        grads = iter(torch.autograd.grad(ctx.output, [t for t in ctx.inputs if t.requires_grad], dout, retain_graph=True))
        return (None, *(next(grads) if t.requires_grad else None for t in ctx.inputs), *[None] * ctx.others)


def backward_recompute(q, k, v, out, lse, mask_bool, dout, scale):
    """The same gradients with PyTorch ops on the GPU from the saved log-sum-exp (the formulas of
    the reference's fallback, python/sparse_attention.py:97-111).  Not used by the autograd
    function; kept as a cross-check for users and tests."""
    qf, kf, vf, do = q.float(), k.float(), v.float(), dout.float()
    # p = exp(s - lse) on kept entries; rows that keep nothing have lse = -inf and p = 0.
    s = (qf @ kf.transpose(-1, -2)) * scale
    safe_lse = torch.where(torch.isinf(lse), torch.zeros_like(lse), lse).unsqueeze(-1)
    p = torch.exp(s - safe_lse).masked_fill(mask_bool.logical_not(), 0.0)
    dv = p.transpose(-1, -2) @ do
    dp = do @ vf.transpose(-1, -2)
    delta = (do * out.float()).sum(dim=-1, keepdim=True)      # = sum_j p_ij dp_ij
    ds = p * (dp - delta) * scale
    dq = ds @ kf
    dk = ds.transpose(-1, -2) @ qf
    return dq.to(q.dtype), dk.to(k.dtype), dv.to(v.dtype)


# ----------------------------------------------------------------------------------------------
# public entry points
# ----------------------------------------------------------------------------------------------

def _check_inputs(q, k, v, mask, mask_packed=None):
    assert q.shape == k.shape == v.shape, "q/k/v must have the same shape"
    B, H, N, _ = q.shape
    if mask_packed is not None:
        mp = tuple(mask_packed.shape)
        assert mask_packed.dtype == torch.int32 and len(mp) == 4 and mp[0] in (1, B) and mp[1] in (1, H) \
            and mp[2:] == (N, (N + 31) // 32), \
            "mask_packed must be the int32 [B or 1, H or 1, N, ceil(N/32)] result of pack_mask"
        assert mask_packed.device == q.device, "all tensors must be on the same device"
        return
    assert q.device == k.device == v.device == mask.device, "all tensors must be on the same device"
    assert mask.dtype == torch.bool, "mask must be a bool tensor"
    ms = tuple(mask.shape)
    assert len(ms) == 4 and ms[0] in (1, B) and ms[1] in (1, H) and ms[2:] == (N, N), \
        "mask must be [B or 1, H or 1, N, N]"


def _unexpand(mask: torch.Tensor) -> torch.Tensor:
    """The mask with its expanded (stride 0) batch / head extents taken back to 1: a mask given as
    ``m.expand(B, H, N, N)`` is read (or packed) once and shared, not B*H times."""
    if mask.size(0) > 1 and mask.stride(0) == 0:
        mask = mask[:1]
    if mask.size(1) > 1 and mask.stride(1) == 0:
        mask = mask[:, :1]
    return mask



def _declined(q, k, v, mask, mask_packed, tile_map, autograd):
    """What ``sparse_attn_cuda.attention`` did not take: the checks that say what is wrong with the
    arguments, and the one thing it leaves to be done beforehand, packing a mask of fewer than 16 columns
    (shorter than one copy of the kernel that reads the boolean mask)."""
    if torch.jit.is_tracing():
        return _TracedCall.apply(sparse_attention if autograd else sparse_attention_func, q, k, v, mask, mask_packed, tile_map)
    _check_inputs(q, k, v, mask, mask_packed)
    if autograd:
        assert tile_map is None or tile_map is True or mask_packed is not None, "a tile_map tensor belongs to a mask_packed"
        assert not (tile_map is True and mask_packed is not None), "with mask_packed, pass the result of tile_map(mask_packed)"
    else:
        assert tile_map is None or tile_map is True or mask_packed is not None, "tile_map belongs to a mask_packed"
    _require_ext(q)
    assert 1 <= q.shape[-1] <= 128, "head_dim must be at most 128"
    if mask_packed is None and q.shape[2] < 16:
        mask_packed = pack_mask(_unexpand(mask))
        if tile_map is True:
            tile_map = sparse_attn_cuda.tile_map(mask_packed) if autograd else None
    out = sparse_attn_cuda.attention(q, k, v, None, mask_packed, tile_map, autograd) if mask_packed is not None else None
    if out is None:
        raise RuntimeError("Unsupported dtype, need BF16 or FP16 (or FP32), the same for q, k and v, on one device")
    return out


def sparse_attention(q, k, v, mask, mask_packed=None, tile_map=None):
    """Masked attention with autograd support.

    q, k, v: ``[B, H, N, D]`` (D <= 128; off multiples of 8 at the price of padding copies) bf16 / fp16 / fp32;
    mask: bool ``[B, H, N, N]``, True = keep (a leading extent of 1 shares the mask between batch entries / heads).
    Returns a tensor of q's shape and original dtype.

    ``mask_packed`` (optional, not in the reference): the result of ``pack_mask(mask)`` kept from an
    earlier call with the same mask; packing (as much HBM traffic as the attention itself at
    N = 512) is then skipped and ``mask`` may be None.  ``tile_map`` (optional): with ``mask_packed``,
    the result of ``tile_map(mask_packed)``; key tiles in which the mask keeps nothing are skipped.
    With a bool ``mask`` under autograd, ``tile_map=True`` says that the mask has empty 64 x 64 blocks:
    the forward then leaves the map behind for the backward (about 1 us at N = 512; off by default,
    because a mask without empty blocks gains nothing from it).
    """
    out = sparse_attn_cuda.attention(q, k, v, mask, mask_packed, tile_map, True) if HAS_CUDA_EXT else None
    return out if out is not None else _declined(q, k, v, mask, mask_packed, tile_map, True)


def sparse_attention_func(q, k, v, mask, mask_packed=None, tile_map=None):
    """Inference-only variant of :func:`sparse_attention`: no autograd graph, no LSE."""
    out = sparse_attn_cuda.attention(q, k, v, mask, mask_packed, tile_map, False) if HAS_CUDA_EXT else None
    return out if out is not None else _declined(q, k, v, mask, mask_packed, tile_map, False)


# ----------------------------------------------------------------------------------------------
# mask helpers
# ----------------------------------------------------------------------------------------------

def pack_mask(mask: torch.Tensor) -> torch.Tensor:
    """bool ``[B, H, N, N]`` -> bit-packed int32 ``[B, H, N, ceil(N/32)]`` (bit j of word w = column 32w+j).
    A mask shared between batch entries / heads is passed (and packed) as ``[1 or B, 1 or H, N, N]``."""
    _require_ext(mask)
    return sparse_attn_cuda.pack_mask(mask)


def tile_map(mask_packed: torch.Tensor, min_skip: float = 0.3):
    """Occupancy of the 64 x 64 blocks of a packed mask, for ``sparse_attention(..., mask_packed=,
    tile_map=)``: int32 ``[B, H, T, 2, ceil(T/32)]`` with T = ceil(N/64); per block of 64 query rows
    one bit per 64-key tile "some entry kept", then one bit per tile "every entry kept".

    Returns None when the map would not pay: the forward walks the key tiles per 128 query rows (two
    row blocks), and below ``min_skip`` (default 0.3) of those visits saved the walk costs what
    it saves (a causal mask at N = 256 skips 2 of 8 visits per head and runs no faster with the
    map).  ``min_skip=0`` returns the map whenever a single visit disappears.  Synchronises with the
    device once, to look at that; meant to be called once for a mask that is used many times."""
    _require_ext(mask_packed)
    tm = sparse_attn_cuda.tile_map(mask_packed)
    T = tm.shape[2]
    live = tm[:, :, :, 0, :]
    if T % 2:                                   # the last work-group has one row block only
        live = torch.cat([live, torch.zeros_like(live[:, :, :1])], dim=2)
    pairs = live[:, :, 0::2] | live[:, :, 1::2]             # what a work-group of 128 rows visits
    bits = (pairs.unsqueeze(-1) >> torch.arange(32, device=tm.device, dtype=torch.int32)) & 1
    visited = int(bits.sum().item())
    total = pairs.shape[0] * pairs.shape[1] * pairs.shape[2] * T
    skipped = total - visited
    return tm if skipped > 0 and skipped >= min_skip * total else None


def generate_random_sparse_mask(B, H, N, sparsity=0.75, device="cuda"):
    """Random mask whose entries are False (masked out) with probability ``sparsity``."""
    return torch.rand(B, H, N, N, device=device) > sparsity
