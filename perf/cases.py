"""The work that users of sparse-mask attention have it do, as cases that can be timed.

A case is a dict of plain values:

  op      "infer"         sparse_attention_func(q, k, v, mask): the boolean mask in, the output out
          "infer_packed"  the same with the mask packed beforehand (``mask_packed=``, ``tile_map=``), as the
                          layers of a model do that all use one mask
          "train"         sparse_attention(q, k, v, mask) and the gradients of q, k and v
          "train_packed"  the same with the mask packed beforehand
          "pack"          pack_mask(mask)
  B, H, N, D, dtype       extents and element type of q, k, v (fp32 is computed in bf16 by the framework)
  layout  "bhnd"          contiguous [B, H, N, D] tensors
          "bnhd"          [B, N, H, D] projection outputs, viewed as [B, H, N, D]
  mask, keep              structure of the mask and the share of entries kept (see make_mask)
  share   "none"          a mask of its own for every head, [B, H, N, N]
          "heads"         one for all heads of a batch entry, [B, 1, N, N]
          "all"           one for everything, [1, 1, N, N]
"""
import importlib
import math
import os
import sys

import torch

# the repository's root is the working folder
_PKG = os.path.abspath("sparse-mask-attention_amd")
if _PKG not in sys.path:
    sys.path.append(_PKG)
importlib.import_module("python.sparse_attention")
sa = sys.modules["python.sparse_attention"]

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, op, B, H, N, D=64, dtype="fp16", layout="bhnd", mask="random", keep=0.25, share="none"):
    c = dict(op=op, B=B, H=H, N=N, D=D, dtype=dtype, layout=layout, mask=mask, keep=keep, share=share)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short request of a small model: nothing but the latency of a call
        _case("infer_tiny", "infer", 1, 2, 128),
        # the headline configuration of the benchmark: a batch of sequences, a random mask used once
        _case("infer_headline", "infer", 16, 12, 512),
        # a length that is no multiple of any tile, bf16, very sparse, every token sees itself
        _case("infer_ragged", "infer", 8, 16, 1000, dtype="bf16", mask="random_diag", keep=0.10),
        # a block-sparse mask that all layers share: packed once, its empty blocks skipped
        _case("infer_blocks", "infer_packed", 16, 12, 1024, mask="block64"),
        # prefill of long prompts, head dim 128, from the projections' own layout, one causal mask for all heads
        _case("infer_long", "infer", 4, 32, 4096, D=128, dtype="bf16", layout="bnhd", mask="causal", keep=1.0, share="all"),
        # the packer by itself, as a program calls it once per mask
        _case("pack", "pack", 16, 12, 1024, mask="block64"),
        # one step of a small model on a few odd-length sequences: host work and launches
        _case("train_tiny", "train", 2, 4, 333, D=32, dtype="bf16", mask="random_diag", keep=0.3),
        # forward and backward of the headline configuration
        _case("train_headline", "train", 16, 12, 512),
        # many short causal sequences
        _case("train_short", "train", 64, 16, 256, mask="causal", keep=0.5),
        # training with a block-sparse mask that all layers share
        _case("train_blocks", "train_packed", 16, 12, 1024, mask="block64"),
        # a model kept in fp32 with a head dim between the kernels' own, from the projections' layout
        _case("train_fp32", "train", 8, 12, 577, D=80, dtype="fp32", layout="bnhd", mask="random_diag", keep=0.25, share="heads"),
        # the largest: long sequences, head dim 128, one random mask for all heads of a sequence
        _case("train_long", "train", 4, 32, 4096, D=128, dtype="bf16", mask="random", keep=0.5, share="heads"),
    ]


# 4, 10 for forward and backward: the products of N x N x D per head, two operations each
_FLOPS = {"infer": 4, "infer_packed": 4, "train": 14, "train_packed": 14, "pack": 0}
_MOST_FLOPS = 14 * 4 * 32 * 4096 ** 2 * 128
_MOST_MASK = 200 * 1024 ** 2          # entries of a boolean mask, as many as the pack case has


def draw(rng):
    op = rng.choice(["infer", "infer", "infer", "infer_packed", "train", "train", "train", "train_packed", "pack"])
    N = int(round(math.exp(rng.uniform(math.log(16), math.log(4096)))))
    if rng.random() < 0.4:                       # lengths padded to a multiple of 64 are as common as any others
        N = max(64, N // 64 * 64)
    D = rng.choice([64, 64, 64, 64, 128, 128, 32, 80, 96])
    dtype = rng.choice(["fp16", "fp16", "bf16", "bf16", "fp32"])
    mask, keep = rng.choice([("random", 0.25), ("random", 0.5), ("random_diag", 0.1), ("block64", 0.25), ("causal", 0.5), ("causal", 1.0)])
    share = rng.choice(["none", "none", "heads", "all"])
    layout = rng.choice(["bhnd", "bnhd"])
    H = rng.choice([1, 2, 4, 8, 12, 16, 32])
    B = int(round(math.exp(rng.uniform(0.0, math.log(64)))))

    def too_large(B, H):
        Bm, Hm = _mask_extents(share, B, H)
        kernel_D = 32 if D <= 32 else (64 if D <= 64 else 128)
        heavy = 2 if dtype == "fp32" or D != kernel_D else 1          # conversions and padding cost passes of their own
        return Bm * Hm * N * N > _MOST_MASK or heavy * _FLOPS[op] * B * H * N * N * kernel_D > _MOST_FLOPS

    while too_large(B, H) and B > 1:
        B = (B + 1) // 2
    while too_large(B, H) and H > 1:
        H //= 2
    if op == "pack":                             # nothing but the mask takes part
        Bm, Hm = _mask_extents(share, B, H)
        return _case(None, op, Bm, Hm, N, mask=mask, keep=keep)
    return _case(None, op, B, H, N, D, dtype, layout, mask, keep, share)


def _mask_extents(share, B, H):
    return {"none": (B, H), "heads": (B, 1), "all": (1, 1)}[share]


def make_mask(kind, keep, B, H, N, g):
    """bool [B, H, N, N] on the GPU.
    random       every entry kept with probability keep
    random_diag  the same, and every token sees itself
    block64      64 x 64 blocks kept with probability keep, those on the diagonal always
    causal       no token sees a later one, entries before kept with probability keep, itself always"""
    if kind == "block64":
        nb = (N + 63) // 64
        blocks = torch.rand(B, H, nb, nb, device="cuda", generator=g) < keep
        blocks |= torch.eye(nb, dtype=torch.bool, device="cuda")
        return blocks.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[:, :, :, :N].contiguous()
    if keep >= 1.0:
        m = torch.ones(B, H, N, N, dtype=torch.bool, device="cuda")
    else:
        m = torch.rand(B, H, N, N, device="cuda", generator=g) < keep
    if kind == "causal":
        m &= torch.ones(N, N, dtype=torch.bool, device="cuda").tril_()
    if kind in ("causal", "random_diag"):
        m |= torch.eye(N, dtype=torch.bool, device="cuda")
    return m


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, B, H, N, D = case["op"], case["B"], case["H"], case["N"], case["D"]
    s = {"op": op}
    mask = make_mask(case["mask"], case["keep"], *_mask_extents(case["share"], B, H), N, g)
    if op == "pack":
        return dict(s, mask=mask)

    def rows():
        shape = (B, H, N, D) if case["layout"] == "bhnd" else (B, N, H, D)
        t = torch.randn(shape, device="cuda", generator=g).to(DTYPES[case["dtype"]])
        return t if case["layout"] == "bhnd" else t.transpose(1, 2)

    s["q"], s["k"], s["v"] = rows(), rows(), rows()
    if op.startswith("train"):
        for name in "qkv":
            s[name].requires_grad_(True)
        s["dout"] = rows()
    if op.endswith("_packed"):
        s["mask"], s["mask_packed"] = None, sa.pack_mask(mask)
        s["tile_map"] = sa.tile_map(s["mask_packed"])
    else:
        s["mask"], s["mask_packed"], s["tile_map"] = mask, None, None
    return s


def run(s):
    if s["op"] == "pack":
        return sa.pack_mask(s["mask"])
    if s["op"].startswith("infer"):
        return sa.sparse_attention_func(s["q"], s["k"], s["v"], s["mask"], mask_packed=s["mask_packed"], tile_map=s["tile_map"])
    out = sa.sparse_attention(s["q"], s["k"], s["v"], s["mask"], mask_packed=s["mask_packed"], tile_map=s["tile_map"])
    dq, dk, dv = torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}


def work(case):
    """q, k, v, the mask and the output gradient read once, the output and the gradients written once; the products
    over the 64 x 64 blocks of the scores in which the mask keeps something."""
    op, B, H, N, D = case["op"], case["B"], case["H"], case["N"], case["D"]
    Bm, Hm = _mask_extents(case["share"], B, H)
    words = 4 * Bm * Hm * N * ((N + 31) // 32)
    if op == "pack":
        return {"bytes": Bm * Hm * N * N + words, "flops": 0}
    nb = (N + 63) // 64
    live = 1.0
    if case["mask"] == "block64":
        live = (1 + case["keep"] * (nb - 1)) / nb
    elif case["mask"] == "causal":
        live = (nb + 1) / (2 * nb)
    matrices = 8 if op.startswith("train") else 4
    size = 4 if case["dtype"] == "fp32" else 2
    mask_bytes = words if op.endswith("_packed") else Bm * Hm * N * N
    return {"bytes": matrices * B * H * N * D * size + mask_bytes, "flops": live * _FLOPS[op] * B * H * N * N * D}


def tolerance(case):
    """Bits for the packer; else what the 16-bit operands, weights and score gradients leave (fp32 tensors are computed
    in bf16)."""
    if case["op"] == "pack":
        return "exact"
    return {"rel": 3e-3 if case["dtype"] == "fp16" else 1e-2}
