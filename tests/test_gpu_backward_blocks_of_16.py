"""The dQ and dK/dV kernels form 16 x 16 blocks: lengths whose last block of 16 or 32 rows and keys holds one, all but one or all of them, head dims
up to, at and between the kernels' own, in one launch and in two, with and without the post-multiplier and a tile map."""
import importlib
import sys

import pytest
import torch

from _launches import launches
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


# Bound: probabilities and dS are rounded to 16 bits before the second product: half a unit in the last place of each factor, 1e-2 (fp16, bf16's
# operands 2e-2) of the entry and of the largest one, as in the other backward tests.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [8, 32, 48, 64, 80, 96, 104, 128])
@pytest.mark.parametrize("N", [513, 527, 528, 529, 560, 575, 576, 593])
@pytest.mark.parametrize("heads", [3, 160])
def test_against_the_oracle(dev, N, D, dtype, heads):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator().manual_seed(1000 * N + D)
    # rows of the projections' layout, inside larger buffers of NaN: nothing beyond a row takes part
    q, k, v, do = (torch.full((1, N, heads, D + 8), float("nan"), dtype=dtype).to(dev)[..., :D].transpose(1, 2) for _ in range(4))
    for t in (q, k, v, do):
        t.copy_(torch.randn(1, heads, N, D, generator=g))
    mask = torch.rand(1, 1, N, N, generator=g) < 0.3
    mask[:, :, N - 1] = False                                    # the last row keeps nothing
    mask[:, :, :, N // 3] = False                                # a key that nobody keeps
    mask[:, :, 32:48, 64:80] = False                             # a block without any, and one of 32 x 32
    mask[:, :, 96:128, 32:64] = False
    mask[:, :, 17] = True
    packed = sa.pack_mask(mask.to(dev))
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*leaves, None, mask_packed=packed)
    grads = []
    ran = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do)))]
    assert ran == (["attn_bwd_delta_kernel", "attn_bwd_both_kernel"] if heads == 3 else ["attn_bwd_dq_kernel", "attn_bwd_dkv_kernel"])
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].detach().float().cpu() for t in (q, k, v, do)]
        refs = O.sparse_attention_bwd_ref(*one[:3], mask, one[3], scale=D ** -0.5)
        for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
            err = (got[:, h:h + 1].float().cpu() - ref).abs()
            assert (err <= 1e-4 + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, h, float(err.max()))


# Scores formed with the post-multiplier (|scale| log2 e > 1; q is smaller by as much, so the scores have the others' size), with and without a tile map, which at
# head dim 64 brings dQ and dK/dV into one launch.  Bound: as above; dQ and dK carry the scale.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("N", [513, 575, 641])
@pytest.mark.parametrize("heads", [3, 160])
@pytest.mark.parametrize("scale, mapped", [(None, True), (-2.5, False), (-2.5, True)])
def test_scales_and_maps_against_the_oracle(dev, N, D, dtype, heads, scale, mapped):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(1000 * N + D + 1)
    q, k, v, do = (torch.randn(1, heads, N, D, generator=g, device=dev) for _ in range(4))
    if scale is not None:
        q *= 2.0 ** -4
    mask = torch.rand(1, 1, N, N, generator=g, device=dev) < 0.3
    mask &= torch.ones(N, N, dtype=torch.bool, device=dev).tril(192)          # tiles without any at the rows' ends
    mask[:, :, 130:260, 64:128] = False                          # ... and in the midst of some rows, at an odd place
    mask[:, :, N - 1] = False
    mask[:, :, :, N // 3] = False
    packed = sa.pack_mask(mask)
    tile_map = sa.tile_map(packed, min_skip=0.0) if mapped else None
    leaves = [t.to(dtype).requires_grad_(True) for t in (q, k, v)]
    do = do.to(dtype)
    out = sa.SparseAttentionFunction.apply(*leaves, packed, None, scale or D ** -0.5, N, tile_map)
    grads = []
    ran = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do)))]
    ran = [name for name in ran if name != "to_bf16_kernel"]
    one_launch = heads == 3 or (mapped and D == 64)
    assert ran == (["attn_bwd_delta_kernel", "attn_bwd_both_kernel"] if one_launch else ["attn_bwd_dq_kernel", "attn_bwd_dkv_kernel"])
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    floor = 1e-4 * max(1.0, abs(scale or 0.0))
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].detach().float().cpu() for t in (*leaves, do)]
        refs = O.sparse_attention_bwd_ref(*one[:3], mask.cpu(), one[3], scale=scale or D ** -0.5)
        for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
            err = (got[:, h:h + 1].float().cpu() - ref).abs()
            assert (err <= floor + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, h, float(err.max()))
