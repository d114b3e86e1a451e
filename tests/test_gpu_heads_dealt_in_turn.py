"""Grids of more than one round whose heads share a mask deal the tiles of several heads out in turn; those with the same mask given
for every head take one head after the other.  Every tile is computed once and by itself, so the results are the same to the bit."""
import importlib
import sys

import pytest
import torch

from _launches import launches, places

pytestmark = pytest.mark.gpu


# heads beyond one round of every kernel, in groups (in the forward at head dims up to 64, at 128) of: 4, 2 of a share of 4; 3, 1 of 3; 5 of 5, a prime; 3, 2 of
# 6; 12, 6 of 12, one head with all the masks shared by the batch; 24, 12 of 24 short ones; and one after the other (no multiple of 8)
@pytest.mark.parametrize("B, H, N", [(2, 16, 3300), (3, 8, 4200), (5, 8, 2600), (4, 12, 4097), (96, 1, 1153), (16, 12, 577), (7, 3, 4750)])
@pytest.mark.parametrize("D", [32, 64, 72, 128])
@pytest.mark.parametrize("mapped", [False, True])
def test_same_bits_as_with_a_mask_for_every_head(dev, B, H, N, D, mapped):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v, do = (torch.randn(B, H, N, D, generator=g, device=dev, dtype=torch.bfloat16) for _ in range(4))
    mask = torch.rand(1, 1, N, N, generator=g, device=dev) < 0.3
    mask &= torch.ones(N, N, dtype=torch.bool, device=dev).tril()
    mask[:, :, 200:300] = False                                  # rows that keep nothing, and a block of them
    shared = sa.pack_mask(mask)
    each = shared.expand(B, H, -1, -1).contiguous()
    results = []
    for packed in (shared, each):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        tile_map = sa.sparse_attn_cuda.tile_map(packed) if mapped else None
        out = sa.sparse_attention(*leaves, None, mask_packed=packed, tile_map=tile_map)
        results.append([out.detach(), *torch.autograd.grad(out, leaves, do)])
    for a, b, name in zip(*results, ("out", "dq", "dk", "dv")):
        assert torch.equal(a, b), name
    # ... and not left over from another call: a head that no group begins with, against the same head by itself
    h = B * H - 2
    pick = lambda t: t[h // H:h // H + 1, h % H:h % H + 1]
    s = torch.matmul(pick(q).float(), pick(k).float().transpose(-1, -2).contiguous()) * D ** -0.5
    p = torch.softmax(s.masked_fill(~mask, float("-inf")), -1).nan_to_num(0.0)
    ref = torch.matmul(p, pick(v).float())
    # q, probabilities and the result are rounded to bf16, by 2**-9 of themselves each: a score moves by at most e, a weight by 2 e of itself
    e = 2 ** -9 * float(torch.matmul(pick(q).float().abs(), pick(k).float().abs().transpose(-1, -2).contiguous()).max()) * D ** -0.5
    assert (pick(results[0][0]).float() - ref).abs().max() <= (2 * e + 2 * 2 ** -9) * pick(v).float().abs().max()


# A mask for every batch entry: groups of several entries (the mask's words change inside a group), of parts of one, and of shares without a divisor near what
# an XCD holds at once; 72 heads at head dim 128: the last eight of the dK/dV kernel's come in work-groups of half the keys, after the dealt ones.
@pytest.mark.parametrize("B, H, N, D", [(64, 2, 1153, 64), (64, 2, 1153, 128), (40, 4, 1000, 32), (16, 12, 577, 96), (29, 8, 1153, 64), (13, 8, 1024, 128),
                                        (9, 8, 2048, 128)])
@pytest.mark.parametrize("mapped", [False, True])
def test_masks_of_batch_entries(dev, B, H, N, D, mapped):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v, do = (torch.randn(B, H, N, D, generator=g, device=dev, dtype=torch.bfloat16) for _ in range(4))
    mask = torch.rand(B, 1, N, N, generator=g, device=dev) < 0.3
    mask[::3] &= torch.ones(N, N, dtype=torch.bool, device=dev).tril()
    mask[1::3, :, 200:300] = False                               # rows that keep nothing
    mask[1::3, :, :, 128:256] = False                            # keys that nobody keeps
    shared = sa.pack_mask(mask)
    results, ran = [], []
    for packed in (shared, shared.expand(B, H, -1, -1).contiguous()):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        tile_map = sa.sparse_attn_cuda.tile_map(packed) if mapped else None
        out = sa.sparse_attention(*leaves, None, mask_packed=packed, tile_map=tile_map)
        grads = []
        ran.append(launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do))))
        results.append([out.detach(), *grads])
    assert ran[0] == ran[1]
    if (B, H) == (9, 8) and places() == 256:
        assert [n for name, args, n in ran[0] if name == "attn_bwd_dkv_kernel" and args[1:3] == ("128", "8")] == [64 * 8 + 8 * 16]
    for a, b, name in zip(*results, ("out", "dq", "dk", "dv")):
        assert torch.equal(a, b), name
