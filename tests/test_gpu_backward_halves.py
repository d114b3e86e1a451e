"""dK/dV at head dim 128 by work-groups of 128 keys whose wavefronts share the rows: whole grids of them, and the last heads of larger ones."""
import importlib
import sys

import pytest
import torch

from _launches import launches, places
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


def _dkv_groups(fn):
    """Work-groups of the dK/dV kernel of eight wavefronts that fn launches."""
    ran = launches(fn)
    groups = [n for name, args, n in ran if name == "attn_bwd_dkv_kernel" and args[1:3] == ("128", "8")]
    assert len(groups) == 1, ran
    return groups[0]


def _expected(heads, N):
    """All in work-groups of 128 keys where these fill one round at most, else the heads beyond the last full round."""
    narrow, wide = (N + 127) // 128, (N + 255) // 256
    if heads * narrow <= places():
        return heads * narrow
    whole = (heads * wide - 1) // places() * places() // wide
    assert 0 < whole < heads and (heads - whole) * narrow <= places()
    return whole * wide + (heads - whole) * narrow


# Bound: probabilities and dS are rounded to 16 bits before the second product, as in the other backward tests.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, N", [(30, 641), (25, 1153), (6, 3000), (87, 641), (70, 897), (66, 1024), (65, 993)])
def test_halves_against_the_oracle(dev, heads, N, dtype):
    """Grids of one round, first and last row of a tile; a second round of one head and of several."""
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + heads)
    q, k, v, do = (torch.randn(1, N, heads, 128, device=dev, generator=g).to(dtype).transpose(1, 2) for _ in range(4))
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    mask[..., N // 2, :] = False                                       # a row that keeps nothing
    mask[..., 128:320, 64:96] = False                                  # rows of one half alone
    mask[..., 128:320, 96:256] &= (torch.arange(128, 320, device=dev) % 64 < 32)[:, None]
    mask[..., N - 1] = False
    mask[..., N - 1, N - 1] = True                                     # the last key is kept by the last row alone
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    packed = sa.pack_mask(mask)
    out = sa.sparse_attention(*leaves, None, mask_packed=packed)
    grads = []
    assert _dkv_groups(lambda: grads.extend(torch.autograd.grad(out, leaves, do, retain_graph=True))) == _expected(heads, N)
    assert all(torch.equal(x, y) for x, y in zip(grads, torch.autograd.grad(out, leaves, do)))
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].float().cpu() for t in (q, k, v, do)]
        refs = O.sparse_attention_bwd_ref(*one[:3], mask.cpu(), one[3], scale=128 ** -0.5)
        for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
            err = (got[:, h:h + 1].float().cpu() - ref).abs()
            assert (err <= 1e-4 + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, h, float(err.max()))


# Map words hold 32 tiles: the last sizes' keys lie in several.  Blocks of 128 keys of which one half of 64 holds nothing, either half; keys
# nobody keeps; rows of whole tiles that keep nothing.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, N", [(30, 641), (25, 1153), (5, 4200), (87, 641), (70, 897), (66, 1024), (16, 4200), (13, 5000)])
@pytest.mark.parametrize("share", [True, False])
def test_same_bits_with_a_tile_map(dev, heads, N, dtype, share):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + heads)
    nb, masks = (N + 63) // 64, 1 if share else heads
    blocks = (torch.rand(1, masks, nb, nb, device=dev, generator=g) < 0.25) | torch.eye(nb, dtype=torch.bool, device=dev)
    blocks[..., 2:4] = False                                           # 128 keys that nobody keeps,
    blocks[..., 5, :] = False                                          # 64 rows that keep nothing
    blocks[..., 6:, 4] = False                                         # the first half of 128 keys kept by few,
    blocks[..., 6:, 7] = False                                         # the second
    mask = blocks.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N].contiguous()
    q, k, v, do = (torch.randn(1, heads, N, 128, device=dev, generator=g).to(dtype) for _ in range(4))
    packed = sa.pack_mask(mask)
    del mask
    tile_map = sa.tile_map(packed, min_skip=0.0)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*leaves, None, mask_packed=packed, tile_map=tile_map)
    with_map = []
    assert _dkv_groups(lambda: with_map.extend(torch.autograd.grad(out, leaves, do))) == _expected(heads, N)
    without = torch.autograd.grad(sa.sparse_attention(*leaves, None, mask_packed=packed), leaves, do)
    assert all(torch.equal(x, y) for x, y in zip(with_map, without))
    assert (with_map[1][:, :, 128:256] == 0).all() and (with_map[2][:, :, 128:256] == 0).all()
