"""The backward whose dQ and dK/dV work-groups share a launch (grids of one round; with a tile map any grid at head dim 64)."""
import importlib
import sys

import pytest
import torch

from _launches import launches
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


def _sa():
    importlib.import_module("python.sparse_attention")
    return sys.modules["python.sparse_attention"]


# Bound: probabilities and dS are rounded to 16 bits before the second product, half a unit in the last place of each factor,
# as in the other backward tests.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [24, 64, 80, 128])
@pytest.mark.parametrize("N", [513, 575, 641, 768, 1000])              # first and last row of a tile, whole ones, whole work-groups
def test_one_round_against_the_oracle(dev, N, D, dtype):
    sa = _sa()
    g = torch.Generator().manual_seed(N + D)
    q, k, v, do = (torch.randn(2, N, 3, D, generator=g).to(dtype).to(dev).transpose(1, 2) for _ in range(4))
    mask = torch.rand(2, 1, N, N, generator=g) < 0.3
    mask[:, :, N // 2] = False                                        # a row that keeps nothing
    mask[:, :, :, N // 3] = False                                     # a key that nobody keeps
    mask[0, :, :, 192:320] = False                                    # a work-group's keys without any
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*leaves, mask.to(dev))
    grads = []
    kernels = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do, retain_graph=True)))]
    assert kernels[-2:] == ["attn_bwd_delta_kernel", "attn_bwd_both_kernel"], kernels
    assert all(torch.equal(x, y) for x, y in zip(grads, torch.autograd.grad(out, leaves, do)))
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for b, h in ((0, 0), (1, 2)):
        one = [t[b:b + 1, h:h + 1].float().cpu() for t in (q, k, v, do)]
        refs = O.sparse_attention_bwd_ref(*one[:3], mask[b:b + 1], one[3], scale=D ** -0.5)
        for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
            err = (got[b:b + 1, h:h + 1].float().cpu() - ref).abs()
            assert (err <= 1e-4 + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, b, h, float(err.max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D, heads, N", [(64, 120, 1000), (64, 190, 600), (96, 70, 640), (72, 90, 513)])      # more than a round
def test_same_bits_with_a_tile_map(dev, D, heads, N, dtype):
    """With the map in one launch, without in two: delta, and with it every gradient, has the same bits."""
    sa = _sa()
    g = torch.Generator(device=dev).manual_seed(N)
    nb = (N + 63) // 64
    blocks = (torch.rand(1, heads, nb, nb, device=dev, generator=g) < 0.25) | torch.eye(nb, dtype=torch.bool, device=dev)
    mask = blocks.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N].contiguous()
    q, k, v, do = (torch.randn(1, heads, N, D, device=dev, generator=g).to(dtype) for _ in range(4))
    packed = sa.pack_mask(mask)
    tile_map = sa.tile_map(packed, min_skip=0.0)
    assert tile_map is not None
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    ways = []
    for given, one in ((tile_map, D == 64), (None, False)):
        out = sa.sparse_attention(*leaves, None, mask_packed=packed, tile_map=given)
        ran = launches(lambda: ways.append(torch.autograd.grad(out, leaves, do)))
        assert any(name == "attn_bwd_both_kernel" for name, _, _ in ran) == one, ran
    with_map, without = ways
    assert all(torch.equal(x, y) for x, y in zip(with_map, without))
