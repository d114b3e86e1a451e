"""The forward whose work-groups have 64 rows and whose wavefronts share the keys of every tile (head dims beyond 64, grids of at most one such
work-group on a CU; the others further down)."""
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


# first and last row and key of a tile and of half a tile, whole tiles, a walk over two words of the tile map
SIZES = [(50, 129), (50, 160), (64, 192), (50, 193), (40, 256), (22, 513), (14, 1025), (5, 3000)]


# Bound: the probabilities (fp16 rounded towards zero, bf16 to nearest) and the result are rounded once each, relative to the largest value of
# a row's weighted mean; 4 units in the last place of 16-bit elements leave room for the exponentials.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [72, 128])
@pytest.mark.parametrize("heads, N", SIZES)
@pytest.mark.parametrize("scale", [None, 1.5])                        # ordinary rows, and rows that one key decides
def test_halves_against_the_oracle(dev, heads, N, D, dtype, scale):
    sa = _sa()
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v = (torch.randn(1, N, heads, D, device=dev, generator=g).to(dtype).transpose(1, 2) for _ in range(3))
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    keys = torch.arange(N, device=dev)
    mask[..., 3, :] = False                                            # a row that keeps nothing,
    mask[..., 4, :] &= keys % 64 < 32                                  # one half of every tile,
    mask[..., 5, :] &= keys % 64 >= 32                                 # the other,
    mask[..., 6, :] = keys == N - 1                                    # the last key alone
    mask[..., 64:96, :64] = False                                      # nothing in a tile for one wavefront's rows
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    scale = D ** -0.5 if scale is None else scale
    packed = sa.pack_mask(mask)
    tile_map = sa.tile_map(packed, min_skip=0.0)
    made = []
    ran = launches(lambda: made.extend([sa.SparseAttentionFunction.apply(*leaves, None, mask, scale, N),
                                        sa.SparseAttentionFunction.apply(*leaves, packed, None, scale, N),
                                        sa.SparseAttentionFunction.apply(*leaves, packed, None, scale, N, tile_map)]))
    assert [args[9] for name, args, _ in ran if name == "attn_fwd_kernel"] == ["true"] * 3, ran           # HALVES
    out, again, mapped = made
    assert torch.equal(out, again) and torch.equal(out, mapped)
    lse, words = out.grad_fn.saved_tensors[4:6]
    assert torch.equal(lse, again.grad_fn.saved_tensors[4]) and torch.equal(words.view_as(packed), packed)      # by-products
    eps = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].detach().float().cpu() for t in (q, k, v)]
        if dtype == torch.float32:
            one = [t.bfloat16().float() for t in one]
        # the kernel rounds the scaled q to 16 bits: so does the reference
        x = (one[0] * scale).double() @ one[1].double().transpose(-1, -2)
        x = x.masked_fill(~mask.cpu(), float("-inf"))
        want_lse = torch.logsumexp(x, -1)
        ref = O.sparse_attention_ref(*one, mask.cpu(), scale=scale)
        assert torch.isinf(lse[:, h, 3]).all() and (out[:, h, 3] == 0).all()
        # a score of n terms whose factor q is rounded once moves by at most eps / 2 of the sum of their magnitudes
        shift = eps * (one[0].abs() * abs(scale)) @ one[1].abs().transpose(-1, -2)
        shift = shift.masked_fill(~mask.cpu(), 0).amax(-1)
        live = torch.isfinite(want_lse)
        assert ((lse[:, h:h + 1].cpu().double() - want_lse).abs() <= 1e-4 + shift)[live].all()
        err = (out[:, h:h + 1].detach().float().cpu() - ref).abs()
        top = one[2].abs().max()
        assert (err <= 1e-4 + top * (4 * eps + 2 * shift[..., None])).all(), (h, float(err.max()))


@pytest.mark.parametrize("heads, N", SIZES)
def test_map_by_product(dev, heads, N):
    """The tile map left behind is the one made from the packed mask: the gradients with it are those without."""
    sa = _sa()
    g = torch.Generator(device=dev).manual_seed(N)
    nb = (N + 63) // 64
    blocks = (torch.rand(1, heads, nb, nb, device=dev, generator=g) < 0.3) | torch.eye(nb, dtype=torch.bool, device=dev)
    mask = blocks.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N].contiguous()
    mask[:, :, 40:50] = False
    q, k, v, do = (torch.randn(1, heads, N, 128, device=dev, generator=g).half() for _ in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    outs = []
    ran = launches(lambda: outs.append(sa.sparse_attention(*leaves, mask, tile_map=True)))
    assert [args[9] for name, args, _ in ran if name == "attn_fwd_kernel"] == ["true"], ran
    out = outs[0]
    made = out.grad_fn.tile_map
    assert torch.equal(made.flatten(), sa.tile_map(sa.pack_mask(mask), min_skip=0.0).flatten())
    plain = sa.sparse_attention(*leaves, mask)
    assert torch.equal(out, plain)
    assert all(torch.equal(x, y) for x, y in zip(torch.autograd.grad(out, leaves, do), torch.autograd.grad(plain, leaves, do)))


# Head dims up to 64 (three work-groups share a CU): one round of more than two of 64 rows on each, beyond ten tiles; and head dim 96 from 1024 rows on, up
# to two.  Pairs of tiles that end in either of their tiles, whole ones (N a multiple of 128), one key beyond a tile and one short of it, a walk over two map
# words.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, N, D", [(50, 641, 64), (48, 704, 32), (44, 705, 64), (60, 767, 40), (50, 768, 32), (33, 1023, 64), (33, 1024, 64), (36, 1025, 48),
                                         (17, 2100, 64), (30, 1025, 80), (10, 2048, 96)])
def test_one_round_of_64_row_groups(dev, heads, N, D, dtype):
    sa = _sa()
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v = (torch.randn(1, heads, N, D, device=dev, generator=g).to(dtype) for _ in range(3))
    nb = (N + 63) // 64
    blocks = torch.rand(1, 1, nb, nb, device=dev, generator=g) < 0.6
    mask = (torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3) & blocks.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N]
    mask[..., 3, :] = False
    mask[..., 4, :] = torch.arange(N, device=dev) == N - 1
    odd = (mask.to(torch.uint8) * 6).view(torch.bool)                  # bytes that are neither 0 nor 1
    packed = sa.pack_mask(mask)
    tile_map = sa.tile_map(packed, min_skip=0.0)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    made = []
    ran = launches(lambda: made.extend([sa.sparse_attention_func(q, k, v, mask), sa.sparse_attention_func(q, k, v, odd),
                                        sa.sparse_attention_func(q, k, v, None, mask_packed=packed),
                                        sa.sparse_attention_func(q, k, v, None, mask_packed=packed, tile_map=tile_map),
                                        sa.sparse_attention(*leaves, mask, tile_map=True)]))
    assert [args[9] for name, args, _ in ran if name == "attn_fwd_kernel"] == ["true"] * 5, ran           # HALVES
    out = made[0]
    assert all(torch.equal(out, x) for x in made[1:])
    lse, words = made[4].grad_fn.saved_tensors[4:6]
    assert torch.equal(words.view_as(packed), packed) and torch.equal(made[4].grad_fn.tile_map.flatten(), tile_map.flatten())
    # the bounds of the first test
    eps = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].double() if dtype != torch.float32 else t[:, h:h + 1].bfloat16().double() for t in (q, k, v)]
        x = ((one[0] * D ** -0.5) @ one[1].transpose(-1, -2)).masked_fill(~mask, float("-inf"))
        ref, want_lse = torch.softmax(x, -1).nan_to_num() @ one[2], torch.logsumexp(x, -1)
        shift = (eps * (one[0].abs() * D ** -0.5) @ one[1].abs().transpose(-1, -2)).masked_fill(~mask, 0).amax(-1)
        err = (out[:, h:h + 1].double() - ref).abs()
        assert (err <= 1e-4 + one[2].abs().max() * (4 * eps + 2 * shift[..., None])).all(), float(err.max())
        assert ((lse[:, h:h + 1].double() - want_lse).abs() <= 1e-4 + shift)[torch.isfinite(want_lse)].all() and torch.isinf(lse[:, h, 3]).all()
