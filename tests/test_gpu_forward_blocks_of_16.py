"""The forward forms 16 x 16 blocks, and a lane works for two rows, 16 apart: one row of a block of 32 whose scores climb from key tile to key tile,
or that meets its first key late, among rows that do neither; by wavefronts of whole work-groups, that split the keys, and that halve the tiles."""
import importlib
import sys

import pytest
import torch

from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


# Bound: probabilities are rounded to 16 bits before the second product, half a unit in the last place: 1e-2 (bf16 2e-2) as in the other tests.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("row", [0, 15, 16, 31])
@pytest.mark.parametrize("D, heads, N", [(32, 2, 333), (64, 2, 257), (64, 200, 321), (32, 300, 130), (96, 16, 209), (128, 10, 333), (128, 160, 257)])
def test_one_row_unlike_the_others(dev, D, heads, N, row, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator().manual_seed(N + D + row)
    q, k, v = (torch.randn(1, heads, N, D, generator=g) for _ in range(3))
    q[..., 0] = 0.0
    q[:, :, row::32, :] = 0.0
    q[:, :, row::32, 0] = 2.0 * D ** 0.5                          # the scores of these rows: twice k's first column, 12 (log2 17) more a tile
    k[..., 0] = 6.0 * torch.arange(N).div(64, rounding_mode="floor")
    mask = torch.rand(1, 1, N, N, generator=g) < 0.3
    mask[:, :, row + 32, :N - 3] = False                          # ... and of the second block, one that meets its first key in the last tile
    mask[:, :, row + 32, N - 3:] = True
    mask[:, :, row + 64] = False                                  # of the third, one that keeps nothing
    q, k, v = (t.to(dtype).to(dev) for t in (q, k, v))
    out = sa.sparse_attention_func(q, k, v, mask.to(dev))
    packed = sa.pack_mask(mask.to(dev))
    assert torch.equal(out, sa.sparse_attention_func(q, k, v, None, mask_packed=packed))
    assert torch.equal(out, sa.sparse_attention_func(q, k, v, None, mask_packed=packed, tile_map=sa.tile_map(packed, min_skip=0.0)))
    assert (out[:, :, row + 64] == 0).all()
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for h in (0, heads - 1):
        ref = O.sparse_attention_ref(*(t[:, h:h + 1].float().cpu() for t in (q, k, v)), mask)
        assert torch.allclose(out[:, h:h + 1].float().cpu(), ref, atol=1e-2, rtol=rtol)
