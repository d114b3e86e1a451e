"""The forward whose wavefronts share 32 query rows and split the keys, which small grids take: edges of the
tiles, of the rule that chooses it, reference points that differ between the wavefronts, rows that only one of
them has keys for."""
import importlib
import sys

import numpy as np
import pytest
import torch

from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sa():
    importlib.import_module("python.sparse_attention")
    return sys.modules["python.sparse_attention"]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 80, 96, 128])
@pytest.mark.parametrize("N", [129, 191, 193, 256, 321, 577])
def test_against_the_oracle(sa, dev, N, D, dtype):
    g = torch.Generator().manual_seed(N + D)
    q, k, v = (torch.randn(1, 2, N, D, generator=g).to(dtype) for _ in range(3))
    big = 6 if dtype == torch.float16 else 2                    # (bf16 operands: what their rounding leaves of such scores)
    q *= 1 + (big - 1) * (torch.arange(N) % 7 == 0)[:, None]     # scores far outside the window in some rows
    k[:, :, N // 3] *= 2                                        # ... by one key, in one wavefront's tiles
    mask = torch.rand(1, 2, N, N, generator=g) < 0.3
    mask[:, :, 1] = False
    mask[:, :, 2] = False
    mask[:, :, 2, N - 1] = True                                  # one key, in the last tile
    mask[:, 1, 3:40, :64] = False                                # nothing for the first wavefront
    want = O.sparse_attention_ref(q.float(), k.float(), v.float(), mask)
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    out = sa.sparse_attention_func(qd, kd, vd, md)
    bar = 2e-2
    assert torch.allclose(out.float().cpu(), want, atol=bar, rtol=bar)
    assert not out[:, :, 1].any()
    packed = sa.pack_mask(md)
    for tm in (None, sa.tile_map(packed, min_skip=0.0)):
        assert torch.equal(out, sa.sparse_attention_func(qd, kd, vd, None, mask_packed=packed, tile_map=tm))
    # training: packed words and tile map as by-products
    leaf = qd.clone().requires_grad_(True)
    again = sa.sparse_attention(leaf, kd, vd, md, tile_map=True)
    assert torch.equal(out, again.detach())
    node = again.grad_fn
    while not hasattr(node, "tile_map"):
        node = node.next_functions[0][0]
    assert np.array_equal(node.tile_map.cpu().numpy(), O.tile_map_ref(mask).view(np.int32))


def test_lse_and_words(dev):
    N, D = 333, 64
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(1, 3, N, D, generator=g).half().to(dev) for _ in range(3))
    mask = torch.rand(1, 3, N, N, generator=g) < 0.2
    mask[:, :, 5] = False
    lse, packed = torch.empty(1, 3, N, device=dev), torch.empty(1, 3, N, (N + 31) // 32, dtype=torch.int32, device=dev)
    m = sys.modules["python.sparse_attention"].sparse_attn_cuda
    m.forward_bool_mask(q, k, v, mask.to(dev), torch.empty_like(q), lse, 0.125, True, packed)
    assert np.array_equal(packed.cpu().numpy(), O.pack_mask_ref(mask))
    s = (q.float() @ k.float().transpose(-1, -2)).cpu() * 0.125
    want = torch.logsumexp(s.masked_fill(~mask, float("-inf")), -1)
    assert torch.allclose(lse.cpu(), want, atol=2e-3) and bool((lse[:, :, 5] == -float("inf")).all())
