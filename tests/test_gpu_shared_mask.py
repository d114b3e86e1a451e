"""A mask that many heads share: packed with its tile map in one launch, before the attention."""
import importlib
import sys

import numpy as np
import pytest
import torch

import _capi
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [8, 9, 63, 64, 511, 512, 513, 1024, 2047, 2049, 2300])
def test_words_and_map_in_one_pass(dev, N):
    """Edges of a lane's 8 columns, of a work-group's 512 and of a map word's 2048, at odd addresses too."""
    g = torch.Generator().manual_seed(N)
    nb = (N + 63) // 64
    blocks = torch.rand(1, 2, nb, nb, generator=g)
    m = torch.rand(1, 2, N, N, generator=g) < 0.3
    at = blocks.repeat_interleave(64, 2).repeat_interleave(64, 3)[:, :, :N, :N]
    m = (m & (at > 0.3)) | (at > 0.7)                       # empty, mixed and full blocks
    m[..., -1] = False
    for shift in (0, 3):
        buf = torch.zeros(m.numel() + 16, dtype=torch.bool, device=dev)
        md = buf[shift:shift + m.numel()].view(m.shape)
        md.copy_(m.to(dev))
        packed, tm = _capi.pack_mask_map(md)
        torch.cuda.synchronize()
        assert np.array_equal(packed.cpu().numpy(), O.pack_mask_ref(m)), (N, shift)
        assert np.array_equal(tm.cpu().numpy(), O.tile_map_ref(m).view(np.int32)), (N, shift)


@pytest.mark.parametrize("share", ["heads", "all"])
def test_shared_mask_gives_the_bits_of_a_mask_per_head(dev, share):
    """4 x 32 heads of 1024 rows: the smallest problem whose shared mask is packed beforehand."""
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(3)
    q, k, v, do = (torch.randn(4, 32, 1024, 32, device=dev, generator=g).half() for _ in range(4))
    m = torch.rand(4 if share == "heads" else 1, 1, 1024, 1024, device=dev, generator=g) < 0.5
    m = m.tril_()
    full = m.expand(4, 32, 1024, 1024).contiguous()
    got, want = [], []
    for mask, to in ((m, got), (full, want)):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = sa.sparse_attention(*leaves, mask)
        to += [sa.sparse_attention_func(q, k, v, mask), out.detach(), *torch.autograd.grad(out, leaves, do)]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
