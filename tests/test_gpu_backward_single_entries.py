"""dK/dV passes over a block of 32 query rows that keeps none of a wavefront's 32 keys: blocks that keep one entry, in a corner, between empty ones."""
import importlib
import sys

import pytest
import torch

from _launches import launches
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


# Bound: as in the other backward tests, the 16-bit roundings of probabilities and dS before the second product.
@pytest.mark.parametrize("row, key", [(0, 0), (31, 31), (31, 0), (0, 31)])
@pytest.mark.parametrize("D, heads, N", [(64, 3, 641), (64, 90, 672), (128, 3, 513), (128, 52, 671)])      # one launch, two; of four wavefronts, of eight
def test_one_entry_in_a_block(dev, D, heads, N, row, key):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator().manual_seed(N + D + row + key)
    nb = (N + 31) // 32
    mask = torch.zeros(nb, 32, nb, 32, dtype=torch.bool)
    mask[:, row, :, key] = torch.rand(nb, nb, generator=g) < 0.5
    mask = mask.view(1, 1, 32 * nb, 32 * nb)[..., :N, :N].contiguous()
    q, k, v, do = (torch.randn(1, heads, N, D, generator=g).to(torch.bfloat16).to(dev) for _ in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    packed = sa.pack_mask(mask.to(dev))
    if N % 32:
        packed[..., -1] |= -1 << (N % 32)                              # bits beyond the last key, as a packer of one's own may leave them
    out = sa.sparse_attention(*leaves, None, mask_packed=packed.expand(1, heads, -1, -1).contiguous())
    grads = []
    ran = launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do)))
    assert any((name, args[2]) == ("attn_bwd_dkv_kernel", "8" if D == 128 else "4") if heads > 3 else name == "attn_bwd_both_kernel" for name, args, _ in ran), ran
    one = [t[:, -1:].detach().float().cpu() for t in (q, k, v, do)]
    refs = O.sparse_attention_bwd_ref(*one[:3], mask, one[3], scale=D ** -0.5)
    for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
        err = (got[:, -1:].float().cpu() - ref).abs()
        assert (err <= 1e-4 + 1e-2 * ref.abs().max() + 2e-2 * ref.abs()).all(), (name, float(err.max()))
