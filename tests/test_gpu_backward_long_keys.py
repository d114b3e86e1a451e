"""The dK/dV kernel of head dim 128 in its two widths (128 and 256 keys per work-group), at the edges of both."""
import importlib
import sys

import pytest
import torch

from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,N", [(1, 1, 128), (2, 65, 129), (1, 129, 256), (2, 64, 384), (1, 65, 513), (1, 64, 639), (1, 33, 1025)])
def test_both_widths_against_the_oracle(dev, B, H, N, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N)
    q, k, v, do = (torch.randn(B, H, N, 128, device=dev, generator=g).to(dtype) for _ in range(4))
    mask = torch.rand(B, H, N, N, device=dev, generator=g) < 0.3
    mask[:, :, :, 64:128] = False                                # a key tile nobody keeps
    mask[:, :, N // 2] = False
    packed = sa.pack_mask(mask)
    want = None
    for tm in (None, sa.tile_map(packed, min_skip=0.0)):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        sa.sparse_attention(*leaves, None, mask_packed=packed, tile_map=tm).backward(do)
        got = [t.grad for t in leaves]
        assert want is None or all(torch.equal(a, b) for a, b in zip(want, got))
        want = got
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for h in (0, H - 1):                                         # the first and the last head against the oracle
        refs = O.sparse_attention_bwd_ref(*(t[-1:, h:h + 1].float().cpu() for t in (q, k, v)), mask[-1:, h:h + 1].cpu(),
                                          do[-1:, h:h + 1].float().cpu())
        for a, r in zip(want, refs):
            assert ((a[-1:, h:h + 1].float().cpu() - r).abs() <= 1e-4 + 1e-2 * r.abs().max() + rtol * r.abs()).all()
