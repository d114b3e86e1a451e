"""The dK/dV kernel of head dim 64 with its V fragments in LDS, which grids of more than two work-groups per CU take, gives
the bits of the one that holds them in registers (the same heads in a smaller grid)."""
import importlib
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [40, 64])
@pytest.mark.parametrize("heads,N", [(172, 321), (130, 513), (103, 639), (257, 300)])       # around 2 and beyond 4 x 256 tiles
def test_same_bits_as_a_small_grid(dev, heads, N, D, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    assert torch.cuda.get_device_properties(dev).multi_processor_count * 2 < heads * ((N + 127) // 128)
    g = torch.Generator(device=dev).manual_seed(N)
    q, k, v, do = (torch.randn(1, heads, N, D, device=dev, generator=g).to(dtype) for _ in range(4))
    mask = torch.rand(1, heads, N, N, device=dev, generator=g) < 0.3
    mask[:, :, :, 64:160] = False
    mask[:, :, N // 2] = False
    packed = sa.pack_mask(mask)
    for scale in (D ** -0.5, -2.5):                              # the second needs the post-multiplier
        def grads(first, last, tm=None):
            leaves = [t[:, first:last].detach().requires_grad_(True) for t in (q, k, v)]
            out = sa.SparseAttentionFunction.apply(*leaves, packed[:, first:last].contiguous(), None, scale, N, tm)
            return torch.autograd.grad(out, leaves, do[:, first:last])
        want = grads(0, heads)
        for a, b in zip(want, grads(0, heads, sa.tile_map(packed, min_skip=0.0))):
            assert torch.equal(a, b)
        half = heads // 2            # at most 2 work-groups per CU, and enough for the forward that does not split the keys
        for first in (0, heads - half):
            for a, b in zip(want, grads(first, first + half)):
                assert torch.equal(a[:, first:first + half], b)
