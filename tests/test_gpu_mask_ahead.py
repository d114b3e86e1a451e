"""The forward from the boolean mask with its bytes requested two tiles ahead (grids that are not one round in step, lengths
that are no multiple of 128): the bits of the forward from the packed words, by-products included, at the ends of the walk."""
import importlib
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("N", [16, 63, 65, 127, 129, 191, 193, 257, 320, 449, 1000])       # 1 to 16 tiles, odd and even
@pytest.mark.parametrize("groups", [400, 900])                                             # fewer and more than three on a CU
def test_same_bits_as_the_packed_words(dev, N, D, dtype, groups):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    heads = groups // ((N + 127) // 128)
    g = torch.Generator(device=dev).manual_seed(N)
    q, k, v = (torch.randn(1, heads, N, D, device=dev, generator=g).to(dtype) for _ in range(3))
    mask = torch.rand(1, heads, N, N, device=dev, generator=g) < 0.3
    packed = sa.pack_mask(mask)
    want = sa.sparse_attention_func(q, k, v, None, mask_packed=packed)
    assert torch.equal(want, sa.sparse_attention_func(q, k, v, mask))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]          # with the words as a by-product, which the gradients use
    out = sa.sparse_attention(*leaves, mask)
    assert torch.equal(want, out)
    ref = torch.autograd.grad(sa.sparse_attention(*leaves, None, mask_packed=packed), leaves, want)
    assert all(torch.equal(a, b) for a, b in zip(ref, torch.autograd.grad(out, leaves, want)))
