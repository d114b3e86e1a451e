"""Head dims between the kernels' own (any multiple of 8, no padding copies) and fp32 tensors (converted in one
launch, results widened by the kernels), at the edges of the tiles."""
import importlib
import sys

import pytest
import torch

from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [8, 24, 56, 72, 80, 88, 96, 104, 120])
@pytest.mark.parametrize("N", [16, 64, 129])
def test_head_dims_between_the_kernels(dev, N, D):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator().manual_seed(N * D)
    q, k, v, do = (torch.randn(2, N, 2, D, generator=g).bfloat16().transpose(1, 2) for _ in range(4))
    mask = torch.rand(2, 2, N, N, generator=g) < 0.4
    mask[1, 0, N - 1] = False
    refs = [t.float().requires_grad_(True) for t in (q, k, v)]
    ref = O.sparse_attention_ref(*refs, mask)
    ref.backward(do.float())
    results = {}
    for dtype in (torch.bfloat16, torch.float32):
        # a larger buffer around the tensors, filled with NaN: nothing beyond a row takes part
        leaves = []
        for t in (q, k, v):
            buf = torch.full((2, N, 2, D + 8), float("nan"), dtype=dtype, device=dev)
            view = buf[..., :D].transpose(1, 2)
            view.copy_(t.to(dev, dtype))
            leaves.append(view.detach().requires_grad_(True))
        out = sa.sparse_attention(*leaves, mask.to(dev))
        assert torch.equal(out, sa.sparse_attention_func(*(t.detach() for t in leaves), mask.to(dev)))
        out.backward(do.to(dev, dtype))
        results[dtype] = [out.detach()] + [t.grad for t in leaves]
        dense = [t.to(dev, dtype).requires_grad_(True) for t in (q, k, v)]
        o2 = sa.sparse_attention(*dense, mask.to(dev))
        o2.backward(do.to(dev, dtype))
        assert o2.dtype == dtype and all(torch.equal(a, b) for a, b in zip(results[dtype], [o2.detach()] + [t.grad for t in dense]))
    for a, b in zip(results[torch.bfloat16], results[torch.float32]):
        assert torch.equal(a.float(), b)                     # fp32 callers get the bf16 results, widened
    for got, want in zip(results[torch.float32], [ref.detach()] + [t.grad for t in refs]):
        assert ((got.cpu() - want).abs() <= 1e-4 + 2e-2 * want.abs().max() + 2e-2 * want.abs()).all()
