"""The native call behind sparse_attention / sparse_attention_func: its autograd node keeps autograd's rules, and it
takes every combination of element type, head dim and layout that the Python API documents."""
import importlib
import sys

import pytest
import torch

from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sa():
    importlib.import_module("python.sparse_attention")
    return sys.modules["python.sparse_attention"]


def _problem(dev, N=70, D=64, dtype=torch.float16, seed=0):
    g = torch.Generator().manual_seed(seed)
    q, k, v, do = (torch.randn(2, 2, N, D, generator=g).to(dtype).to(dev) for _ in range(4))
    return q, k, v, do, (torch.rand(2, 2, N, N, generator=g) < 0.4).to(dev)


def test_node_follows_the_rules_of_autograd(sa, dev):
    q, k, v, do, mask = _problem(dev)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*leaves, mask)
    assert out.grad_fn.name() == "SparseAttentionFunctionBackward" and out.grad_fn.scale == 0.125
    want = torch.autograd.grad(out, leaves, do, retain_graph=True)
    again = torch.autograd.grad(out, leaves, do)
    assert all(torch.equal(a, b) for a, b in zip(want, again))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, leaves, do)
    # one of the three only, through an operation on either side
    kl = k.clone().requires_grad_(True)
    (gk,) = torch.autograd.grad(sa.sparse_attention(q, kl * 1.0, v, mask) * 2.0, (kl,), do)
    assert torch.allclose(gk.float(), want[1].float() * 2.0, rtol=1e-3, atol=1e-5)
    # an input changed in place between forward and backward is noticed
    x = q.clone().requires_grad_(True)
    y = x * 1.0
    out = sa.sparse_attention(y, k, v, mask)
    with torch.no_grad():
        y.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(do)
    # the function behind it, with the scale given
    f = sa.SparseAttentionFunction.apply(*leaves, None, mask, 0.125, 70)
    assert torch.equal(f, sa.sparse_attention_func(q, k, v, mask))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [1, 7, 8, 32, 40, 64, 65, 80, 96, 100, 120, 128])
@pytest.mark.parametrize("N", [5, 77, 200])
def test_types_head_dims_and_layouts(sa, dev, N, D, dtype):
    """Both layouts of every combination against the oracle, forward and backward."""
    g = torch.Generator().manual_seed(N + D)
    q, k, v, do = (torch.randn(2, N, 3, D, generator=g).to(dtype) for _ in range(4))
    mask = torch.rand(2, 1, N, N, generator=g) < 0.4
    mask[0, 0, min(3, N - 1)] = False
    refs = [t.transpose(1, 2).float().requires_grad_(True) for t in (q, k, v)]
    ref = O.sparse_attention_ref(*refs, mask.expand(2, 3, N, N))
    ref.backward(do.transpose(1, 2).float())
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for strided in (True, False):
        leaves = [(t.to(dev).transpose(1, 2) if strided else t.to(dev).transpose(1, 2).contiguous()).requires_grad_(True)
                  for t in (q, k, v)]
        out = sa.sparse_attention(*leaves, mask.to(dev))
        assert out.dtype == dtype and out.shape == (2, 3, N, D)
        assert torch.allclose(out.float().cpu(), ref.detach(), atol=2e-2, rtol=rtol)
        out.backward(do.to(dev).transpose(1, 2))
        for leaf, want in zip(leaves, refs):
            assert leaf.grad.dtype == dtype and leaf.grad.shape == want.grad.shape
            bound = 1e-4 + 2e-2 * want.grad.abs().max() + rtol * want.grad.abs()
            assert ((leaf.grad.float().cpu() - want.grad).abs() <= bound).all()
        with torch.no_grad():
            assert torch.equal(out, sa.sparse_attention(*leaves, mask.to(dev)))
