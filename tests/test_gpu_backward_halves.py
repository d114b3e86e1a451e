"""dK/dV at head dim 128 by work-groups of 128 keys whose wavefronts share the rows: whole grids of them, and the last heads of larger ones."""
import importlib
import sys

import pytest
import torch

from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


# Bound: probabilities and dS are rounded to 16 bits before the second product, as in the other backward tests.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, N", [(30, 641), (25, 1153), (5, 3000), (87, 641), (70, 897), (66, 1024), (65, 993)])
def test_halves_against_the_oracle(dev, heads, N, dtype):
    """Grids of one round, first and last row of a tile; a second round of one head and of several."""
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + heads)
    q, k, v, do = (torch.randn(1, N, heads, 128, device=dev, generator=g).to(dtype).transpose(1, 2) for _ in range(4))
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    mask[..., N // 2, :] = False                                       # a row that keeps nothing
    mask[..., 128:320, 64:96] = False                                  # rows of one half alone
    mask[..., 128:320, 96:256] &= (torch.arange(128, 320, device=dev) % 64 < 32)[:, None]
    mask[..., N - 1] = False
    mask[..., N - 1, N - 1] = True                                     # the last key is kept by the last row alone
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    packed = sa.pack_mask(mask)
    out = sa.sparse_attention(*leaves, None, mask_packed=packed)
    grads = torch.autograd.grad(out, leaves, do, retain_graph=True)
    assert all(torch.equal(x, y) for x, y in zip(grads, torch.autograd.grad(out, leaves, do)))
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].float().cpu() for t in (q, k, v, do)]
        refs = O.sparse_attention_bwd_ref(*one[:3], mask.cpu(), one[3], scale=128 ** -0.5)
        for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
            err = (got[:, h:h + 1].float().cpu() - ref).abs()
            assert (err <= 1e-4 + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, h, float(err.max()))
