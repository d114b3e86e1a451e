"""The dQ and dK/dV kernels form 16 x 16 blocks: lengths whose last block of 16 or 32 rows and keys holds one, all but one or all of them, head dims
up to, at and between the kernels' own, in one launch and in two."""
import importlib
import sys

import pytest
import torch

from _launches import launches
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


# Bound: probabilities and dS are rounded to 16 bits before the second product: half a unit in the last place of each factor, 1e-2 (fp16, bf16's
# operands 2e-2) of the entry and of the largest one, as in the other backward tests.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [8, 32, 48, 64, 80, 96, 104, 128])
@pytest.mark.parametrize("N", [513, 527, 528, 529, 560, 575, 576, 593])
@pytest.mark.parametrize("heads", [3, 160])
def test_against_the_oracle(dev, N, D, dtype, heads):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator().manual_seed(1000 * N + D)
    # rows of the projections' layout, inside larger buffers of NaN: nothing beyond a row takes part
    q, k, v, do = (torch.full((1, N, heads, D + 8), float("nan"), dtype=dtype).to(dev)[..., :D].transpose(1, 2) for _ in range(4))
    for t in (q, k, v, do):
        t.copy_(torch.randn(1, heads, N, D, generator=g))
    mask = torch.rand(1, 1, N, N, generator=g) < 0.3
    mask[:, :, N - 1] = False                                    # the last row keeps nothing
    mask[:, :, :, N // 3] = False                                # a key that nobody keeps
    mask[:, :, 32:48, 64:80] = False                             # a block without any, and one of 32 x 32
    mask[:, :, 96:128, 32:64] = False
    mask[:, :, 17] = True
    packed = sa.pack_mask(mask.to(dev))
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*leaves, None, mask_packed=packed)
    grads = []
    ran = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do)))]
    assert ran == (["attn_bwd_delta_kernel", "attn_bwd_both_kernel"] if heads == 3 else ["attn_bwd_dq_kernel", "attn_bwd_dkv_kernel"])
    rtol = 1e-2 if dtype == torch.float16 else 2e-2
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].detach().float().cpu() for t in (q, k, v, do)]
        refs = O.sparse_attention_bwd_ref(*one[:3], mask, one[3], scale=D ** -0.5)
        for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
            err = (got[:, h:h + 1].float().cpu() - ref).abs()
            assert (err <= 1e-4 + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, h, float(err.max()))
