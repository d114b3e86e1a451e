"""The backward that holds a whole head in one work-group (N <= 256, head dim <= 64), at the edges of its sizes (128 and 256 keys, wavefronts of 32 and of
64) and of its blocks of 32 rows and keys."""
import importlib
import sys

import pytest
import torch

from _launches import launches
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [1, 31, 33, 64, 65, 97, 128, 129, 160, 192, 193, 225, 256]


def _inputs(B, H, N, D, dtype, dev):
    g = torch.Generator().manual_seed(1000 * N + D)
    # rows of the projections' layout, inside larger buffers of NaN: nothing beyond a row takes part
    out = []
    for _ in range(4):
        buf = torch.full((B, N, H, D + 8), float("nan"), dtype=dtype)
        buf[..., :D] = torch.randn(B, N, H, D, generator=g)
        out.append(buf.to(dev)[..., :D].transpose(1, 2))
    mask = torch.rand(B, H, N, N, generator=g) < 0.3
    mask[:, :, N // 2] = False                                   # a row that keeps nothing
    mask[:, :, :, N // 3] = False                                # a key that nobody keeps
    if N > 96:
        mask[0, 0, 32:64, 64:96] = False                         # a block of 32 x 32 without any
        mask[0, 0, :, 96:] = False                               # wavefronts without any
    return out, mask


# Scores are products with 16-bit q, scaled and rounded once more (2^-9 in bf16) as in the forward.  The inputs of the
# large scale are therefore small, so that its scores have the others' size.
# Bound: probabilities and dS are rounded to 16 bits before the second product, as in the longer kernels: half a unit
# in the last place of each factor, 1e-2 (fp16, bf16's operands 2e-2) of the entry and of the largest one.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [8, 32, 40, 64])
@pytest.mark.parametrize("N", LENGTHS)
@pytest.mark.parametrize("heads", [2, 150])                      # more heads than compute units in the second
def test_against_the_oracle(dev, N, D, dtype, heads):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    (q0, k, v, do), mask = _inputs(2, heads, N, D, dtype, dev)
    packed = sa.pack_mask(mask.to(dev))
    for scale in (D ** -0.5, -2.5):                                   # the second needs the post-multiplier
        q = q0 if scale > 0 else q0 * 2.0 ** -4
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        out = sa.SparseAttentionFunction.apply(*leaves, packed, None, scale, N)
        grads = []
        kernels = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do, retain_graph=True)))]
        assert kernels == ["attn_bwd_head_kernel"]
        assert all(torch.equal(x, y) for x, y in zip(grads, torch.autograd.grad(out, leaves, do)))
        rtol = 1e-2 if dtype == torch.float16 else 2e-2
        floor = 1e-4 * max(1.0, abs(scale))
        for b, h in ((0, 0), (1, heads - 1)):
            one = [t[b:b + 1, h:h + 1].float().cpu() for t in (q, k, v, do)]
            refs = O.sparse_attention_bwd_ref(*one[:3], mask[b:b + 1, h:h + 1], one[3], scale=scale)
            for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
                err = (got[b:b + 1, h:h + 1].float().cpu() - ref).abs()
                assert (err <= floor + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, b, h, scale, float(err.max()))
