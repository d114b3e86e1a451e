"""The backward that holds a whole head in one work-group where test_gpu_backward_short.py does not reach: 257 to 512 keys at
head dims up to 64, up to 256 at those above, at the edges of its sizes, of its 32 rows and of its wavefronts' keys."""
import importlib
import sys

import pytest
import torch

from _launches import launches, places
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu

CASES = [(N, D, 96) for N in (257, 288, 289, 321, 384, 449, 480, 511, 512) for D in (16, 64)]           # 192 heads fill their round
CASES += [(N, D, h) for N in (1, 33, 64, 65, 127, 128) for D in (72, 96, 128) for h in (1, 150)]
CASES += [(N, D, 80) for N in (129, 160, 192, 193, 255, 256) for D in (80, 96, 120, 128)]


# Bound: as in test_gpu_backward_short.py, which the shorter sizes of the same kernel pass: probabilities and dS are rounded
# to 16 bits before the second product, half a unit in the last place of each factor.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N, D, heads", CASES)
def test_against_the_oracle(dev, N, D, heads, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator().manual_seed(1000 * N + D)
    given = []
    for _ in range(4):                               # inside larger buffers of NaN: nothing beyond a row takes part
        buf = torch.full((2, N, heads, D + 8), float("nan"), dtype=dtype)
        buf[..., :D] = torch.randn(2, N, heads, D, generator=g)
        given.append(buf.to(dev)[..., :D].transpose(1, 2))
    mask = torch.rand(2, heads, N, N, generator=g) < 0.3
    mask[:, :, N // 2] = False                       # a row that keeps nothing
    mask[:, :, :, N // 3] = False                    # a key that nobody keeps
    if N > 96:
        mask[0, 0, :32, :64] = False                 # the first rows' first wavefronts without any
        mask[0, 0, 32:64, 64:128] = False            # others in the midst
        mask[0, 0, 64:, 96:] = False                 # the last ones from there on
    packed = sa.pack_mask(mask.to(dev))
    for scale in (D ** -0.5, -2.5):                  # the second needs the post-multiplier; its scores have the others' size
        q, k, v, do = given
        leaves = [t.detach().requires_grad_(True) for t in (q if scale > 0 else q * 2.0 ** -4, k, v)]
        out = sa.SparseAttentionFunction.apply(*leaves, packed, None, scale, N)
        grads = []
        kernels = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do, retain_graph=True)))]
        assert kernels == ["attn_bwd_head_kernel"]
        assert all(torch.equal(x, y) for x, y in zip(grads, torch.autograd.grad(out, leaves, do)))
        rtol = 1e-2 if dtype == torch.float16 else 2e-2
        floor = 1e-4 * max(1.0, abs(scale))
        for b, h in {(0, 0), (1, heads - 1)}:
            one = [t[b:b + 1, h:h + 1].detach().float().cpu() for t in (*leaves, do)]
            refs = O.sparse_attention_bwd_ref(*one[:3], mask[b:b + 1, h:h + 1], one[3], scale=scale)
            for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
                err = (got[b:b + 1, h:h + 1].float().cpu() - ref).abs()
                assert (err <= floor + 1e-2 * ref.abs().max() + rtol * ref.abs()).all(), (name, b, h, scale, float(err.max()))


# Heads as 32nds of a round of one work-group on a CU.  Gradients are the same bits with and without a tile map, so it is the same kernel.
@pytest.mark.parametrize("N, D, part, whole", [
    (512, 64, 16, False), (512, 64, 20, True), (385, 64, 24, True), (512, 64, 40, False), (512, 64, 48, True), (385, 64, 80, True), (512, 64, 66, False),
    (320, 64, 20, False), (320, 64, 22, True), (257, 64, 50, False), (384, 64, 55, True), (320, 64, 84, False), (320, 64, 88, True),
    (512, 32, 20, True), (512, 32, 44, False), (512, 32, 50, True), (512, 32, 74, False), (400, 32, 80, True),
    (384, 32, 22, True), (384, 32, 56, False), (320, 32, 60, True), (384, 32, 96, False)])
def test_grids_that_take_it(dev, N, D, part, whole):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    heads = part * places() // 32
    g = torch.Generator(device=dev).manual_seed(N + part)
    q, k, v, do = (torch.randn(1, heads, N, D, device=dev, generator=g).half() for _ in range(4))
    nb = (N + 63) // 64
    blocks = (torch.rand(1, 1, nb, nb, device=dev, generator=g) < 0.25) | torch.eye(nb, dtype=torch.bool, device=dev)
    mask = blocks.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N].contiguous()
    packed = sa.pack_mask(mask)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    ways = []
    for tile_map in (None, sa.tile_map(packed, min_skip=0.0)):
        out = sa.sparse_attention(*leaves, None, mask_packed=packed, tile_map=tile_map)
        grads = []
        kernels = [name for name, _, _ in launches(lambda: grads.extend(torch.autograd.grad(out, leaves, do)))]
        assert (kernels == ["attn_bwd_head_kernel"]) == whole, kernels
        ways.append(grads)
    assert all(torch.equal(x, y) for x, y in zip(*ways))
    h = heads - 1
    refs = O.sparse_attention_bwd_ref(*(t[:, h:h + 1].detach().float().cpu() for t in (q, k, v)), mask.cpu(), do[:, h:h + 1].float().cpu(), scale=D ** -0.5)
    for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):          # the bound of the test above
        err = (got[:, h:h + 1].float().cpu() - ref).abs()
        assert (err <= 1e-4 + 1e-2 * ref.abs().max() + 1e-2 * ref.abs()).all(), (name, float(err.max()))
