"""Head dims between the kernels' own (any multiple of 8, no padding copies) and fp32 tensors (converted in one
launch, results widened by the kernels), at the edges of the tiles."""
import importlib
import sys

import pytest
import torch

from _launches import launches, places
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


# 65 to 80 have kernels with five blocks of 16 result columns: the second 64 columns of a row's store are 16 wide.  One key beyond whole tiles, few heads (dQ
# and dK/dV in one launch) and more than fit that, a walk over tiles of a map.
@pytest.mark.parametrize("D", [72, 80])
@pytest.mark.parametrize("heads, N, blocks", [(3, 257, False), (80, 300, False), (60, 577, True), (34, 1024, False), (4, 1025, True)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_kernels_for_80(dev, heads, N, blocks, D, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + D)
    rounded = torch.bfloat16 if dtype == torch.float32 else dtype
    leaves = []
    for _ in range(4):                                       # rows between columns of NaN
        buf = torch.full((1, N, heads, D + 8), float("nan"), dtype=dtype, device=dev)
        view = buf[..., :D].transpose(1, 2)
        view.copy_(torch.randn(1, heads, N, D, device=dev, generator=g).to(rounded))
        leaves.append(view)
    q, k, v, do = leaves
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    if blocks:
        nb = (N + 63) // 64
        mask &= (torch.rand(1, 1, nb, nb, device=dev, generator=g) < 0.5).repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N]
    mask[..., 5, :] = False
    qkv = [t.detach().requires_grad_(True) for t in (q, k, v)]
    made = []

    def step():
        out = sa.sparse_attention(*qkv, mask, tile_map=True if blocks else None)
        made.extend([out.detach(), *torch.autograd.grad(out, qkv, do)])
    ran = [(name, args) for name, args, _ in launches(step) if name.startswith("attn_") and name != "attn_bwd_delta_kernel"]
    assert {name: args[3 if name == "attn_fwd_kernel" else 1] for name, args in ran} == {name: "80" for name, _ in ran}, ran
    dense = [t.contiguous().detach().requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*dense, mask, tile_map=True if blocks else None)
    assert all(torch.equal(a, b) for a, b in zip(made, [out.detach(), *torch.autograd.grad(out, dense, do.contiguous())]))
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].detach().double().requires_grad_(True) for t in (q, k, v)]
        ref = O.sparse_attention_ref(*one, mask)
        wanted = [ref.detach(), *torch.autograd.grad(ref, one, do[:, h:h + 1].double())]
        for got, want in zip(made, wanted):                  # the bound of the test above
            assert ((got[:, h:h + 1].double() - want).abs() <= 1e-4 + 2e-2 * want.abs().max() + 2e-2 * want.abs()).all()


# The forward's tiles that have short rows (head dims to 32: 64 bytes;  in the second column half 65 to 80: 32 bytes, in training 64; 81 to 96: 64, fp32 whole ones): one tile and two, keys that end in either half
# and in the first or last of the rows that one request fills, work-groups of 64 rows (from 1024 rows on), two on a CU by the launcher's choice (800 heads).  With a whole head dim
# (80, 96) and rows that end before it.
@pytest.mark.parametrize("D", [24, 32, 72, 80, 88, 96])
@pytest.mark.parametrize("heads, N", [(3, 33), (800, 65), (800, 128), (110, 127), (110, 129), (60, 656), (60, 673), (90, 720), (20, 1025), (12, 1104)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_short_rows_of_the_second_half(dev, heads, N, D, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v = (torch.randn(1, heads, N, D, device=dev, generator=g).to(dtype) for _ in range(3))
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    mask[..., 3, :] = False
    mask[..., 4, :] = torch.arange(N, device=dev) == N - 1
    packed = sa.pack_mask(mask)
    out = sa.sparse_attention_func(q, k, v, mask)
    odd = (mask.to(torch.uint8) * 6).view(torch.bool)                  # bytes that are neither 0 nor 1
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    strided = [torch.nn.functional.pad(t, (0, 8), value=float("nan"))[..., :D] for t in (q, k, v)]
    for x in (sa.sparse_attention_func(q, k, v, odd), sa.sparse_attention_func(q, k, v, None, mask_packed=packed), sa.sparse_attention_func(*strided, mask),
              sa.sparse_attention_func(q, k, v, None, mask_packed=packed, tile_map=sa.tile_map(packed, min_skip=0.0)), sa.sparse_attention(*leaves, mask)):
        assert torch.equal(out, x)
    # the bound of the work-groups of 64 rows: the probabilities and the result are rounded once each, relative to the largest value of a row's mean
    eps = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].double() if dtype != torch.float32 else t[:, h:h + 1].bfloat16().double() for t in (q, k, v)]
        x = ((one[0] * D ** -0.5) @ one[1].transpose(-1, -2)).masked_fill(~mask, float("-inf"))
        ref = torch.softmax(x, -1).nan_to_num() @ one[2]
        shift = (eps * (one[0].abs() * D ** -0.5) @ one[1].abs().transpose(-1, -2)).masked_fill(~mask, 0).amax(-1)
        assert ((out[:, h:h + 1].double() - ref).abs() <= 1e-4 + one[2].abs().max() * (4 * eps + 2 * shift[..., None])).all()


# Head dim 32 in one round of more than three work-groups on a CU, which four share: wavefronts yield to each other as they advance, by the visits that a map of one
# word leaves them (a longer map: they don't).  Whole tiles and a last one of one key, pairs of tiles that end in either of theirs.
@pytest.mark.parametrize("N, tiles", [(257, 3), (320, 3), (512, 4), (700, 6), (2048, 16), (2100, 17)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_one_round_of_four_on_a_cu(dev, N, tiles, dtype):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    D, heads = 32, 4 * places() // tiles
    assert 3 * places() < heads * tiles <= 4 * places()
    g = torch.Generator(device=dev).manual_seed(N)
    q, k, v = (torch.randn(1, heads, N, D, device=dev, generator=g).to(dtype) for _ in range(3))
    nb = (N + 63) // 64
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    mask &= (torch.rand(1, 1, nb, nb, device=dev, generator=g) < 0.5).repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N]
    mask[..., 3, :] = False
    packed = sa.pack_mask(mask)
    out = sa.sparse_attention_func(q, k, v, mask)
    for x in (sa.sparse_attention_func(q, k, v, None, mask_packed=packed),
              sa.sparse_attention_func(q, k, v, None, mask_packed=packed, tile_map=sa.tile_map(packed, min_skip=0.0))):
        assert torch.equal(out, x)
    eps = 2.0 ** (-10 if dtype == torch.float16 else -7)               # the bound of the short rows' test
    for h in (0, heads - 1):
        one = [t[:, h:h + 1].double() if dtype != torch.float32 else t[:, h:h + 1].bfloat16().double() for t in (q, k, v)]
        x = ((one[0] * D ** -0.5) @ one[1].transpose(-1, -2)).masked_fill(~mask, float("-inf"))
        ref = torch.softmax(x, -1).nan_to_num() @ one[2]
        shift = (eps * (one[0].abs() * D ** -0.5) @ one[1].abs().transpose(-1, -2)).masked_fill(~mask, 0).amax(-1)
        assert ((out[:, h:h + 1].double() - ref).abs() <= 1e-4 + one[2].abs().max() * (4 * eps + 2 * shift[..., None])).all()
