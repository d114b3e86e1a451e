"""fp32 tensors whose q the forward itself rounds to bf16: the same bits as from tensors that were rounded beforehand, the backward included."""
import importlib
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


# below the size from which the forward does it; keys split between wavefronts (up to head dim 64, at 128), one row block, edges of tiles and
# of 16-byte pieces, two mask tiles per request at any N and at multiples of 128
@pytest.mark.parametrize("heads, N", [(3, 200), (3, 1), (62, 200), (30, 193), (2000, 33), (3000, 16), (520, 129), (96, 577), (100, 1000), (110, 1024)])
@pytest.mark.parametrize("D", [8, 32, 64, 80, 128])
@pytest.mark.parametrize("layout", ["bhnd", "bnhd"])
def test_same_bits_as_from_rounded_tensors(dev, heads, N, D, layout):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + D)

    def rows():
        t = torch.randn((1, heads, N, D) if layout == "bhnd" else (1, N, heads, D), device=dev, generator=g)
        return t if layout == "bhnd" else t.transpose(1, 2)

    q, k, v, do = (rows() for _ in range(4))
    q[0, 0, N // 2, D // 2] = float("inf")                             # a row of NaN among the others
    q[0, -1, 0, 0] = 3.4e38                                            # rounds to an infinity
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    packed = sa.pack_mask(mask)

    def run(dtype, m, p):
        leaves = [t.to(dtype).requires_grad_(True) for t in (q, k, v)]
        out = sa.sparse_attention(*leaves, m, mask_packed=p)
        saved = out.grad_fn.saved_tensors[:3]
        grads = torch.autograd.grad(out, leaves, do.to(dtype))
        plain = sa.sparse_attention_func(*(t.detach() for t in leaves), m, mask_packed=p)
        return [out.detach(), plain, *grads, *saved]

    for m, p in ((mask, None), (None, packed)):
        for a, b in zip(run(torch.float32, m, p), run(torch.bfloat16, m, p)):
            assert torch.equal(a.float().nan_to_num(nan=7e37, posinf=8e37, neginf=9e37), b.float().nan_to_num(nan=7e37, posinf=8e37, neginf=9e37))
