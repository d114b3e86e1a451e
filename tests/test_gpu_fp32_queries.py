"""fp32 tensors whose q the forward itself rounds to bf16: the same bits as from tensors that were rounded beforehand, the backward included."""
import ctypes
import importlib
import sys

import pytest
import torch

import _capi
from _launches import launches

pytestmark = pytest.mark.gpu


# below the size from which the forward does it; one row block, edges of tiles and of 16-byte pieces, two mask tiles per request at any N and at
# multiples of 128; keys split between wavefronts and work-groups of 64 rows (test_forms_of_the_forward)
@pytest.mark.parametrize("heads, N", [(3, 200), (3, 1), (62, 200), (30, 193), (2000, 33), (3000, 16), (520, 129), (96, 577), (100, 1000), (110, 1024),
                                      (64, 256), (32, 512), (16, 1024)])
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


# Inference from 11 * 2^16 elements on; training from 2^20 and 512 keys on, head dims beyond 32, unless every head has a boolean mask of its own.
@pytest.mark.parametrize("heads, N, D, training, masks, rounds", [
    (44, 256, 64, False, "own", True), (44, 255, 64, False, "own", False), (256, 128, 32, False, "shared", True), (64, 64, 128, False, "packed", False),
    (64, 512, 64, True, "shared", True), (64, 512, 64, True, "packed", True), (64, 512, 64, True, "own", False), (31, 512, 64, True, "packed", False), (64, 511, 80, True, "shared", False),
    (1000, 64, 64, True, "shared", False), (512, 64, 128, True, "packed", False), (96, 577, 32, True, "shared", False), (96, 577, 80, True, "shared", True)])
def test_which_forward_rounds_q(dev, heads, N, D, training, masks, rounds):
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v = (torch.randn(1, heads, N, D, device=dev, generator=g).requires_grad_(training) for _ in range(3))
    mask = torch.rand(1, heads if masks == "own" else 1, N, N, device=dev, generator=g) < 0.3
    packed = sa.pack_mask(mask)
    given = dict(mask_packed=packed) if masks == "packed" else {}
    m = None if masks == "packed" else mask
    ran = launches(lambda: (sa.sparse_attention if training else sa.sparse_attention_func)(q, k, v, m, **given))
    names = [name for name, _, _ in ran]
    wide = [args[8] for name, args, _ in ran if name == "attn_fwd_kernel"]
    assert names.count("to_bf16_kernel") == 1 and wide == ["true" if rounds else "false"], ran


@pytest.mark.parametrize("heads, N, D, training, split, halves", [(64, 256, 64, False, True, False), (32, 512, 64, True, True, False),
                                                                  (64, 256, 80, False, False, True), (16, 1024, 128, True, False, True)])
def test_forms_of_the_forward(dev, heads, N, D, training, split, halves):
    """Sizes of test_same_bits_as_from_rounded_tensors are those at which these forms round q."""
    importlib.import_module("python.sparse_attention")
    sa = sys.modules["python.sparse_attention"]
    q, k, v = (torch.randn(1, heads, N, D, device=dev).requires_grad_(training) for _ in range(3))
    mask = torch.rand(1, 1, N, N, device=dev) < 0.3
    for m, packed in ((mask, None), (None, sa.pack_mask(mask))):
        ran = launches(lambda: (sa.sparse_attention if training else sa.sparse_attention_func)(q, k, v, m, mask_packed=packed))
        forms = [tuple(a == "true" for a in args[7:10]) for name, args, _ in ran if name == "attn_fwd_kernel"]
        assert forms == [(split, True, halves)], ran


# Callers of the C interface may have any size rounded, with any by-products: work-groups of one round and of several, keys split, halves.
@pytest.mark.parametrize("D", [32, 64, 80, 128])
@pytest.mark.parametrize("heads, N", [(3, 200), (3, 16), (30, 193), (400, 130), (400, 256), (16, 333), (260, 300)])
def test_c_call_with_by_products(dev, capi, heads, N, D):
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k, v = (torch.randn(1, heads, N, D, device=dev, generator=g) for _ in range(3))
    k16, v16 = k.bfloat16(), v.bfloat16()
    mask = torch.rand(1, heads, N, N, device=dev, generator=g) < 0.3

    def run(wide):
        made = dict(out=torch.empty_like(k16), q=torch.zeros_like(k16), lse=torch.empty(1, heads, N, device=dev),
                    packed=torch.empty(1, heads, N, (N + 31) // 32, dtype=torch.int32, device=dev),
                    map=torch.empty(_capi.load().sma_tile_map_words(N) * heads, dtype=torch.int32, device=dev))
        q16 = q.bfloat16()
        t = {name: ctypes.pointer(_capi.SmaTensor.of(x)) for name, x in (("q", q if wide else q16), ("k", k16), ("v", v16), ("out", made["out"]))}
        call = _capi.SmaFwdCall(mask=mask.data_ptr(), mask_stride_b=heads * N * N, mask_stride_h=N * N, lse=made["lse"].data_ptr(),
                                packed_out=made["packed"].data_ptr(), map_out=made["map"].data_ptr(), B=1, H=heads, N=N, D=D, scale=D ** -0.5,
                                dtype=_capi.SMA_DTYPE_BF16, **t)
        stream = torch.cuda.current_stream().cuda_stream
        if wide:
            assert capi.sma_attn_fwd_call_q32(ctypes.byref(call), ctypes.pointer(_capi.SmaTensor.of(made["q"])), stream) == _capi.SMA_OK
        else:
            assert capi.sma_attn_fwd_call(ctypes.byref(call), stream) == _capi.SMA_OK
            made["q"] = q16
        torch.cuda.synchronize()
        return made

    got, want = run(True), run(False)
    for name in got:
        assert torch.equal(got[name], want[name]), name
