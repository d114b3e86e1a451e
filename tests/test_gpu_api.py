"""GPU tests of the Python surface (python/sparse_attention.py over the sparse_attn_cuda module):
same calls a user of the reference makes, checked against the oracle."""
import importlib
import math
import os
import sys

import numpy as np
import pytest
import torch

import harness
from oracle import sma_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sa():
    importlib.import_module("python.sparse_attention")
    mod = sys.modules["python.sparse_attention"]
    assert mod.HAS_CUDA_EXT, mod._EXT_ERROR
    return mod


def _inputs(B, H, N, dtype, seed, keep=0.25):
    g = torch.Generator().manual_seed(seed)
    q, k, v = [torch.randn(B, H, N, 64, generator=g).to(dtype) for _ in range(3)]
    mask = torch.rand(B, H, N, N, generator=g) < keep
    return q, k, v, mask


def test_pack_mask_returns_int32_words(sa, dev):
    _, _, _, mask = _inputs(2, 3, 100, torch.float16, 0)
    packed = sa.pack_mask(mask.to(dev))
    assert packed.dtype == torch.int32 and packed.shape == (2, 3, 100, 4) and packed.is_cuda
    assert np.array_equal(packed.cpu().numpy(), O.pack_mask_ref(mask))
    # a non-contiguous mask (transposed view) is packed by value, like any torch op would
    mt = mask.to(dev).transpose(-1, -2)
    assert np.array_equal(sa.pack_mask(mt).cpu().numpy(), O.pack_mask_ref(mask.transpose(-1, -2).contiguous()))


@pytest.mark.parametrize("fn_name", ["sparse_attention", "sparse_attention_func"])
@pytest.mark.parametrize("dtype,rtol", [(torch.float16, 1e-2), (torch.bfloat16, 2e-2)])
def test_forward_matches_oracle(sa, dev, fn_name, dtype, rtol):
    q, k, v, mask = _inputs(2, 4, 256, dtype, 1)
    mask[1, 2, 5, :] = False
    out = getattr(sa, fn_name)(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    assert out.dtype == dtype and out.shape == q.shape
    ref = O.sparse_attention_ref(q.float(), k.float(), v.float(), mask)
    assert torch.allclose(out.float().cpu(), ref, atol=1e-2, rtol=rtol)
    assert (out[1, 2, 5] == 0).all()


def test_fp32_inputs_are_computed_in_bf16_and_returned_as_fp32(sa, dev):
    """python/sparse_attention.py:140-142,151-152 of the reference."""
    q, k, v, mask = _inputs(1, 2, 128, torch.float32, 2)
    out = sa.sparse_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    assert out.dtype == torch.float32
    ref = O.sparse_attention_ref(q.bfloat16().float(), k.bfloat16().float(), v.bfloat16().float(), mask)
    assert torch.allclose(out.cpu(), ref, atol=1e-2, rtol=2e-2)
    assert torch.equal(out.cpu(), out.cpu().bfloat16().float())          # values are bf16 numbers


def test_non_contiguous_inputs_and_other_stream(sa, dev):
    q, k, v, mask = _inputs(2, 2, 192, torch.float16, 3)
    qd = q.to(dev).transpose(1, 2).contiguous().transpose(1, 2)           # [B,H,N,D] view, strided
    assert not qd.is_contiguous()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        out = sa.sparse_attention_func(qd, k.to(dev), v.to(dev), mask.to(dev))
    s.synchronize()
    ref = O.sparse_attention_ref(q.float(), k.float(), v.float(), mask)
    assert torch.allclose(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)


def test_binding_rejects_bad_arguments(sa, dev):
    import sparse_attn_cuda as ext
    q, k, v, mask = _inputs(1, 1, 64, torch.float16, 4)
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    packed = ext.pack_mask(md)
    out = torch.empty_like(qd)
    with pytest.raises(RuntimeError, match="head_dim"):
        ext.forward(qd[..., :48].contiguous(), kd[..., :48].contiguous(), vd[..., :48].contiguous(),
                    packed, out[..., :48].contiguous(), None, 0.125, False)
    with pytest.raises(RuntimeError, match="Unsupported dtype"):
        ext.forward(qd.float(), kd.float(), vd.float(), packed, out.float(), None, 0.125, False)
    with pytest.raises(RuntimeError, match="lse"):
        ext.forward(qd, kd, vd, packed, out, None, 0.125, True)
    with pytest.raises(RuntimeError, match="mask_packed"):
        ext.forward(qd, kd, vd, packed[..., :1].contiguous(), out, None, 0.125, False)
    with pytest.raises(RuntimeError, match="bool"):
        ext.pack_mask(md.to(torch.uint8))
    ext.forward(qd, kd, vd, packed, out, None, 0.125, False)             # and the good call works
    torch.cuda.synchronize()
    assert not torch.isnan(out).any()


def test_lse_is_saved_and_backward_matches_autograd_of_the_formulation(sa, dev):
    """.backward() of the reference raises AttributeError (sparse_attn_cuda.backward was never
    written, python/sparse_attention.py:91-94); here it must give the gradient of the operator."""
    q, k, v, mask = _inputs(1, 2, 96, torch.float16, 5, keep=0.4)
    mask[0, 1, 7, :] = False
    leaves = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    out = sa.sparse_attention(*leaves, mask.to(dev))
    g = torch.randn(out.shape, generator=torch.Generator().manual_seed(6)).to(torch.float16)
    out.backward(g.to(dev))
    ref_leaves = [t.float().requires_grad_(True) for t in (q, k, v)]
    ref = O.sparse_attention_ref(*ref_leaves, mask)
    ref.backward(g.float())
    for got, want, name in zip(leaves, ref_leaves, "qkv"):
        assert got.grad is not None and got.grad.dtype == torch.float16
        err = (got.grad.float().cpu() - want.grad).abs().max().item()
        assert torch.allclose(got.grad.float().cpu(), want.grad, atol=2e-2, rtol=2e-2), f"d{name} max err {err}"
    assert (leaves[0].grad[0, 1, 7] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_hip_backward_agrees_with_the_pytorch_recomputation(sa, dev, dtype):
    """The autograd function's HIP kernels against backward_recompute (PyTorch ops on the GPU from
    the same saved tensors); fp32 inputs go through bf16 as in the forward."""
    q, k, v, mask = _inputs(2, 3, 200, torch.float16, 9, keep=0.3)
    q, k, v = (t.to(dtype) for t in (q, k, v))
    leaves = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    md = mask.to(dev)
    out = sa.sparse_attention(*leaves, md)
    g = torch.randn(out.shape, generator=torch.Generator().manual_seed(10)).to(dtype).to(dev)
    out.backward(g)
    cdt = torch.bfloat16 if dtype == torch.float32 else dtype
    qc, kc, vc = (t.detach().to(cdt) for t in leaves)
    packed = sa.pack_mask(md)
    o2 = torch.empty_like(qc)
    lse = torch.empty(2, 3, 200, device=dev, dtype=torch.float32)
    ext = importlib.import_module("sparse_attn_cuda")
    ext.forward(qc, kc, vc, packed, o2, lse, 0.125, True)
    want = sa.backward_recompute(qc, kc, vc, o2, lse, md, g.to(cdt), 0.125)
    for got, ref, name in zip(leaves, want, "qkv"):
        assert got.grad.dtype == dtype
        ref = ref.float()
        bound = 1e-4 + 1e-2 * ref.abs().max() + 2e-2 * ref.abs()
        assert ((got.grad.float() - ref).abs() <= bound).all(), f"d{name}"


def test_extension_backward_checks_its_arguments(sa, dev):
    ext = importlib.import_module("sparse_attn_cuda")
    q, k, v, mask = _inputs(1, 1, 64, torch.float16, 3)
    qd, kd, vd = (t.to(dev) for t in (q, k, v))
    packed = ext.pack_mask(mask.to(dev))
    out, lse = torch.empty_like(qd), torch.empty(1, 1, 64, device=dev)
    ext.forward(qd, kd, vd, packed, out, lse, 0.125, True)
    dq, dk, dv = (torch.empty_like(qd) for _ in range(3))
    with pytest.raises(RuntimeError, match="dtype"):
        ext.backward(out.float(), qd, kd, vd, out, lse, packed, dq, dk, dv, 0.125)
    with pytest.raises(RuntimeError, match="lse"):
        ext.backward(out, qd, kd, vd, out, lse[..., :32], packed, dq, dk, dv, 0.125)
    with pytest.raises(RuntimeError, match="contiguous"):
        ext.backward(out, qd.transpose(2, 3).contiguous().transpose(2, 3), kd, vd, out, lse, packed, dq, dk, dv, 0.125)
    ext.backward(out, qd, kd, vd, out, lse, packed, dq, dk, dv, 0.125)
    torch.cuda.synchronize()
    assert torch.isfinite(dq).all() and torch.isfinite(dk).all() and torch.isfinite(dv).all()


def test_prepacked_mask_fast_path(sa, dev):
    q, k, v, mask = _inputs(1, 2, 130, torch.float16, 12)
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    packed = sa.pack_mask(md)
    a = sa.sparse_attention_func(qd, kd, vd, md)
    b = sa.sparse_attention_func(qd, kd, vd, None, mask_packed=packed)
    c = sa.sparse_attention(qd, kd, vd, None, mask_packed=packed)
    assert torch.equal(a, b) and torch.equal(a, c)
    with pytest.raises(AssertionError):
        sa.sparse_attention_func(qd, kd, vd, None, mask_packed=packed[..., :2])


def test_forward_can_be_captured_in_a_graph_and_replayed(sa, dev):
    """pack_mask + forward launch on the capturing stream, allocate only through PyTorch's allocator and
    never synchronise: a captured graph replays them; every replay is checked against an eager call."""
    q, k, v, mask = _inputs(2, 2, 192, torch.float16, 21)
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    sa.sparse_attention_func(qd, kd, vd, md)                 # warm-up outside the capture
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        sa.sparse_attention_func(qd, kd, vd, md)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_g = sa.sparse_attention_func(qd, kd, vd, md)
    for rep in range(3):
        g = torch.Generator().manual_seed(100 + rep)
        qd.copy_(torch.randn(q.shape, generator=g).to(torch.float16))
        md.copy_(torch.rand(mask.shape, generator=g) < 0.3)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        eager = sa.sparse_attention_func(qd, kd, vd, md)
        torch.cuda.synchronize()
        assert torch.equal(out_g, eager), f"replay {rep}"


def test_training_step_can_be_captured_in_a_graph_and_replayed(sa, dev):
    """Forward from the bool mask (packed words kept for the backward) and both backward kernels in
    one captured graph; the only allocations are PyTorch's.  Each replay, on new values in the same
    buffers and with eager work in between, must reproduce the eager step bit for bit."""
    q, k, v, mask = _inputs(2, 2, 160, torch.float16, 22)
    md = mask.to(dev)
    leaves = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(5)).to(torch.float16).to(dev)

    def step():
        out = sa.sparse_attention(*leaves, md)
        out.backward(dout)
        return out

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    for t in leaves:
        t.grad = None
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_g = step()
    grads_g = [t.grad for t in leaves]
    for rep in range(3):
        g = torch.Generator().manual_seed(200 + rep)
        with torch.no_grad():
            for t in leaves:
                t.copy_(torch.randn(q.shape, generator=g).to(torch.float16))
            md.copy_(torch.rand(mask.shape, generator=g) < 0.3)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = [out_g.clone()] + [x.clone() for x in grads_g]
        eager_leaves = [t.detach().clone().requires_grad_(True) for t in leaves]
        out_e = sa.sparse_attention(*eager_leaves, md)
        out_e.backward(dout)
        torch.cuda.synchronize()
        want = [out_e] + [t.grad for t in eager_leaves]
        for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
            assert torch.equal(a, b), f"replay {rep}: {name}"


@pytest.mark.parametrize("mshape", ["11", "B1", "BH"])
def test_views_of_a_fused_projection_and_shared_masks_through_autograd(sa, dev, mshape):
    """q, k, v as slices of one [B, N, 3, H, D] projection output (no copies are made), the mask
    shared between heads and/or batch entries; output and gradients against the oracle on the
    expanded mask.  The gradient arrives through a transpose, so dout is a strided view as well."""
    B, H, N = 2, 3, 136
    g = torch.Generator().manual_seed(21)
    qkv = torch.randn(B, N, 3, H, 64, generator=g).to(torch.float16)
    Bm, Hm = (1 if mshape[0] == "1" else B), (1 if mshape[1] == "1" else H)
    mask = torch.rand(Bm, Hm, N, N, generator=g) < 0.3
    mask[..., 5, :] = False
    leaf = qkv.to(dev).requires_grad_(True)
    q, k, v = (leaf[:, :, i].permute(0, 2, 1, 3) for i in range(3))          # [B, H, N, D] views
    assert sa._rows(q) is q and not q.is_contiguous()
    out = sa.sparse_attention(q, k, v, mask.to(dev))
    w = torch.randn(B, N, H, 64, generator=g).to(torch.float16)
    (out.permute(0, 2, 1, 3) * w.to(dev)).sum().backward()

    ref_leaf = qkv.float().requires_grad_(True)
    rq, rk, rv = (ref_leaf[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    ref = O.sparse_attention_ref(rq, rk, rv, mask.expand(B, H, N, N))
    (ref.permute(0, 2, 1, 3) * w.float()).sum().backward()
    assert torch.allclose(out.float().cpu(), ref.detach(), atol=1e-2, rtol=1e-2)
    assert (out[:, :, 5] == 0).all()
    bound = 1e-4 + 1e-2 * ref_leaf.grad.abs().max() + 2e-2 * ref_leaf.grad.abs()
    assert ((leaf.grad.float().cpu() - ref_leaf.grad).abs() <= bound).all()
    # the packed mask has the mask's own leading extents and can be reused
    packed = sa.pack_mask(mask.to(dev))
    assert packed.shape == (Bm, Hm, N, (N + 31) // 32)
    again = sa.sparse_attention_func(q.detach(), k.detach(), v.detach(), None, mask_packed=packed)
    assert torch.equal(again, out.detach())


def test_layouts_the_kernels_cannot_address_are_copied(sa, dev):
    """Odd strides (rows of 72 elements are fine, rows of 68 are not) and a transposed last dimension."""
    q, k, v, mask = _inputs(1, 2, 64, torch.float16, 8)
    md = mask.to(dev)
    want = sa.sparse_attention_func(q.to(dev), k.to(dev), v.to(dev), md)
    for pad in (72, 68):
        store = torch.zeros(1, 2, 64, pad, dtype=torch.float16, device=dev)
        store[..., :64] = q.to(dev)
        view = store[..., :64]
        assert (sa._rows(view) is view) == (pad == 72)
        assert torch.equal(sa.sparse_attention_func(view, k.to(dev), v.to(dev), md), want)
    qt = q.to(dev).transpose(2, 3).contiguous().transpose(2, 3)
    assert torch.equal(sa.sparse_attention_func(qt, k.to(dev), v.to(dev), md), want)


@pytest.mark.parametrize("shape", [(0, 2, 16), (2, 0, 16), (1, 1, 0)])
def test_empty_problems_are_no_ops(sa, dev, shape):
    """Zero batch entries, heads or sequence length: nothing is launched, shapes come back right,
    and autograd still returns (empty) gradients."""
    B, H, N = shape
    q, k, v = [torch.zeros(B, H, N, 64, dtype=torch.float16, device=dev, requires_grad=True) for _ in range(3)]
    mask = torch.zeros(B, H, N, N, dtype=torch.bool, device=dev)
    packed = sa.pack_mask(mask)
    assert packed.shape == (B, H, N, (N + 31) // 32) and packed.dtype == torch.int32
    out = sa.sparse_attention(q, k, v, mask)
    assert out.shape == (B, H, N, 64)
    out.sum().backward()
    assert q.grad.shape == q.shape and k.grad.shape == k.shape and v.grad.shape == v.shape
    assert sa.sparse_attention_func(q.detach(), k.detach(), v.detach(), mask).shape == (B, H, N, 64)
    torch.cuda.synchronize()


def test_backward_from_an_expanded_gradient(sa, dev):
    """out.sum().backward() hands the autograd function a gradient whose strides are all zero."""
    q, k, v, mask = _inputs(1, 2, 80, torch.float16, 12, keep=0.4)
    leaves = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    sa.sparse_attention(*leaves, mask.to(dev)).sum().backward()
    refs = [t.float().requires_grad_(True) for t in (q, k, v)]
    O.sparse_attention_ref(*refs, mask).sum().backward()
    for got, want in zip(leaves, refs):
        bound = 1e-4 + 1e-2 * want.grad.abs().max() + 1e-2 * want.grad.abs()
        assert ((got.grad.float().cpu() - want.grad).abs() <= bound).all()


def test_expanded_mask_is_packed_once(sa, dev, monkeypatch):
    """mask.expand(B, H, N, N) (zero strides) must reach the packer with the extents it really has."""
    B, H, N = 3, 4, 12                             # shorter than 16: the packing path
    q, k, v, _ = _inputs(B, H, N, torch.float16, 14)
    g = torch.Generator().manual_seed(15)
    small = (torch.rand(1, 1, N, N, generator=g) < 0.3).to(dev)
    seen = []
    real = sa.pack_mask
    monkeypatch.setattr(sa, "pack_mask", lambda m: (seen.append(tuple(m.shape)), real(m))[1])
    out = sa.sparse_attention_func(q.to(dev), k.to(dev), v.to(dev), small.expand(B, H, N, N))
    out_h = sa.sparse_attention_func(q.to(dev), k.to(dev), v.to(dev), small.expand(1, H, N, N).contiguous().expand(B, H, N, N))
    assert seen == [(1, 1, N, N), (1, H, N, N)]
    ref = O.sparse_attention_ref(q.float(), k.float(), v.float(), small.cpu().expand(B, H, N, N))
    assert torch.allclose(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    assert torch.equal(out, out_h)


def test_inference_entry_point_reads_the_bool_mask_itself(sa, dev, monkeypatch):
    """For shapes the single-launch kernel takes, sparse_attention_func must not pack the mask, and
    must return exactly what the packing path returns; other shapes still go through pack_mask."""
    calls = []
    real = sa.pack_mask
    monkeypatch.setattr(sa, "pack_mask", lambda m: (calls.append(tuple(m.shape)), real(m))[1])
    q, k, v, mask = _inputs(2, 3, 192, torch.float16, 16)
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    out = sa.sparse_attention_func(qd, kd, vd, md)
    assert calls == []
    assert torch.equal(out, sa.sparse_attention_func(qd, kd, vd, None, mask_packed=real(md)))
    assert torch.equal(out, sa.sparse_attention(qd, kd, vd, md))            # nothing requires grad: same path
    assert calls == []
    leaves = [t.clone().requires_grad_(True) for t in (qd, kd, vd)]
    tracked = sa.sparse_attention(*leaves, md)       # autograd: same launch, which also leaves lse and the packed words
    assert torch.equal(out, tracked) and calls == []
    tracked.sum().backward()                          # ... for the backward, which therefore needs no packing pass either
    assert calls == [] and all(t.grad is not None for t in leaves)
    with torch.no_grad():
        assert torch.equal(out, sa.sparse_attention(*leaves, md))
    shared = sa.sparse_attention_func(qd, kd, vd, md[:1, :1].expand(2, 3, 192, 192))      # expanded view: read once
    assert calls == []
    ref = O.sparse_attention_ref(q.float(), k.float(), v.float(), mask[:1, :1].expand(2, 3, 192, 192))
    assert torch.allclose(shared.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    calls.clear()
    q, k, v, mask = _inputs(1, 2, 101, torch.float16, 17)                                   # rows at odd addresses
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    odd = sa.sparse_attention_func(qd, kd, vd, md)
    assert calls == [] and torch.equal(odd, sa.sparse_attention_func(qd, kd, vd, None, mask_packed=real(md)))
    calls.clear()
    q, k, v, mask = _inputs(1, 2, 12, torch.float16, 17)                                    # N < 16
    sa.sparse_attention_func(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    assert calls == [(1, 2, 12, 12)]
    # fp32 inputs: computed in bf16 through the same path, returned as fp32
    q, k, v, mask = _inputs(1, 2, 128, torch.float32, 18)
    o32 = sa.sparse_attention_func(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    assert o32.dtype == torch.float32
    ref = O.sparse_attention_ref(q.bfloat16().float(), k.bfloat16().float(), v.bfloat16().float(), mask)
    assert torch.allclose(o32.cpu(), ref, atol=1e-2, rtol=2e-2)


def test_autograd_from_a_bool_mask_with_empty_blocks_uses_the_map_and_changes_nothing(sa, dev):
    """With a bool mask the one-launch forward hands the backward the packed words and, when the caller
    says `tile_map=True`, the tile map; either way the gradients are those of the path that packs
    first and walks every tile, bit for bit."""
    g = torch.Generator().manual_seed(21)
    B, H, N = 2, 3, 320
    blocks = torch.rand(B, H, 5, 5, generator=g) < 0.3
    mask = (blocks.repeat_interleave(64, 2).repeat_interleave(64, 3) & (torch.rand(B, H, N, N, generator=g) < 0.5))
    q, k, v, do = (torch.randn(B, H, N, 64, generator=g).half().to(dev) for _ in range(4))
    md = mask.to(dev)
    grads = []
    for kw in ({}, {"tile_map": True}, {"mask_packed": sa.pack_mask(md)}):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = sa.sparse_attention(*leaves, None if "mask_packed" in kw else md, **kw)
        out.backward(do)
        grads.append([out.detach()] + [t.grad for t in leaves])
    for other in grads[1:]:
        for a, b in zip(grads[0], other):
            assert torch.equal(a, b)
    # tile_map=True really hands a map to the backward, the default hands none
    for kw, has_map in (({}, False), ({"tile_map": True}, True)):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = sa.sparse_attention(*leaves, md, **kw)
        node = out.grad_fn                  # the slice back to D columns sits on top of the function's node
        while node is not None and not hasattr(node, "tile_map"):
            node = node.next_functions[0][0] if node.next_functions else None
        assert node is not None and (node.tile_map is not None) == has_map
    wanted = O.sparse_attention_bwd_ref(q.float().cpu(), k.float().cpu(), v.float().cpu(), mask, do.float().cpu())
    for got, want in zip(grads[0][1:], wanted):
        assert torch.allclose(got.float().cpu(), want, atol=1e-4 + 1e-2 * want.abs().max().item(), rtol=1e-2)


def test_mfma_stream_probe_runs_and_reports_a_clock(dev):
    """The benchmark's yardstick kernel: finishes, and the two tick counts it leaves give a shader
    clock that a GPU of this kind can have."""
    import _capi
    lib = _capi.load_probe()
    groups = 8
    stamps = torch.zeros(2 * groups, dtype=torch.int64, device=dev)
    for stream, random_operands in ((lib.sma_probe_mfma_stream, 0), (lib.sma_probe_mfma_stream, 1), (lib.sma_probe_mfma_stream_32x32x16, 1)):
        assert stream(random_operands, 2000, groups, stamps.data_ptr(), None) == 0
        torch.cuda.synchronize()
        st = stamps.view(groups, 2).double().cpu()
        assert (st > 0).all()
        ghz = (st[:, 0] / (st[:, 1] * 10.0)).mean().item()
        assert 0.3 < ghz < 3.0, ghz
    assert lib.sma_probe_mfma_stream(1, 10, 0, None, None) == 0
    assert lib.sma_probe_mfma_stream(1, 10, 4, None, None) == -1          # stamps missing
    assert lib.sma_probe_mfma_stream(1, (1 << 22) + 1, 4, stamps.data_ptr(), None) == -2     # iteration cap
    assert not hasattr(_capi.load(), "sma_probe_mfma_stream")             # not part of the product library


def test_command_line_harness_acceptance_run_and_sweeps(dev, capsys):
    """run.py: the reference's acceptance run (run.py:349-404 there) passes, and the sweep tables
    print a row for every size with a latency above zero."""
    import importlib
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparse-mask-attention_amd")
    if pkg not in sys.path:
        sys.path.insert(0, pkg)
    run = importlib.import_module("run")
    assert run.run_correctness(dev) is True
    text = capsys.readouterr().out
    assert text.count("[PASS]") == 5 and "FAIL" not in text
    run.run_perf(dev)
    rows = [line.split() for line in capsys.readouterr().out.splitlines() if line.strip()[:1].isdigit()]
    assert [int(r[0]) for r in rows] == [64, 128, 256, 512, 1024, 1, 4, 8, 16, 32, 64]
    assert all(float(r[1]) > 0 and float(r[2]) > 0 for r in rows)
