"""What a call promises beyond its numbers: autograd notices what it must, checks are made before anything is
launched, and limits lie where the documentation puts them."""
import importlib
import sys
import threading

import pytest
import torch
import torch.autograd.forward_ad as fwd_ad

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sa():
    importlib.import_module("python.sparse_attention")
    return sys.modules["python.sparse_attention"]


def _problem(dev, N=70, D=64, dtype=torch.float16, seed=0):
    g = torch.Generator().manual_seed(seed)
    q, k, v, do = (torch.randn(2, 2, N, D, generator=g).to(dtype).to(dev) for _ in range(4))
    return q, k, v, do, (torch.rand(2, 2, N, N, generator=g) < 0.4).to(dev)


@pytest.mark.parametrize("D", [60, 64, 80])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_an_output_changed_in_place_is_noticed(sa, dev, D, dtype):
    """The backward needs the output as it was.  D = 60 is the narrowed part of a padded result."""
    q, k, v, do, mask = _problem(dev, D=D, dtype=dtype)

    def through(change):
        leaf = q.clone().requires_grad_(True)
        out = sa.sparse_attention(leaf, k, v, mask)
        changed = change(out)
        (changed if changed is not None else out).backward(do)
        return leaf.grad

    def unseen(out):
        with torch.no_grad():
            out.add_(1.0)

    def one_row(out):
        out[:, :, 0].zero_()

    for change in (lambda o: o.mul_(2.0), lambda o: o.add_(do), unseen, one_row):
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            through(change)
    assert torch.equal(through(lambda o: o * 2.0), through(lambda o: o.float().mul_(2.0).to(dtype)))


@pytest.mark.parametrize("D", [60, 64])
def test_an_fp32_output_may_be_changed_in_place(sa, dev, D):
    """It is a copy of what the backward keeps."""
    q, k, v, do, mask = _problem(dev, D=D, dtype=torch.float32)
    got = []
    for change in (lambda o: o * 2.0, lambda o: o.mul_(2.0)):
        leaf = q.clone().requires_grad_(True)
        change(sa.sparse_attention(leaf, k, v, mask)).backward(do)
        got.append(leaf.grad)
    assert torch.equal(*got)


def test_the_function_behind_the_api_refuses_what_it_cannot_address(sa, dev):
    """SparseAttentionFunction.apply makes the checks of sparse_attention, before anything is launched: the kernels
    address every tensor by q's extents."""
    q, k, v, do, mask = _problem(dev)
    packed = sa.pack_mask(mask)
    tm = sa.sparse_attn_cuda.tile_map(packed)
    N = q.shape[2]

    def call(q=q, k=k, v=v, packed=None, mask=mask, tile_map=None):
        return sa.SparseAttentionFunction.apply(q, k, v, packed, mask, 0.125, N, tile_map)

    wrong = [dict(mask=None)]
    wrong += [dict(mask=m) for m in (mask[:, :, :, :-1], mask[:, :, :-1], mask[:, :, :64, :64], mask[:1].expand(3, 2, N, N), mask[0],
                                     mask[:, :1].expand(2, 4, N, N), mask.to(torch.uint8), mask.half(), mask.cpu())]
    wrong += [dict(packed=p) for p in (packed[:, :, :-1], packed[..., :-1], packed[0], packed.float(), packed.long(), packed.cpu(),
                                       packed.expand(2, 2, N, 3).transpose(2, 3).contiguous().transpose(2, 3),
                                       packed[:1].expand(3, 2, N, 3))]
    wrong += [dict(q=t(q), k=t(k), v=t(v)) for t in (torch.Tensor.double, torch.Tensor.int, torch.Tensor.cpu,
                                                     lambda x: x[0], lambda x: torch.cat([x, x, x], -1))]
    wrong += [{name: t(x)} for name, x in (("k", k), ("v", v))
              for t in (torch.Tensor.float, torch.Tensor.bfloat16, torch.Tensor.cpu, lambda x: x[:, :, :-1], lambda x: x[..., :32])]
    wrong += [dict(q=q.float(), k=k.float()), dict(q=q.float(), v=v.float()), dict(q=q.float(), k=k.float(), v=v.double())]
    wrong += [dict(packed=packed, tile_map=t) for t in (True, tm[:, :, :1], tm.cpu(), tm.float(), 3)]
    for args in wrong:
        with pytest.raises(RuntimeError):
            call(**args)
    want = sa.sparse_attention_func(q, k, v, mask)
    for args in ({}, dict(mask=mask, tile_map=True), dict(mask=None, packed=packed), dict(mask=None, packed=packed, tile_map=tm)):
        assert torch.equal(call(**args), want)
    wide = [t.float() for t in (q, k, v)]
    assert torch.equal(call(*wide), sa.sparse_attention_func(*wide, mask))


def test_a_shared_mask_longer_than_a_tile_map_allows(sa, dev):
    """N > 131072, one mask for four heads: packed without a map.  Every row keeps three keys, one of them the last."""
    N, D = 131136, 32
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(1, 4, N, D, generator=g).half().to(dev) for _ in range(3))
    mask = torch.eye(N, dtype=torch.bool, device=dev)[None, None]
    mask[..., 5] = True
    mask[..., N - 1] = True
    leaf = q.clone().requires_grad_(True)
    out = sa.sparse_attention_func(q, k, v, mask)
    assert torch.equal(out, sa.sparse_attention(leaf, k, v, mask).detach())
    keys = torch.stack([torch.full((N,), 5, device=dev), torch.full((N,), N - 1, device=dev), torch.arange(N, device=dev)], 1)
    s = (q.float()[:, :, :, None] * k.float()[:, :, keys]).sum(-1) * D ** -0.5                  # [1, 4, N, 3]
    s[:, :, 5, 2] = s[:, :, N - 1, 2] = -float("inf")                                           # the same key a second time
    want = (torch.softmax(s, -1)[..., None] * v.float()[:, :, keys]).sum(-2)
    # weights (rounded toward zero, numerator and denominator alike) and output of 11 bits
    assert torch.allclose(out.float(), want, atol=1e-2, rtol=1e-2)


def test_fp32_rows_further_apart_than_the_kernels_store_them(sa, dev):
    """[B, N, H, D] with H * D = 131072: the slab of a head passes 2^31 bytes in fp32, not in the 16 bits that the
    kernels compute in.  The same heads in a tensor of their own are stored as fp32 by the kernels: the same bits."""
    N, H, D = 4100, 1024, 128
    g = torch.Generator(device=dev).manual_seed(4)
    q, k, v, do = (torch.randn(1, N, H, D, device=dev, generator=g).transpose(1, 2) for _ in range(4))
    assert (N - 1) * H * D * 4 + 4 * D >= 2 ** 31 > (N - 1) * H * D * 2 + 2 * D
    mask = torch.rand(1, 1, N, N, device=dev, generator=g) < 0.3
    mask[..., 64:] &= torch.rand(N, 1, device=dev, generator=g) < 0.01          # few tiles with anything in them
    mask |= torch.eye(N, dtype=torch.bool, device=dev)

    def run(heads):
        few = heads < H
        leaves = [(t[:, :heads].contiguous() if few else t).detach().requires_grad_(True) for t in (q, k, v)]
        out = sa.sparse_attention(*leaves, mask)
        with torch.no_grad():
            assert torch.equal(out, sa.sparse_attention(*leaves, mask))
        assert out.dtype == torch.float32 and out.stride() == leaves[0].stride()
        return [out.detach()] + list(torch.autograd.grad(out, leaves, do[:, :heads].contiguous() if few else do))

    wide, few = run(H), run(256)
    for name, a, b in zip(("out", "dq", "dk", "dv"), wide, few):
        assert a.dtype == torch.float32 and torch.equal(a[:, :256], b), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_a_tangent_is_refused_and_not_dropped(sa, dev, dtype):
    q, k, v, do, mask = _problem(dev, dtype=dtype)
    for which in range(3):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        with fwd_ad.dual_level():
            leaves[which] = fwd_ad.make_dual(leaves[which], torch.ones_like(q))
            with pytest.raises(NotImplementedError, match="forward mode"):
                sa.sparse_attention(*leaves, mask)
            if dtype == torch.float16:
                plain = [t.detach() for t in (q, k, v)]
                plain[which] = fwd_ad.make_dual(plain[which], torch.ones_like(q))
                for tensors in (leaves, plain):
                    with pytest.raises(NotImplementedError, match="forward mode"):
                        sa.SparseAttentionFunction.apply(*tensors, None, mask, 0.125, q.shape[2])
        assert torch.equal(sa.sparse_attention(*leaves, mask), sa.sparse_attention_func(q, k, v, mask))      # the level is over


@pytest.mark.parametrize("D", [60, 64])
def test_the_node_shows_what_it_saved(sa, dev, D):
    """grad_fn.saved_tensors: q, k, v, out, lse and the packed mask, until the backward has freed them."""
    q, k, v, do, mask = _problem(dev, D=D)
    leaf = q.clone().requires_grad_(True)
    out = sa.sparse_attention(leaf, k, v, mask)
    for _ in range(2):
        saved = out.grad_fn.saved_tensors
        assert len(saved) == 6
        for a, b in zip(saved, (q, k, v, out.detach())):
            assert torch.equal(a[..., :D], b) and not a[..., D:].any()
        s = (q.float() @ k.float().transpose(-1, -2) * D ** -0.5).masked_fill(~mask, -float("inf"))
        assert torch.allclose(saved[4], torch.logsumexp(s, -1), atol=2e-3)
        assert torch.equal(saved[5], sa.pack_mask(mask))
        out.backward(do, retain_graph=True)
    if D == 64:
        assert saved[0] is leaf and saved[3].grad_fn is out.grad_fn
    out.backward(do)
    with pytest.raises(RuntimeError, match="freed"):
        out.grad_fn.saved_tensors
    # through hooks, and from inside of one that the backward calls
    seen = []

    def unpack(t):
        seen.append(t)
        if len(seen) == 7:
            assert len(out.grad_fn.saved_tensors) == 6
        return t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.clone(), unpack):
        out = sa.sparse_attention(leaf, k, v, mask)
    assert len(out.grad_fn.saved_tensors) == 6 and len(seen) == 6
    out.backward(do)
    assert len(seen) == 18


@pytest.mark.parametrize("D", [60, 64])
def test_what_saved_tensor_hooks_give_back_is_checked(sa, dev, D):
    """The backward addresses what it saved by the gradient's extents: hooks that change device, type or shape are an
    error, as they were for a function written in Python; hooks that give back an equal tensor are fine."""
    q, k, v, do, mask = _problem(dev, D=D)

    def grads(which, change):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        count = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (len(count), count.append(0), t.detach().clone())[::2],
                                                      lambda p: change(p[1]) if p[0] == which else p[1]):
            out = sa.sparse_attention(*leaves, mask)
        assert len(count) == 6
        return torch.autograd.grad(out, leaves, do)

    want = grads(-1, None)
    for which in range(6):
        for a, b in zip(want, grads(which, lambda t: t.cpu().to(dev))):
            assert torch.equal(a, b)
        for change in (torch.Tensor.cpu, torch.Tensor.double, lambda t: t[:, :, :-1], lambda t: t[:0], lambda t: t[0],
                       lambda t: t[..., :-8] if t.size(-1) > 8 else t[..., :-1]):
            with pytest.raises(RuntimeError):
                grads(which, change)


@pytest.mark.parametrize("D", [60, 64, 80])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gradients_leave_no_gaps(sa, dev, D, dtype):
    """Gradients of contiguous tensors are contiguous, also where the kernels compute with padded rows."""
    q, k, v, do, mask = _problem(dev, D=D, dtype=dtype)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    for g in torch.autograd.grad(sa.sparse_attention(*leaves, mask), leaves, do):
        assert g.is_contiguous() and g.view(-1).numel() == q.numel()


@pytest.mark.parametrize("D", [60, 64])
@pytest.mark.parametrize("entry", ["sparse_attention", "sparse_attention_func", "apply", "packed"])
@pytest.mark.filterwarnings("ignore:.*torch.jit.*:DeprecationWarning")
def test_a_trace_records_the_call(sa, dev, D, entry):
    """torch.jit.trace: the call is an operation of the trace, computed anew from the inputs and masks of each run."""

    class Model(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.weight = torch.nn.Parameter(torch.linspace(0.5, 1.5, D).half())

        def forward(self, x, k, v, mask):
            q = x * self.weight
            if entry == "apply":
                return sa.SparseAttentionFunction.apply(q, k, v, None, mask, 0.125, x.shape[2]) * 2
            if entry == "packed":
                return sa.sparse_attention(q, k, v, None, mask) * 2
            return getattr(sa, entry)(q, k, v, mask) * 2

    model = Model().to(dev)
    inputs = []
    for seed in (1, 2):
        q, k, v, do, mask = _problem(dev, D=D, seed=seed)
        inputs.append((q, k, v, sa.pack_mask(mask) if entry == "packed" else mask))
    for tracked in (True, False):
        with torch.set_grad_enabled(tracked and entry != "sparse_attention_func"):
            traced = torch.jit.trace(model, inputs[0], check_trace=False)
            for args in reversed(inputs):
                got, want = traced(*args), model(*args)
                assert torch.equal(got, want)
                if want.requires_grad:
                    a, b = (torch.autograd.grad(o, model.weight, do)[0] for o in (got, want))
                    assert torch.equal(a, b)
    with pytest.raises(AssertionError):
        torch.jit.trace(lambda x, m: sa.sparse_attention(x, x, x, m), (q, mask[..., :-1]), check_trace=False)


def test_a_long_chain_of_calls_is_freed(sa, dev):
    """Each call's query is the output of the one before: the graph is one node after the other.  Freed by recursion,
    20000 of them take more than the 256 KiB of stack that they are freed on here."""
    q = torch.randn(1, 1, 16, 32, device=dev, dtype=torch.float16)
    mask = torch.ones(1, 1, 16, 16, dtype=torch.bool, device=dev)
    leaf = q.clone().requires_grad_(True)
    chain = [leaf]
    for _ in range(20000):
        chain[0] = sa.sparse_attention(chain[0], q, q, mask)
    before = threading.stack_size(256 * 1024)
    try:
        thread = threading.Thread(target=chain.clear)
        thread.start()
    finally:
        threading.stack_size(before)
    thread.join()
    assert torch.equal(sa.sparse_attention(leaf, q, q, mask), sa.sparse_attention_func(q, q, q, mask))
