"""What a call promises beyond its numbers: autograd notices what it must, checks are made before anything is
launched, and limits lie where the documentation puts them."""
import importlib
import sys

import pytest
import torch

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
