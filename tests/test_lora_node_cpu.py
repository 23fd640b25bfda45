"""The low-rank term over an unfused base as one autograd node
(lora._LowRankFunction) against the composed form, on the CPU."""
import pytest
import torch

from rwkvq import lora


@pytest.fixture
def poisoned(monkeypatch):
    """Memory that new_empty hands out holds NaN."""
    new_empty = torch.Tensor.new_empty
    monkeypatch.setattr(torch.Tensor, "new_empty",
                        lambda t, *a, **k: new_empty(t, *a, **k).fill_(float("nan")))


def term(x, base, a, b, scale):
    return base + scale * ((x @ a.to(x.dtype).t()) @ b.to(x.dtype).t())


def operands(m=5, K=24, R=12, rank=3):
    g = torch.Generator().manual_seed(0)
    t = lambda *s: torch.randn(*s, generator=g).requires_grad_(True)  # noqa: E731
    return t(m, K), t(m, R), t(rank, K), t(R, rank)


@pytest.mark.parametrize("wrt", [(0, 1, 2, 3), (2, 3), (2,), (3,), (0,)])
def test_vmapped_backward(poisoned, wrt):
    """The vector-Jacobian products of many incoming gradients at once."""
    ops_ = operands()
    dys = torch.randn(7, 5, 12, generator=torch.Generator().manual_seed(1))
    got, want = [], []
    for f, out in ((lora._LowRankFunction.apply, got), (term, want)):
        y = f(*ops_, 0.7)
        out += torch.vmap(lambda d: torch.autograd.grad(y, [ops_[i] for i in wrt], d, retain_graph=True))(dys)
        out += torch.autograd.grad(y, [ops_[i] for i in wrt], dys, is_grads_batched=True, retain_graph=True)
        out += torch.autograd.grad(y, [ops_[i] for i in wrt], dys[0])
    for p, q in zip(got, want):
        torch.testing.assert_close(p, q)  # fp32, sums of at most 24 products
