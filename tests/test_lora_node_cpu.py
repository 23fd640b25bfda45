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


class Base(torch.nn.Module):
    """An fp32 base product that autocast does not reach, as the packed ones."""
    in_features, out_features = 24, 12

    def __init__(self):
        super().__init__()
        self.register_buffer("w", torch.randn(12, 24, generator=torch.Generator().manual_seed(2)))

    def forward(self, x):
        with torch.autocast(x.device.type, enabled=False):
            return x @ self.w.t()


def layer(monkeypatch, dropout=0.0):
    """A LoRALinear that takes CPU tensors for eager GPU ones."""
    monkeypatch.setattr(lora.ops, "_eager", lambda *ts: True)
    lay = lora.LoRALinear(rank=3, alpha=2.0, base_module=Base(), dropout=dropout)
    with torch.no_grad():
        lay.lora_b.copy_(torch.randn(12, 3, generator=torch.Generator().manual_seed(3)))
    return lay


def composed(lay, x):
    z = x @ lay.lora_a.to(x.dtype).t()
    if lay.dropout is not None:
        z = lay.dropout(z)
    return lay.linear(x) + lay.scale * (z @ lay.lora_b.to(x.dtype).t())


def run(lay, f):
    x = torch.randn(4, 5, 24, generator=torch.Generator().manual_seed(4)).requires_grad_(True)
    y = f(x)
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(5)).to(y.dtype)
    return lambda: (y, *torch.autograd.grad(y, [x, lay.lora_a, lay.lora_b], dy))


def test_the_node_runs_and_matches(monkeypatch):
    lay = layer(monkeypatch)
    x = torch.randn(4, 24, requires_grad=True)
    assert "LowRankFunction" in type(lay(x).grad_fn.next_functions[0][0]).__name__
    for p, q in zip(run(lay, lay)(), run(lay, lambda t: composed(lay, t))()):
        torch.testing.assert_close(p, q)


@pytest.mark.parametrize("backward_inside", [False, True])
def test_autocast_keeps_the_base_product(monkeypatch, backward_inside):
    """The term's products run in bf16, the fp32 base product is not rounded, and
    the backward runs: the composed form's dtypes and values."""
    lay = layer(monkeypatch)
    out = []
    for f in (lay, lambda t: composed(lay, t)):
        with torch.autocast("cpu", torch.bfloat16):
            grads = run(lay, f)
            if backward_inside:
                out.append(grads())
        if not backward_inside:
            out.append(grads())
    for p, q in zip(*out):
        assert p.dtype == q.dtype
        torch.testing.assert_close(p, q)


@pytest.mark.parametrize("training,dropping", [(True, True), (True, False), (False, True), (False, False)])
def test_dropout_follows_its_own_module(monkeypatch, training, dropping):
    """A dropout module switched by itself (sampling over masks at inference)."""
    lay = layer(monkeypatch, dropout=0.5).train(training)
    lay.dropout.train(dropping)
    out = []
    for f in (lay, lambda t: composed(lay, t)):
        torch.manual_seed(0)
        out.append(run(lay, f)())
    for p, q in zip(*out):
        torch.testing.assert_close(p, q)


def test_adapters_stepped_before_the_backward(monkeypatch):
    """bf16 adapters under fp32 activations: an update in place between forward and
    backward leaves the gradients those of the forward's adapters."""
    lay = layer(monkeypatch)
    assert lay.lora_a.dtype == torch.bfloat16
    want = run(lay, lambda t: composed(lay, t))()
    grads = run(lay, lay)
    with torch.no_grad():
        lay.lora_a.mul_(2.0)
        lay.lora_b.add_(1.0)
    for p, q in zip(grads(), want):
        torch.testing.assert_close(p, q)
