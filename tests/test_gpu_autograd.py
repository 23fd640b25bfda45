"""quantized_matmul's eager autograd against the registered op's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xdt,sdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                     (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("transpose", [True, False])
def test_eager_autograd_equals_registered_op(rq, dev, transpose, xdt, sdt):
    g = torch.Generator().manual_seed(3)
    R, K, M = 192, 512, 20
    wq, s, b = rq.quantize((torch.randn(R, K, generator=g) * 0.02).to(sdt).to(dev), 64, 4)
    n_in, n_out = (K, R) if transpose else (R, K)
    x = torch.randn(2, M, n_in, generator=g).to(xdt).to(dev)
    dy = torch.randn(2, M, n_out, generator=g).to(dev)
    out = []
    for f in (rq.quantized_matmul, torch.ops.rwkvq.quantized_matmul):
        xg = x.clone().requires_grad_(True)
        y = f(xg, wq, s, b, transpose, 64, 4)
        (dx,) = torch.autograd.grad(y, xg, dy.to(y.dtype))
        out.append((y.detach(), dx))
    assert out[0][1].dtype == xdt
    for a, c in zip(*out):
        assert a.dtype == c.dtype and torch.equal(a, c)
    assert torch.is_grad_enabled() and rq.quantized_matmul(x, wq, s, b, transpose, 64, 4).grad_fn is None


def test_eager_autograd_second_order_and_hooks(rq, dev):
    """A gradient of a gradient, saved-tensor hooks (the words, scales and biases
    are saved, nothing of x) and a non-contiguous incoming gradient."""
    g = torch.Generator().manual_seed(4)
    wq, s, b = rq.quantize((torch.randn(128, 256, generator=g) * 0.02).to(dev), 64, 4)
    x = torch.randn(7, 256, generator=g).to(dev).requires_grad_(True)
    dy = torch.randn(128, 7, generator=g).to(dev).t().requires_grad_(True)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t), t)[1], lambda t: t):
        y = rq.quantized_matmul(x, wq, s, b, True, 64, 4)
    assert [tuple(t.shape) for t in seen] == [tuple(t.shape) for t in (wq, s, b)]
    (dx,) = torch.autograd.grad(y, x, dy, create_graph=True)
    v = torch.randn(7, 256, generator=g).to(dev)
    (ddy,) = torch.autograd.grad(dx, dy, v)
    assert torch.equal(ddy, rq.quantized_matmul(v, wq, s, b, True, 64, 4))
    assert torch.equal(dx.detach(), rq.quantized_matmul(dy.detach().contiguous(), wq, s, b, False, 64, 4))


@pytest.mark.parametrize("backend", ["native", "hybrid", "dense"])
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
def test_low_rank_term_over_sb6(rq, dev, xdt, backend):
    """LoRALinear over an sb6 base: y and the gradients against the composed form
    in float64 (bf16: 2^-8 per rounding of y, z and dz), and a second derivative
    against autograd of the composed form."""
    import sb6_k3
    R, K, r = 256, 512, 16
    arrays = sb6_k3.random_sb6(R, K, 1, 8, 5)
    lin = rq.RwkvqLinear(*(t.to(dev) for t in sb6_k3.encode(*arrays, 1)), (R, K), 32, 8, 1)
    base = {"native": rq.RwkvqNativeLinear, "hybrid": rq.RwkvqHybridLinear, "dense": lambda b: b}[backend](lin)
    lay = rq.LoRALinear(rank=r, alpha=32.0, base_module=base)
    g = torch.Generator().manual_seed(1)
    with torch.no_grad():
        lay.lora_b.copy_(torch.randn(R, r, generator=g) * 0.05)
    x = torch.randn(3, 40, K, generator=g).to(xdt).to(dev).requires_grad_(True)
    dy = torch.randn(3, 40, R, generator=g).to(xdt).to(dev)
    y = lay(x)
    got = torch.autograd.grad(y, [x, lay.lora_a, lay.lora_b], dy)
    w = lin._dequant_w_fp32().double()
    xd, a, b = (t.detach().double().requires_grad_(True) for t in (x, lay.lora_a, lay.lora_b))
    ref = xd @ w.t() + lay.scale * ((xd @ a.t()) @ b.t())
    want = torch.autograd.grad(ref, [xd, a, b], dy.double())
    tol = 1e-2   # the base's bf16 weights, bf16 gradients; bf16 x: z, dz and y too
    for p, q in zip((y, *got), (ref, *want)):
        assert p.shape == q.shape and (p.double() - q).norm() <= tol * q.norm()
    if xdt == torch.float32 and backend == "native":
        def second(lay_fn):
            (gb,) = torch.autograd.grad(lay_fn(x), lay.lora_b, dy, create_graph=True)
            return torch.autograd.grad(gb.float().square().sum(), [x, lay.lora_a])
        def composed(t):
            z = t @ lay.lora_a.float().t()
            return base(t) + lay.scale * (z @ lay.lora_b.float().t())
        for p, q in zip(second(lay), second(composed)):
            assert (p.float() - q.float()).norm() <= 1e-2 * q.float().norm()


def sb6_layer(rq, dev, R, K, r, backend="native", dropout=0.0):
    import sb6_k3
    arrays = sb6_k3.random_sb6(R, K, 1, 8, 5)
    lin = rq.RwkvqLinear(*(t.to(dev) for t in sb6_k3.encode(*arrays, 1)), (R, K), 32, 8, 1)
    base = {"native": rq.RwkvqNativeLinear, "hybrid": rq.RwkvqHybridLinear}[backend](lin)
    lay = rq.LoRALinear(rank=r, alpha=32.0, base_module=base, dropout=dropout)
    with torch.no_grad():
        lay.lora_b.copy_(torch.randn(R, r, generator=torch.Generator().manual_seed(1)) * 0.05)
    return lay, base


def composed(lay, base, x):
    """LoRALinear's term as separate ops."""
    z = x @ lay.lora_a.to(x.dtype).t()
    return base(x) + lay.scale * (z @ lay.lora_b.to(x.dtype).t())


def test_low_rank_term_vmapped_backward(rq, dev, monkeypatch):
    """Many incoming gradients at once, where memory that new_empty hands out holds
    NaN.  bf16 adapters: their gradients round to bf16 (2^-8 between neighbours)."""
    lay, base = sb6_layer(rq, dev, 256, 512, 16)
    g = torch.Generator().manual_seed(2)
    x, dys = torch.randn(6, 512, generator=g).to(dev), torch.randn(3, 6, 256, generator=g).to(dev)
    new_empty = torch.Tensor.new_empty
    monkeypatch.setattr(torch.Tensor, "new_empty", lambda t, *a, **k: new_empty(t, *a, **k).fill_(float("nan")))
    out = []
    for y in (lay(x), composed(lay, base, x)):
        out.append(torch.vmap(lambda d: torch.autograd.grad(y, (lay.lora_a, lay.lora_b), d, retain_graph=True))(dys))
    for p, q in zip(*out):
        assert p.shape == q.shape and (p.float() - q.float()).norm() <= 2.0 ** -8 * q.float().norm()


@pytest.mark.parametrize("kind", ["native", "hybrid", "rank8"])
def test_low_rank_term_under_autocast(rq, dev, kind):
    """fp32 y, its base product not rounded, and gradients: the composed form's."""
    R, K = 256, 512
    if kind == "rank8":   # a QuantizedLinear whose term is not fused
        base = rq.QuantizedLinear.from_linear(torch.nn.Linear(K, R, bias=False, device=dev).bfloat16(), 64, 4)
        lay = rq.LoRALinear(rank=8, alpha=32.0, base_module=base)
        with torch.no_grad():
            lay.lora_b.copy_(torch.randn(R, 8, generator=torch.Generator().manual_seed(1)) * 0.05)
    else:
        lay, base = sb6_layer(rq, dev, R, K, 16, kind)
    g = torch.Generator().manual_seed(2)
    x = torch.randn(3, 20, K, generator=g).to(dev).requires_grad_(True)
    dy = torch.randn(3, 20, R, generator=g).to(dev)
    out = []
    for f in (lay, lambda t: composed(lay, base, t)):
        with torch.autocast("cuda", torch.bfloat16):
            y = f(x)
        assert y.dtype == torch.float32
        out.append((y, *torch.autograd.grad(y, [x, lay.lora_a, lay.lora_b], dy)))
    for p, q in zip(*out):
        assert p.dtype == q.dtype
        torch.testing.assert_close(p, q)


@pytest.mark.parametrize("requires_grad", [True, False])
def test_jit_trace_records_the_registered_op(rq, dev, tmp_path, requires_grad):
    """A trace holds the op, not this call's result or a Python function: it runs
    on other inputs and can be saved."""
    g = torch.Generator().manual_seed(6)
    wq, s, b = rq.quantize((torch.randn(64, 128, generator=g) * 0.02).bfloat16().to(dev), 32, 4)
    x, x2 = (torch.randn(20, 128, generator=g).bfloat16().to(dev).requires_grad_(requires_grad) for _ in range(2))
    f = torch.jit.trace(lambda t: rq.quantized_matmul(t, wq, s, b, True, 32, 4), x, check_trace=False)
    f.save(str(tmp_path / "f.pt"))
    want = rq.quantized_matmul(x2, wq, s, b, True, 32, 4)
    assert torch.equal(f(x2), want) and torch.equal(torch.jit.load(str(tmp_path / "f.pt"))(x2), want)
