"""fp32 activations rounded to bf16 by a pass of their own before the large
GEMMs (ops._round_first) against the GEMMs that round them as they stage them:
the same bits on the 64-wide-stage kernels (the same tiles and sums), fp32 sums
in another order on the 256-row tiles of the other widths."""
import pytest
import torch

import rwkvq
from rwkvq import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,rows,cols,transpose,gs,bits,sdt", [
    (1528, 2560, 2560, True, 64, 4, torch.bfloat16),   # just past 1e10 multiply-adds
    (1001, 4224, 2560, True, 32, 3, torch.bfloat16),   # odd rows of x, a partial column tile
    (513, 8192, 2560, True, 64, 8, torch.float16),
    (3577, 2048, 8192, True, 64, 4, torch.bfloat16),   # split contraction's shape
    (256, 1536, 768, False, 64, 4, torch.bfloat16),    # the smallest transposed one
    (1003, 2048, 2048, False, 64, 6, torch.float16),
    (700, 2560, 768, True, 64, 4, torch.bfloat16),     # 12 groups: no 64-wide stages
])
def test_rounded_first_matches_staged(monkeypatch, m, rows, cols, transpose, gs, bits, sdt):
    g = torch.Generator(device="cuda").manual_seed(m)
    w = (torch.randn(rows, cols, generator=g, device="cuda") * 0.02).to(sdt)
    q = rwkvq.quantize(w, gs, bits)
    n_in = cols if transpose else rows
    x = torch.randn(m, n_in, generator=g, device="cuda")
    x[0, 0], x[m - 1, n_in - 1], x[1, 1] = float("inf"), float("nan"), 3.4e38
    assert ops._round_first(m, q[0], sdt, transpose, gs, bits)
    strided = torch.empty(n_in, m, device="cuda").t().copy_(x)
    offset = torch.empty(m * n_in + 1, device="cuda")[1:].view(m, n_in).copy_(x)
    ys = [rwkvq.quantized_matmul(t, *q, transpose, gs, bits) for t in (x, strided, offset)]
    monkeypatch.setattr(ops, "_round_first", lambda *a: False)
    want = rwkvq.quantized_matmul(x, *q, transpose, gs, bits)
    assert want.dtype == torch.float32
    k64 = not transpose or (cols // gs) % 8 == 0
    for y in ys:
        assert y.dtype == torch.float32 and y.shape == want.shape
        finite = slice(2, m - 1)
        assert torch.equal(y.isfinite(), want.isfinite())
        if k64:
            assert torch.equal(y.nan_to_num(), want.nan_to_num())
        else:  # fp32 sums of cols products in another order: cols * 2^-24 at most
            d = (y[finite] - want[finite]).double().norm() / want[finite].double().norm()
            assert d <= cols * 2.0 ** -24


def test_small_products_are_not_rounded_first():
    w_q = torch.empty(2560, 2560 * 4 // 32, dtype=torch.int32)
    bf16 = torch.bfloat16
    assert not ops._round_first(255, w_q, bf16, True, 64, 4)
    assert not ops._round_first(512, w_q, bf16, True, 64, 4)
    assert not ops._round_first(4096, w_q, torch.float32, True, 64, 4)
