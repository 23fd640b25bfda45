"""The short-batch GEMMs (fewer than 256 activation rows) at the edges of their
tiles: rows and columns past a tile, contractions that end inside a span, every
tile shape, bit width, group size and dtype."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def packed(rq, dev, R, K, gs, bits, sdt, seed):
    """Random codes with scales and biases of their own, and the bf16 weights
    bf16(s * q + b) the GEMMs multiply, in float64."""
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(0, 1 << bits, (R, K), generator=g, dtype=torch.uint8).to(dev)
    s = ((torch.rand(R, K // gs, generator=g) + 0.5) * 0.04 / (1 << bits)).to(sdt).to(dev)
    b = (torch.randn(R, K // gs, generator=g) * 0.02).to(sdt).to(dev)
    w = q.double().reshape(R, -1, gs) * s.double()[..., None] + b.double()[..., None]
    return (rq.pack_codes(q, bits), s, b), w.float().bfloat16().double().reshape(R, K)


def check(y, ref, K, what):
    """fp32 sums of K products of bf16 values (2^-24 each), weights that round
    to the other bf16 neighbour where fp32 and float64 differ (2^-8 of one
    weight in 2^16), then the output's own rounding
    (half a unit in the last of 8 significant bits in bf16, 11 in fp16)."""
    y = y.double()
    out = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[ref[1]]
    ref = ref[0]
    assert torch.isfinite(y).all(), what
    rms = ref.square().mean().sqrt()
    err = (y - ref).abs() - 1.01 * out * ref.abs()
    assert err.max() <= 1e-3 * rms, f"{what}: {err.max() / rms:.2e} of the rms"
    fro = ((y - ref).norm() / ref.norm()).item()
    assert fro <= 1e-4 + out, f"{what}: {fro:.2e}"


def out_dtype(xdt, sdt):
    return xdt if xdt == sdt else torch.float32


# m, rows, cols: each 16*tm x 16*tn tile, with partial last tiles, rows that are
# no multiple of four, and contractions that end inside a 128-wide span
TILES = [(17, 1, 32), (255, 3, 64), (33, 203, 96), (60, 8191, 128), (150, 5001, 96),
         (64, 3300, 416), (100, 3071, 800), (77, 8131, 2080), (128, 8190, 2080), (129, 257, 2080)]


@pytest.mark.parametrize("xdt,sdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32),
                                     (torch.float32, torch.bfloat16), (torch.float16, torch.float16),
                                     (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("m,R,K", TILES)
def test_mid_forward_tiles(rq, dev, m, R, K, xdt, sdt):
    gs = 32
    (wq, s, b), w = packed(rq, dev, R, K, gs, 4, sdt, m + R)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(m)).to(xdt).to(dev)
    print("mid forward", m, R, K, xdt, sdt, flush=True)
    y = rq.quantized_matmul(x, wq, s, b, True, gs, 4)
    ref = x.bfloat16().double() @ w.t()
    check(y, (ref, out_dtype(xdt, sdt)), K, "mid forward")


@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("groups", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
def test_mid_forward_groups(rq, dev, bits, gs, groups, sdt):
    """Odd group counts put a row's scales at 2-byte aligned addresses."""
    m, R, K = 37, 77, groups * gs
    (wq, s, b), w = packed(rq, dev, R, K, gs, bits, sdt, bits + groups)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(gs)).to(dev)
    print("mid forward groups", bits, gs, groups, sdt, flush=True)
    y = rq.quantized_matmul(x, wq, s, b, True, gs, bits)
    check(y, (x.bfloat16().double() @ w.t(), torch.float32), K, "mid groups")


def test_mid_forward_repeats_and_unaligned_output(rq, dev):
    """The sum over the waves is in a fixed order; an output buffer that is only
    element-aligned takes scalar stores."""
    m, R, K = 77, 2048, 2048
    (wq, s, b), w = packed(rq, dev, R, K, 64, 4, torch.bfloat16, 5)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
    y = rq.quantized_matmul(x, wq, s, b, True, 64, 4)
    for _ in range(5):
        assert torch.equal(y, rq.quantized_matmul(x, wq, s, b, True, 64, 4))
    buf = torch.zeros(m * R + 3, dtype=torch.bfloat16, device=dev)
    bound = rq.BoundQmm(x, wq, s, b, True, 64, 4, out=buf[1:1 + m * R].view(m, R))
    assert torch.equal(bound.run(), y)
    assert buf[0] == 0 and (buf[1 + m * R:] == 0).all()


def test_mid_forward_infinite_rows_stay_in_their_row(rq, dev):
    """An infinity in one activation row reaches that row's outputs only, also
    where the contraction ends inside a span."""
    m, R, K = 20, 50, 160
    (wq, s, b), w = packed(rq, dev, R, K, 32, 4, torch.bfloat16, 9)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(1))
    x[3, K - 1] = float("inf")
    y = rq.quantized_matmul(x.to(dev), wq, s, b, True, 32, 4)
    ref = x.to(dev).double() @ w.t()
    assert torch.equal(torch.isinf(y), torch.isinf(ref))
    assert torch.isfinite(y[[i for i in range(m) if i != 3]]).all()
    assert torch.equal(y[3].sign(), ref[3].sign().float())


# m, rows, cols of the transposed product: each tile, contractions (rows) that
# are no multiple of 64, 32 or 8, columns that end inside a tile
N_TILES = [(1, 1, 32), (17, 7, 64), (255, 33, 96), (130, 2049, 2080), (200, 515, 2048),
           (200, 1000, 4128), (60, 203, 8192), (60, 1000, 16384), (77, 130, 16416),
           (250, 1000, 2080), (300, 77, 800)]


@pytest.mark.parametrize("xdt,sdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32),
                                     (torch.float32, torch.bfloat16), (torch.float16, torch.float16),
                                     (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("m,R,K", N_TILES)
def test_mid_transposed_tiles(rq, dev, m, R, K, xdt, sdt):
    gs = 32
    (wq, s, b), w = packed(rq, dev, R, K, gs, 4, sdt, m + R)
    x = torch.randn(m, R, generator=torch.Generator().manual_seed(m)).to(xdt).to(dev)
    print("mid transposed", m, R, K, xdt, sdt, flush=True)
    y = rq.quantized_matmul(x, wq, s, b, False, gs, 4)
    check(y, (x.bfloat16().double() @ w, out_dtype(xdt, sdt)), R, "mid transposed")


@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("groups", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
def test_mid_transposed_groups(rq, dev, bits, gs, groups, sdt):
    K = groups * gs
    for m, R in ((37, 77), (100, 640)):
        (wq, s, b), w = packed(rq, dev, R, K, gs, bits, sdt, bits + groups)
        x = torch.randn(m, R, generator=torch.Generator().manual_seed(gs)).to(dev)
        print("mid transposed groups", bits, gs, groups, sdt, flush=True)
        y = rq.quantized_matmul(x, wq, s, b, False, gs, bits)
        check(y, (x.bfloat16().double() @ w, torch.float32), R, "mid transposed groups")


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
def test_mid_transposed_wide_tiles(rq, dev, bits):
    """The 128-column tile of every bit width."""
    m, R, K = 77, 130, 16384 + 32
    (wq, s, b), w = packed(rq, dev, R, K, 32, bits, torch.bfloat16, bits)
    x = torch.randn(m, R, generator=torch.Generator().manual_seed(3)).to(dev)
    y = rq.quantized_matmul(x, wq, s, b, False, 32, bits)
    check(y, (x.bfloat16().double() @ w, torch.float32), R, "mid transposed 128")


def test_mid_transposed_infinite_rows_stay_in_their_row(rq, dev):
    m, R, K = 20, 45, 96
    (wq, s, b), w = packed(rq, dev, R, K, 32, 4, torch.bfloat16, 9)
    x = torch.randn(m, R, generator=torch.Generator().manual_seed(1))
    x[3, R - 1] = float("inf")
    y = rq.quantized_matmul(x.to(dev), wq, s, b, False, 32, 4)
    ref = x.to(dev).double() @ w
    assert torch.equal(torch.isinf(y), torch.isinf(ref))
    assert torch.isfinite(y[[i for i in range(m) if i != 3]]).all()


@pytest.mark.parametrize("rank", [16, 32, 48, 64])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,R,K,bits,gs,sdt", [(17, 96, 160, 4, 32, torch.bfloat16),
                                               (200, 3072, 768, 4, 64, torch.bfloat16),
                                               (255, 256, 2048, 8, 128, torch.bfloat16),
                                               (100, 352, 416, 5, 32, torch.float32),
                                               (300, 320, 1024, 3, 64, torch.bfloat16),
                                               (300, 96, 768, 4, 64, torch.bfloat16)])
def test_qlora_two_launches(rq, dev, m, R, K, bits, gs, sdt, xdt, rank):
    """rq_qlora / rq_qlora_dx outside the in-kernel down-projection: z (u) is that
    of x (dY) itself, rounded once to bf16; the product gets the term of that
    z before its one rounding."""
    from rwkvq import ops
    (wq, s, b), w = packed(rq, dev, R, K, gs, bits, sdt, m + R)
    g = torch.Generator().manual_seed(rank)
    A = (torch.randn(rank, K, generator=g) * K ** -0.5).bfloat16().to(dev)
    B = (torch.randn(R, rank, generator=g) * 0.05).bfloat16().to(dev)
    x = torch.randn(m, K, generator=g).to(xdt).to(dev)
    dy = torch.randn(m, R, generator=g).to(xdt).to(dev)
    odt = out_dtype(xdt, sdt)
    print("qlora two launches", m, R, K, bits, rank, xdt, flush=True)
    y, z = ops.qlora_product(x, wq, s, b, A, B, 2.0, True, gs, bits, odt)
    assert y.dtype == odt
    check(z, (x.double() @ A.double().t(), torch.bfloat16), K, "z")
    check(y, (x.bfloat16().double() @ w.t() + 2.0 * z.double() @ B.double().t(), odt), K, "y")
    dx, u = ops.qlora_dx_product(dy, wq, s, b, A, B, 2.0, gs, bits, odt)
    check(u, (dy.double() @ B.double(), torch.bfloat16), R, "u")
    check(dx, (dy.bfloat16().double() @ w + 2.0 * u.double() @ A.double(), odt), R, "dx")


def test_fp32_down_projection_is_not_less_exact(rq, dev):
    """z of fp32 x as two bf16 values per element: no further from float64 than
    the fp32 product, both rounded once to bf16."""
    from rwkvq import ops
    (wq, s, b), _ = packed(rq, dev, 64, 4096, 64, 4, torch.bfloat16, 1)
    g = torch.Generator().manual_seed(0)
    x = torch.randn(128, 4096, generator=g).to(dev)
    A = (torch.randn(32, 4096, generator=g) / 64).bfloat16().to(dev)
    B = torch.zeros(64, 32, dtype=torch.bfloat16, device=dev)
    _, z = ops.qlora_product(x, wq, s, b, A, B, 1.0, True, 64, 4, torch.float32)
    ref = x.double() @ A.double().t()
    old = (x @ A.float().t()).bfloat16()
    err = lambda t: ((t.double() - ref).norm() / ref.norm()).item()  # noqa: E731
    assert err(z) <= 1.01 * err(old), (err(z), err(old))


@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m", [3, 7, 9, 16])
@pytest.mark.parametrize("groups", [1, 3, 5, 17])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
def test_qmv_mid_groups(rq, dev, bits, gs, groups, m, sdt):
    """The decode GEMV of any layout: weights unrounded, x rounded to bf16 once
    (sums of K products: 2^-24 each)."""
    R, K = 37, groups * gs
    (wq, s, b), _ = packed(rq, dev, R, K, gs, bits, sdt, bits + groups)
    w = rq.unpack_codes(wq, bits).double().reshape(R, -1, gs)
    w = (w * s.double()[..., None] + b.double()[..., None]).reshape(R, K)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(gs)).to(dev)
    print("qmv mid", bits, gs, groups, m, sdt, flush=True)
    y = rq.quantized_matmul(x, wq, s, b, True, gs, bits).double()
    ref = x.bfloat16().double() @ w.t()
    assert (y - ref).norm() <= 1e-5 * ref.norm() and (y - ref).abs().max() <= 3e-5 * ref.abs().max()


@pytest.mark.parametrize("xdt", [torch.float32, torch.float16])
@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("R,K,gs,bits", [(50, 160, 32, 6), (2048, 2048, 32, 5), (33, 768 + 64, 64, 4),
                                         (7, 10240, 32, 8)])
def test_qmv_mid_split_activations(rq, dev, R, K, gs, bits, m, xdt):
    """fp32 and f16 x at m <= 2 as two bf16 rows (16 significant bits), fp32
    scales: within 2^-17 of the product of x itself, and its fp32 sums."""
    (wq, s, b), _ = packed(rq, dev, R, K, gs, bits, torch.float32, R)
    w = rq.unpack_codes(wq, bits).double().reshape(R, -1, gs)
    w = (w * s.double()[..., None] + b.double()[..., None]).reshape(R, K)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(m)).to(xdt).to(dev)
    y = rq.quantized_matmul(x, wq, s, b, True, gs, bits).double()
    ref = x.double() @ w.t()
    assert (y - ref).norm() <= 1e-5 * ref.norm() and (y - ref).abs().max() <= 3e-5 * ref.abs().max()


def test_qmv_mid_grouped_matches_single(rq, dev):
    """Several problems of one launch, ragged rows, against their single ones."""
    K, m = 2048, 11
    ws = [packed(rq, dev, R, K, 64, 4, torch.bfloat16, R)[0] for R in (2048, 77, 2048, 16, 1)]
    xs = [torch.randn(m, K, generator=torch.Generator().manual_seed(i)).bfloat16().to(dev) for i in range(5)]
    ys = rq.grouped_qmv(xs, ws, 64, 4)
    ref = [rq.quantized_matmul(x, *w, True, 64, 4) for x, w in zip(xs, ws)]
    for y, r in zip(ys, ref):
        err = ((y.double() - r.double()).norm() / r.double().norm()).item()
        assert err <= 2.0 ** -8, err  # another split of K: outputs round either way


@pytest.mark.parametrize("rank", [16, 48])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m", [1, 2, 3, 16])
@pytest.mark.parametrize("R,K,bits,gs", [(768, 768, 4, 64), (96, 416, 3, 32)])
def test_qlora_decode_rows_keep_the_unrounded_weights(rq, dev, R, K, bits, gs, m, xdt, rank):
    """A LoRALinear step of up to 16 rows is quantized_matmul's product, whose
    weights are not rounded, plus the term of the bf16 z: the bits of the two
    composed, and for fp32 x their fp32 sums (2^-24 an addition)."""
    from rwkvq import ops
    (wq, s, b), _ = packed(rq, dev, R, K, gs, bits, torch.bfloat16, R)
    base = rq.QuantizedLinear(K, R, bias=False, group_size=gs, bits=bits, device=dev)
    base.weight, base.scales, base.biases = wq, s, b
    lay = rq.LoRALinear(rank=rank, alpha=32.0, base_module=base)
    g = torch.Generator().manual_seed(m)
    with torch.no_grad():
        lay.lora_b.copy_(torch.randn(R, rank, generator=g) * 0.05)
    x = torch.randn(m, K, generator=g).to(xdt).to(dev)
    print("qlora decode rows", m, R, K, bits, rank, xdt, flush=True)
    A, B = lay.lora_a.detach(), lay.lora_b.detach()
    z, y = ops.lora_down(x, A), lay(x)
    assert torch.equal(y, ops.quantized_matmul_lora(x, wq, s, b, z, B, lay.scale, True, gs, bits))
    ref = rq.quantized_matmul(x, wq, s, b, True, gs, bits).double() + lay.scale * (z.double() @ B.double().t())
    assert y.dtype == xdt
    if xdt == torch.float32:
        assert (y.double() - ref).norm() <= 1e-6 * ref.norm()


def _z_and_u(rq, dev, x, A, transposed):
    """z = x A^T of the two-launch forward, or u = dY B of the two-launch dX for
    dY = x and B = A^T, through a weight that plays no part."""
    from rwkvq import ops
    rank, K = A.shape
    if not transposed:
        (wq, s, b), _ = packed(rq, dev, 32, K, 32, 4, torch.bfloat16, 1)
        B = torch.zeros(32, rank, dtype=torch.bfloat16, device=dev)
        return ops.qlora_product(x, wq, s, b, A, B, 1.0, True, 32, 4, torch.float32)[1]
    (wq, s, b), _ = packed(rq, dev, K, 32, 32, 4, torch.bfloat16, 1)
    A2 = torch.zeros(rank, 32, dtype=torch.bfloat16, device=dev)
    return ops.qlora_dx_product(x, wq, s, b, A2, A.t().contiguous(), 1.0, 32, 4, torch.float32)[1]


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("rank", [16, 32, 48, 64])
def test_fp32_down_projection_takes_all_24_bits(rq, dev, rank, transposed):
    """Neighbouring elements of x, all 24 bits in use, that differ from the 17th on, against
    adapter columns of opposite sign: z is the sum of the differences (each below
    2^-16, K/2 of them), rounded to bf16 (half a unit in the last of 8
    significant bits: 2^-8), its fp32 sums K additions of
    partial sums below 2^4 (2^-24 each, of either sign)."""
    K, m = 1024, 37
    g = torch.Generator().manual_seed(rank)
    v = 1.0 + torch.randint(0, 2 ** 22, (m, K // 2), generator=g).float() * 2.0 ** -23
    x = torch.empty(m, K)
    x[:, 0::2], x[:, 1::2] = v + torch.randint(0, 128, v.shape, generator=g) * 2.0 ** -23, v
    A = torch.ones(rank, K)
    A[:, 1::2] = -1.0
    A = (A * torch.where(torch.arange(rank) % 2 == 0, 1.0, -2.0)[:, None]).bfloat16().to(dev)
    z = _z_and_u(rq, dev, x.to(dev), A, transposed).double()
    ref = x.double().to(dev) @ A.double().t()
    sums = K ** 0.5 * 2.0 ** -24 * 2 ** 4
    assert ((z - ref).abs() <= 2.0 ** -8 * ref.abs() + sums).all(), ((z - ref) / ref).abs().max()


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("rank", [16, 32, 48, 64])
@pytest.mark.parametrize("val", [float("inf"), -float("inf"), float("nan"), 3.402e38, -3.4e38, 1e-40])
def test_fp32_down_projection_special_values(rq, dev, val, rank, transposed):
    """An infinity gives infinities of its sign times the adapter's, a finite value
    above bf16's largest stays finite, a NaN stays in its row."""
    K, m = 96, 20
    g = torch.Generator().manual_seed(rank)
    x = torch.randn(m, K, generator=g)
    x[3, 41] = val
    if val != val:  # payload in the lower half only
        x.view(torch.int32)[3, 41] = 0x7f800001
    A = ((torch.rand(rank, K, generator=g) + 0.5) / 64).bfloat16()
    A[1::2] *= -1
    z = _z_and_u(rq, dev, x.to(dev), A.to(dev), transposed).cpu().double()
    ref = x.double() @ A.double().t()
    assert torch.equal(z.isnan(), ref.isnan()) and torch.equal(z.isinf(), ref.isinf())
    assert torch.equal(z.sign().nan_to_num(), ref.sign().nan_to_num())
    ok = ref.isfinite()
    # fp32 sums of K terms, rounded once to 8 significant bits (half a unit: 2^-8)
    assert ((z - ref)[ok].abs() <= 2.0 ** -8 * ref[ok].abs() + K * 2.0 ** -24).all()


@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R", [1, 31, 45, 77, 96])
@pytest.mark.parametrize("m", [3, 40, 300])
def test_mid_transposed_infinite_weights_of_the_last_row(rq, dev, m, R, sdt):
    """A contraction that ends inside a 32-row step pads with zeros of both
    operands: infinite weights of the last row give infinities, no NaN."""
    K, gs = 96, 32
    (wq, s, b), w = packed(rq, dev, R, K, gs, 4, sdt, R)
    b[R - 1, 1] = float("inf")
    w[R - 1, gs:2 * gs] = float("inf")
    x = torch.rand(m, R, generator=torch.Generator().manual_seed(1)).to(dev) + 0.1
    y, ref = rq.quantized_matmul(x, wq, s, b, False, gs, 4), x.double() @ w
    assert torch.equal(y.isinf(), ref.isinf()) and torch.equal(y.isfinite(), ref.isfinite())


@pytest.mark.parametrize("xdt,sdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32),
                                     (torch.float16, torch.float16), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("m,R,K,bits,gs", [(255, 65537, 64, 4, 64), (129, 60001, 96, 8, 32), (200, 65536, 160, 3, 32),
                                           (130, 65530, 128, 5, 128), (255, 65500, 384, 6, 64), (255, 65536, 256, 2, 32)])
def test_forward_128_tiles_of_many_weight_rows(rq, dev, m, R, K, bits, gs, xdt, sdt):
    """Rows and columns past a tile, contractions that end inside a 64-wide stage."""
    (wq, s, b), w = packed(rq, dev, R, K, gs, bits, sdt, m + K)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(m)).to(xdt).to(dev)
    print("forward 128 tiles", m, R, K, bits, xdt, sdt, flush=True)
    y = rq.quantized_matmul(x, wq, s, b, True, gs, bits)
    check(y, (x.bfloat16().double() @ w.t(), out_dtype(xdt, sdt)), K, "128 tiles")
    if xdt == torch.float32 and sdt == torch.float32:
        assert torch.equal(y, rq.quantized_matmul(x.bfloat16(), wq, s, b, True, gs, bits))


@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("R,K,gs,bits,sdt", [(8200, 2048, 64, 4, torch.float32), (12290, 2080, 32, 4, torch.float32),
                                             (16380, 2176, 128, 8, torch.float32), (12300, 2112, 64, 3, torch.float32),
                                             (8193, 2144, 32, 2, torch.float32), (24000, 1344, 64, 4, torch.bfloat16),
                                             (8200, 1344, 64, 2, torch.float16)])
def test_qmv_waves_splitting_k(rq, dev, R, K, gs, bits, sdt, m):
    """Few bf16 rows against fp32 scales or odd group counts: ragged rows, spans
    that end inside the contraction; weights unrounded, sums of K products
    (2^-24 each), a 16-bit y rounded once."""
    (wq, s, b), _ = packed(rq, dev, R, K, gs, bits, sdt, bits)
    w = rq.unpack_codes(wq, bits).double().reshape(R, -1, gs)
    w = (w * s.double()[..., None] + b.double()[..., None]).reshape(R, K)
    x = torch.randn(m, K, generator=torch.Generator().manual_seed(gs)).bfloat16().to(dev)
    print("qmv ksplit", R, K, gs, bits, sdt, m, flush=True)
    y = rq.quantized_matmul(x, wq, s, b, True, gs, bits)
    ref = x.double() @ w.t()
    out = 2.0 ** -8 if y.dtype == torch.bfloat16 else 0.0
    assert (y.double() - ref).norm() <= (1e-5 + out) * ref.norm()
    assert ((y.double() - ref).abs() <= 3e-5 * ref.abs().max() + 1.01 * out * ref.abs()).all()
