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
