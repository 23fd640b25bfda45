"""Which kernel a product takes (rq_mid.h, host code) against measured times."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = """
#include "rwkv-metal_amd/csrc/rq_mid.h"
extern "C" int short_takes_128(long m, long rows, long cols, int bits) {
    return rq::t128_us(m, rows, cols, bits) < rq::mid_short_us(m, rows, cols, bits);
}
extern "C" int takes_mid(int x_dt, int k64, int lora, long m, long rows, long cols, int gs, int bits) {
    return rq::forward_takes_mid(x_dt, k64, lora, m, rows, cols, gs, bits);
}
extern "C" int splits_k(int x_dt, long m, long cols, int gs, int bits, long rowblocks) {
    return rq::qmv_splits_k(x_dt, m, cols, gs, bits, rowblocks);
}
extern "C" int over_split(int x_dt, long m, long cols, int bits, long rowblocks) {
    return rq::qmv_mid_over_split(x_dt, m, cols, bits, rowblocks);
}
extern "C" int large_mid(int x_dt, int sb_dt, long m, long cols, int gs, int bits) {
    return rq::qmv_large_takes_mid(x_dt, sb_dt, m, cols, gs, bits);
}
"""
BF16, F32 = 0, 2


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    so = str(tmp_path_factory.mktemp("choice") / "choice.so")
    subprocess.run([cxx, "-std=c++17", "-shared", "-fPIC", "-I", ROOT, "-x", "c++", "-", "-o", so],
                   input=SHIM.encode(), check=True)
    lib = ctypes.CDLL(so)
    lib.short_takes_128.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int]
    lib.takes_mid.argtypes = [ctypes.c_int] * 3 + [ctypes.c_long] * 3 + [ctypes.c_int] * 2
    lib.splits_k.argtypes = [ctypes.c_int] + [ctypes.c_long] * 2 + [ctypes.c_int] * 2 + [ctypes.c_long]
    lib.over_split.argtypes = [ctypes.c_int] + [ctypes.c_long] * 2 + [ctypes.c_int, ctypes.c_long]
    lib.large_mid.argtypes = [ctypes.c_int] * 2 + [ctypes.c_long] * 2 + [ctypes.c_int] * 2
    return lib


@pytest.mark.parametrize("m,rows,cols,bits,big", [
    # us measured 128 x 128 tiles / short-batch tiles, bf16 x
    (200, 65536, 768, 4, True),     # 63 / 87
    (128, 65536, 768, 8, True),     # 40 / 51
    (255, 65536, 2048, 3, True),    # 148 / 189
    (200, 65536, 2048, 6, True),    # 176 / 198
    (64, 65536, 2048, 4, False),    # 76 / 45
    (200, 16384, 4096, 4, False),   # 115 / 72
    (200, 10240, 2560, 4, False),   # 68 / 40
    (128, 32000, 512, 5, False),    # 36 / 22
    (77, 2048, 2048, 4, False)])    # 58 / 7
def test_fewer_than_256_rows(choice, m, rows, cols, bits, big):
    assert bool(choice.short_takes_128(m, rows, cols, bits)) == big


@pytest.mark.parametrize("x_dt,lora,m,rows,cols,bits,mid", [
    # us measured 256-row tiles / short-batch tiles; fp32 scales at group size 32
    (BF16, 0, 1024, 8192, 2048, 4, False),   # 69 / 93
    (BF16, 0, 2048, 4096, 4096, 4, False),   # 114 / 180
    (BF16, 0, 512, 16384, 4096, 4, False),   # 116 / 152
    (F32, 0, 2048, 4096, 4096, 4, False),    # 270 / 553
    (F32, 0, 2048, 8192, 2048, 4, False),    # 312 / 567
    (F32, 1, 2048, 4096, 4096, 4, False),
    (BF16, 0, 2048, 2048, 2048, 4, True),    # 55 / 48
    (F32, 0, 1024, 4096, 4096, 5, True),     # 287 / 236
    (BF16, 0, 300, 768, 768, 4, True),       # 26 / 5
    (F32, 0, 512, 2048, 2048, 6, True),
    (F32, 1, 100, 65536, 768, 4, True)])
def test_256_rows_outside_the_64_wide_stages(choice, x_dt, lora, m, rows, cols, bits, mid):
    assert bool(choice.takes_mid(x_dt, 0, lora, m, rows, cols, 32, bits)) == mid


@pytest.mark.parametrize("x_dt,m,rows,cols,gs,bits,ks", [
    # us measured qmv_kernel splitting K / qmv_mid, fp32 scales
    (BF16, 1, 16384, 4096, 64, 4, True),     # 14.1 / 23.0
    (BF16, 3, 16384, 4096, 64, 4, True),     # 17.5 / 23.5
    (BF16, 4, 16384, 4096, 64, 4, False),    # 28.6 / 22.8
    (F32, 1, 16384, 4096, 64, 4, False),
    (BF16, 1, 2048, 2048, 64, 4, True),      # 4.3 / 5.1
    (BF16, 1, 4096, 4096, 32, 4, False),     # 8.9 / 8.3
    (BF16, 1, 8192, 2048, 32, 4, True),      # 7.2 / 8.2
    (BF16, 2, 16384, 4096, 128, 8, True),    # 20.2 / 26.5
    (BF16, 1, 10240, 2560, 64, 3, False),    # 14.9 / 13.5
    (BF16, 2, 16384, 4096, 128, 3, True),    # 21.4 / 22.9
    (BF16, 1, 12288, 3072, 128, 2, True),    # 10.2 / 14.5
    (BF16, 1, 16384, 4096, 32, 6, False),
    (BF16, 2, 2560, 10240, 64, 8, True),     # 13.7 / 15.8, bf16 scales
    (BF16, 2, 2560, 10240, 32, 8, False),    # 23.0 / 17.1
    (BF16, 3, 10240, 10240, 64, 4, False)])
def test_small_decode_launches_outside_the_split_gemv(choice, x_dt, m, rows, cols, gs, bits, ks):
    assert bool(choice.splits_k(x_dt, m, cols, gs, bits, (rows + 15) // 16)) == ks


@pytest.mark.parametrize("x_dt,m,rows,cols,bits,mid", [
    # us measured split GEMV / qmv_mid
    (BF16, 8, 768, 768, 4, True),        # 5.5 / 4.1
    (BF16, 5, 10240, 2560, 4, True),     # 12.8 / 11.2
    (BF16, 5, 16384, 768, 4, False),     # 7.0 / 7.5
    (BF16, 5, 2048, 2048, 6, False),     # 7.4 / 8.3
    (BF16, 6, 16384, 4096, 2, False),    # 19.1 / 22.2
    (F32, 5, 10240, 2560, 8, False),     # 12.8 / 13.7
    (BF16, 8, 10240, 2560, 6, True),     # 20.1 / 17.5
    (F32, 8, 10240, 2560, 5, False),     # 17.4 / 20.0
    (BF16, 5, 1024, 1024, 3, True),      # 5.6 / 4.8
    (BF16, 4, 768, 768, 4, False)])
def test_5_to_8_decode_rows(choice, x_dt, m, rows, cols, bits, mid):
    assert bool(choice.over_split(x_dt, m, cols, bits, (rows + 15) // 16)) == mid


@pytest.mark.parametrize("x_dt,sb_dt,m,cols,gs,bits,mid", [
    # us measured qmv_kernel / qmv_mid, 65536 rows unless noted; fp32 x at 1 and 2 rows
    # counts twice
    (BF16, BF16, 1, 768, 64, 2, False),    # 11.8 / 16.3
    (BF16, BF16, 8, 2048, 64, 2, False),   # 28.6 / 38.9
    (F32, BF16, 8, 768, 64, 2, True),      # 23.2 / 18.5
    (BF16, BF16, 1, 768, 64, 3, False),    # 17.7 / 18.9
    (BF16, BF16, 2, 768, 64, 6, True),     # 36.4 / 30.1
    (BF16, BF16, 8, 2048, 64, 5, True),    # 82 / 70
    (BF16, BF16, 9, 2048, 64, 4, True),
    (BF16, F32, 1, 768, 64, 4, False),     # 10.1 / 16.6
    (BF16, F32, 4, 2048, 64, 4, False),    # 26.7 / 38.8
    (F32, F32, 4, 3072, 64, 4, False),     # 42 / 49 (49152 rows)
    (BF16, F32, 8, 2048, 64, 4, False),    # 36.9 / 40.1
    (F32, F32, 8, 2048, 64, 4, True),
    (BF16, F32, 1, 2048, 32, 4, False),    # 27.7 / 37.9
    (F32, F32, 4, 2048, 32, 4, True),
    (BF16, F32, 1, 2048, 64, 6, False),    # 70 / 77
    (BF16, F32, 2, 2048, 32, 6, True)])
def test_large_decode_launches_outside_the_streamed_gemv(choice, x_dt, sb_dt, m, cols, gs, bits, mid):
    assert bool(choice.large_mid(x_dt, sb_dt, m, cols, gs, bits)) == mid
