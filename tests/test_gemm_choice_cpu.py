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
