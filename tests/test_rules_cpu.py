"""The size rules of csrc/hy_rules.hpp against the times they were made from (us on one
MI355X): a batch takes a kernel that is at most a tenth slower than the other one."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = """
#include "hy_rules.hpp"
extern "C" int gemv_batch(int wt, unsigned T, int K, int E, int H, int I, int sh) {
    return hy::gemv_batch(wt, T, K, E, H, I, sh);
}
extern "C" int few_batch(int wt, int T, int K, int E, int I, int sh, int cached) {
    return hy::few_batch(wt, T, K, E, I, sh, cached != 0);
}
extern "C" int gemm_mid_size(int M, int N, int K) { return hy::gemm_mid_size(M, N, K); }
extern "C" int gemm_takes_scratch(int M, int N, int K) { return hy::gemm_takes_scratch(M, N, K); }
extern "C" int norm_in_registers(int T, int H) { return hy::norm_in_registers(T, H); }
"""
Q4, Q8 = 2, 8


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT}/include",
                    f"-I{ROOT}/hunyuan-image-3-80b.cpp_amd/csrc", str(d / "shim.cpp"), "-o", str(d / "shim.so")], check=True)
    return C.CDLL(str(d / "shim.so"))


# type, E, K, H, I: (T, GEMV, stream of hy_mfma_few.hip)
GEMV_TIMES = [
    (Q4, 64, 8, 4096, 3072, (24, 295, 296), (28, 324, 298), (40, 438, 332), (64, 630, 341)),
    (Q4, 32, 4, 4096, 3072, (20, 166, 165), (32, 209, 205), (40, 236, 208)),
    (Q4, 32, 4, 2048, 1536, (24, 66, 71), (28, 76, 68), (40, 79, 75)),
    (Q4, 32, 4, 1024, 768, (28, 42.4, 44.3), (32, 42.4, 44.0), (40, 45.6, 46.3)),
    (Q4, 16, 4, 1024, 768, (17, 38.1, 44.1), (20, 39.1, 44.1)),
    (Q4, 16, 4, 1024, 1408, (17, 63.5, 49.7), (20, 63.5, 49.5)),
    (Q4, 16, 2, 4096, 3072, (28, 126, 123), (40, 154, 135)),
    (Q4, 16, 2, 2048, 1536, (28, 60.2, 60.6), (40, 67.1, 63.2)),
    (Q4, 16, 2, 1024, 768, (28, 37.6, 46.2), (32, 38.1, 46.3), (40, 41.7, 45.2)),
    (Q4, 16, 2, 1024, 1408, (28, 62.4, 52.3), (40, 69.0, 51.0)),
    (Q4, 8, 2, 2048, 1536, (17, 51.4, 62.0), (20, 52.8, 59.3)),
    (Q4, 8, 1, 4096, 3072, (28, 93, 94), (32, 102, 94), (40, 119, 95)),
    (Q4, 8, 1, 2048, 1536, (28, 50.8, 62.1), (32, 52.0, 61.6), (40, 57.0, 61.4)),
    (Q4, 8, 1, 1024, 768, (28, 35.1, 45.4), (40, 38.5, 47.3)),
    (Q4, 4, 1, 2048, 1536, (17, 46.9, 61.6), (20, 48.3, 61.3)),
    (Q8, 64, 8, 4096, 3072, (17, 437, 403), (24, 468, 410)),
    (Q8, 64, 8, 1024, 768, (17, 51.0, 54.1), (20, 53.1, 54.6)),
    (Q8, 32, 4, 1024, 768, (17, 39.2, 45.1), (20, 39.9, 45.0)),
    (Q8, 32, 4, 1024, 1408, (17, 68.6, 55.3), (20, 70.3, 55.8)),
    (Q8, 16, 2, 4096, 3072, (17, 148, 127), (20, 132, 125)),
    (Q8, 16, 2, 2048, 1536, (17, 56.6, 62.4), (20, 56.7, 62.4)),
    (Q8, 16, 2, 1024, 768, (17, 35.5, 43.5), (20, 36.4, 44.1)),
    (Q8, 8, 1, 4096, 3072, (17, 90.5, 109.9), (20, 92.9, 109.0)),
    (Q8, 8, 1, 2048, 1536, (17, 47.4, 59.2), (20, 47.2, 59.1)),
    (Q8, 16, 1, 1024, 768, (40, 38.4, 45.9)),
]


@pytest.mark.parametrize("row", GEMV_TIMES, ids=lambda r: "-".join(map(str, r[:5])))
def test_gemv_or_stream(rules, row):
    wt, E, K, H, I = row[:5]
    for T, gemv, stream in row[5:]:
        took = gemv if rules.gemv_batch(wt, T, K, E, H, I, 1) else stream
        assert took <= 1.1 * min(gemv, stream), T


def test_gemv_line_ends(rules):
    """Decode batches always, prompts and unquantized weights never; with and without a
    shared expert."""
    for sh in (0, 1):
        for E, K in ((64, 8), (1, 1), (64, 64)):
            for T in (1, 16):
                assert rules.gemv_batch(Q4, T, K, E, 4096, 3072, sh) and rules.gemv_batch(Q8, T, K, E, 128, 128, sh)
            assert not rules.gemv_batch(Q4, 5 * E + 17, K, E, 4096, 3072, sh)
            assert not rules.gemv_batch(Q8, 5 * E + 17, K, E, 4096, 3072, sh)
            assert not rules.gemv_batch(0, 17, K, E, 4096, 3072, sh)


# type, E, K, H, I (weights in the Infinity Cache): (T, stream, tall shape)
FEW_TIMES = [
    (Q4, 32, 4, 2048, 1536, (256, 99, 130), (400, 127, 134), (512, 149, 172)),
    (Q4, 64, 8, 1024, 768, (300, 77, 94), (400, 90, 95), (512, 97, 115)),
    (Q4, 16, 4, 4096, 3072, (200, 212, 220), (256, 242, 288)),
    (Q8, 16, 4, 2048, 1536, (150, 91, 108), (200, 93, 110), (256, 105, 113)),
    (Q8, 32, 4, 2048, 1536, (256, 132, 133), (300, 155, 136), (400, 157, 137), (448, 158, 138), (496, 165, 164)),
    (Q8, 32, 4, 1024, 1408, (256, 78, 88), (300, 89, 88), (400, 100, 91), (496, 102, 108)),
    (Q8, 32, 4, 1024, 768, (300, 69, 74), (400, 72, 75), (512, 82, 83)),
    (Q8, 64, 8, 1024, 768, (256, 87, 89), (300, 92, 92), (400, 105, 93), (448, 107, 94), (496, 109, 110)),
    (Q8, 48, 6, 1536, 1024, (270, 104, 106), (400, 116, 108), (448, 118, 110), (496, 123, 132)),
    (Q8, 64, 8, 1024, 1408, (256, 121, 129), (300, 135, 131), (400, 153, 137), (448, 156, 138)),
    (Q8, 8, 1, 4096, 3072, (256, 149, 180), (300, 174, 183), (400, 175, 188)),
    (Q8, 8, 2, 4096, 3072, (150, 150, 178), (200, 169, 180), (256, 171, 186)),
    (Q8, 16, 2, 2048, 1536, (300, 90, 110), (400, 104, 112), (512, 103, 113)),
]


@pytest.mark.parametrize("row", FEW_TIMES, ids=lambda r: "-".join(map(str, r[:5])))
def test_stream_or_tall(rules, row):
    wt, E, K, H, I = row[:5]
    for T, few, tall in row[5:]:
        took = few if rules.few_batch(wt, T, K, E, I, 1, 1) else tall
        assert took <= 1.05 * min(few, tall), T


def test_stream_line_without_the_cache(rules):
    for wt in (Q4, Q8):
        for E, K in ((64, 8), (16, 4)):
            T = 26 * E // K
            assert rules.few_batch(wt, T, K, E, 3072, 1, 0) and not rules.few_batch(wt, T + 1, K, E, 3072, 1, 0)
            assert not rules.few_batch(wt, 64 * E // K + 1, K, E, 64, 0, 1)


# H, T, rows in registers, one wave per row
@pytest.mark.parametrize("H,T,regs,wave", [(4096, 1, 6.3, 10.7), (4096, 8192, 39.7, 58.5), (2816, 300, 6.2, 9.3),
                                           (1536, 4096, 10.2, 13.4), (1536, 8192, 17.7, 22.7), (1024, 2000, 6.4, 6.4),
                                           (1024, 4096, 8.1, 7.7), (256, 2000, 6.2, 6.3), (256, 8192, 10.9, 6.2)])
def test_norm_kernel(rules, H, T, regs, wave):
    assert (regs if rules.norm_in_registers(T, H) else wave) <= 1.02 * min(regs, wave)


def test_norm_registers_hold_the_row(rules):
    assert not any(rules.norm_in_registers(5, H) for H in (64, 1088, 4100, 4352, 8192))


def test_decode_lm_head_takes_no_scratch(rules):
    """One to 16 rows stream over W; more rows of a mid-size grid are cut into pieces."""
    for N, K in ((32000, 2048), (128256, 4096), (8192, 1024)):
        assert rules.gemm_mid_size(1, N, K) and not rules.gemm_takes_scratch(1, N, K)
        assert rules.gemm_mid_size(16, N, K) and not rules.gemm_takes_scratch(16, N, K)
        assert not rules.gemm_mid_size(17, N, K) or rules.gemm_takes_scratch(17, N, K)
    for M, N, K in ((256, 4096, 1024), (1290, 6150, 1024), (17, 32000, 2048)):
        assert rules.gemm_mid_size(M, N, K) and rules.gemm_takes_scratch(M, N, K)
    for M, N, K in ((256, 4095, 1040), (100, 512, 4096), (4096, 65536, 4096), (128, 8192, 32)):
        assert not rules.gemm_mid_size(M, N, K) and not rules.gemm_takes_scratch(M, N, K)
