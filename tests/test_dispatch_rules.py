"""CPU check of the rules that choose a kernel (quant_ops_amd/csrc/dispatch_rules.h),
compiled as they are, at the lines that their measurements drew (256 CUs)."""
import ctypes
import os
import subprocess

import pytest

from test_gpu_f6_tiles import CASES, SPLIT_CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256

SOURCE = r"""
#include "dispatch_rules.h"
extern "C" int padded_mfma(int M, int N, int64_t tokens, int f16, int64_t cus) {
  return qo::fq_padded_mfma(M, N, tokens, f16 != 0, cus);
}
extern "C" int generic_small(int64_t M, int64_t N, int64_t K, int b_nk, int over_skinny, int64_t cus) {
  return qo::gemm_generic_small(M, N, K, b_nk != 0, over_skinny != 0, cus);
}
extern "C" int tile(int64_t M, int64_t N, int64_t K, int f32, int64_t cus) { return qo::f6_tile(M, N, K, f32 != 0, cus); }
extern "C" int generic_few(int M, int N, int64_t tokens, int f32, int pack, int64_t cus) {
  return qo::fq_generic_few(M, N, tokens, f32 != 0, pack != 0, cus);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, lib = d / "rules.cpp", d / "librules.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{ROOT}/quant_ops_amd/csrc", str(src), "-o",
                    str(lib)], check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("m,n,f16,first,last", [
    (56, 64, True, 769, 1024), (56, 64, False, 769, 1024),
    (64, 80, True, 513, None), (64, 112, True, 257, 512), (72, 96, False, 257, 512), (80, 112, False, 257, 512),
])
def test_padded_shapes_on_the_fragment_kernel(rules, m, n, f16, first, last):
    def takes(tokens):
        return bool(rules.padded_mfma(m, n, ctypes.c_int64(tokens), int(f16), ctypes.c_int64(CUS)))

    assert not takes(1) and not takes(first - 1) and takes(first)
    assert takes(8192) if last is None else takes(last) and not takes(last + 1) and not takes(8192)


def test_other_shapes_stay_on_the_tile_kernel(rules):
    for m, n, f16 in [(64, 80, 0), (128, 144, 1), (86, 128, 1), (108, 128, 0), (76, 128, 1), (96, 96, 1), (112, 64, 1)]:
        for tokens in (1, 256, 300, 512, 600, 1024, 4096):
            assert not rules.padded_mfma(m, n, ctypes.c_int64(tokens), f16, ctypes.c_int64(CUS)), (m, n, f16, tokens)


def test_few_features_and_tokens_on_the_generic_kernel(rules):
    def takes(m, n, tokens, f32, pack):
        return bool(rules.generic_few(m, n, ctypes.c_int64(tokens), int(f32), int(pack), ctypes.c_int64(CUS)))

    for tokens in (1, 255):
        assert takes(8, 8, tokens, False, False) and takes(8, 12, tokens, True, False) and takes(4, 4, tokens, True, True)
        assert takes(4, 6, tokens, True, False)
        assert not takes(8, 12, tokens, False, False) and not takes(12, 12, tokens, True, False)
        assert not takes(5, 8, tokens, False, False) and not takes(8, 8, tokens, False, True) and not takes(4, 8, tokens, True, True)
    for f32 in (False, True):
        for pack in (False, True):
            assert not takes(4, 4, 256, f32, pack) and not takes(64, 64, 1, f32, pack)


def test_small_ragged_products_on_the_generic_kernel(rules):
    def takes(m, n, k, over_skinny, b_nk=True):
        return bool(rules.generic_small(*(ctypes.c_int64(v) for v in (m, n, k)), int(b_nk), int(over_skinny),
                                        ctypes.c_int64(CUS)))

    for m, n, k in [(1, 64, 8), (1024, 64, 8), (256, 37, 64), (300, 64, 200), (128, 1001, 200), (256, 1001, 64), (1, 1, 64)]:
        assert takes(m, n, k, False) and takes(m, n, k, False, b_nk=False), (m, n, k)
    assert takes(128, 513, 264, False) and not takes(128, 513, 264, False, b_nk=False)
    for m, n, k in [(512, 1001, 64), (256, 1001, 200), (1, 5, 328), (1, 1, 4096), (16, 1631, 8064), (4096, 4095, 64)]:
        assert not takes(m, n, k, False) and not takes(m, n, k, False, b_nk=False), (m, n, k)
    for m, n, k in [(1, 5, 32), (64, 37, 64), (64, 2051, 32)]:
        assert takes(m, n, k, True), (m, n, k)
    for m, n, k in [(1, 5, 96), (64, 2051, 64), (16, 151643, 4096), (64, 4095, 64)]:
        assert not takes(m, n, k, True), (m, n, k)


TILES = ["256x224", "256x256", "128x128", "128x64", "split 128x128", "split 128x64"]   # F6Tile's order


@pytest.mark.parametrize("m,n,k,tile,tile_f32", CASES + SPLIT_CASES)
def test_fp6_tile_of_the_gpu_cases(rules, m, n, k, tile, tile_f32):
    """The sizes of test_gpu_f6_tiles.py run on the tiles that they are there for."""
    got = [TILES[rules.tile(*(ctypes.c_int64(v) for v in (m, n, k)), f32, ctypes.c_int64(CUS))] for f32 in (0, 1)]
    assert got == [tile, tile_f32]


def test_fp6_tile_of_common_products(rules):
    def tile(m, n, k):
        return TILES[rules.tile(*(ctypes.c_int64(v) for v in (m, n, k)), 0, ctypes.c_int64(CUS))]

    assert tile(4096, 14336, 4096) == "256x224" and tile(2048, 14336, 4096) == "256x224"
    assert tile(4096, 4096, 14336) == "256x256"
    assert tile(512, 14336, 4096) == "128x128" and tile(512, 4096, 14336) == "split 128x64"
    assert tile(400, 8192, 28672) == "split 128x128"
