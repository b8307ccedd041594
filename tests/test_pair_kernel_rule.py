"""Which sizes the gradient kernel of short sequences takes (csrc/attention_pair_rule.h, plain arithmetic, compiled here with
the host compiler): none whose LDS a compute unit does not have, and no size refused that has it."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nnlib.jl_amd", "csrc")
SHIM = """#include "attention_pair_rule.h"
extern "C" int64_t lds(int64_t Lq, int64_t Lkv, int words) { return (int64_t)pair_kernel_lds(Lq, Lkv, words != 0); }
extern "C" int takes(int64_t Lq, int64_t Lkv, int64_t pairs, int words) { return pair_kernel_sizes(Lq, Lkv, pairs, words != 0); }
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "shim.cpp"), "-o", str(d / "shim.so")], check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    lib.lds.restype = ctypes.c_int64
    lib.lds.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    lib.takes.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return lib


@pytest.mark.parametrize("pairs", [1, 255, 256])
@pytest.mark.parametrize("words", [0, 1])
def test_admitted_sizes_fit_the_lds(rule, pairs, words):
    refused = 0
    for Lkv in range(1, 300):
        for Lq in list(range(1, 800)) + [4096]:
            takes = bool(rule.takes(Lq, Lkv, pairs, words))
            assert not takes or rule.lds(Lq, Lkv, words) <= 160 * 1024, (Lq, Lkv)
            shape = Lkv <= 256 and (Lq <= 3 * Lkv or Lq <= 64) and (Lq <= 256 or pairs >= 256)
            assert takes <= shape
            refused += shape and not takes
    assert refused == (0 if pairs < 256 or not words else sum(1 for Lkv in range(225, 257) for Lq in range(705, 3 * Lkv + 1)))


def test_lds_of_the_largest_sizes(rule):
    # 8 blocks of K rows and dS, two tiles of Q and dO, 12 tiles of statistics, 8 x 32 words for each 64 queries
    assert rule.lds(768, 256, 0) == 8 * (4096 + 8192) + 32768 + 12 * 768
    assert rule.lds(720, 255, 1) == 8 * (4096 + 8192) + 32768 + 12 * 768 + 8 * 32 * 8 * 12
    assert rule.lds(128, 128, 1) == 4 * (4096 + 4096) + 16384 + 12 * 128 + 4 * 32 * 8 * 2
