"""The unpack step of the packed formats (csrc/kv_codes.h, compiled for the host): for every B = 4..7 and every code
at every value position (between random neighbours), the magic pair read as fp16 plus its bias is the signed code exactly, in the order
pair_at states, whatever the bits around the word's high field."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen38-megakernel_amd", "csrc")
SRC = """
#include "kv_codes.h"
#define F(B) extern "C" void pairs##B(const uint32_t * W, const uint32_t * hd, int idx, uint32_t * p, int n) { \\
    for (int i = 0; i < n; i++) { uint32_t q[4]; qkv::code_pairs<B>(W[i], hd[i], idx, q); for (int k = 0; k < 4; k++) p[4 * i + k] = q[k]; } } \\
    extern "C" float lo##B() { return qkv::CodeBias<B>::lo; } extern "C" float hi##B() { return qkv::CodeBias<B>::hi; }
F(4) F(5) F(6) F(7)
extern "C" int at(int i, int e) { return qkv::pair_at(i, e); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("codes")
    (d / "c.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", str(d / "c.cpp"), "-o", str(d / "c.so")], check=True)
    return ctypes.CDLL(str(d / "c.so"))


@pytest.mark.parametrize("B", [4, 5, 6, 7])
def test_pairs_are_the_codes(lib, B):
    hb, rng = B - 4, np.random.default_rng(B)
    parts = {4: [0], 5: [0, 1, 2, 3], 6: [0, 1], 7: [0]}[B]
    codes = rng.integers(0, 1 << B, (1 << 16, 8), dtype=np.uint64)
    for k in range(8):  # every code at every value position
        codes[(k << B):((k + 1) << B), k] = np.arange(1 << B)
    n = codes.shape[0]
    W = np.zeros(n, np.uint64)
    H = np.zeros(n, np.uint64)
    for k in range(8):
        W |= (codes[:, k] & 15) << np.uint64(8 * (k % 4) + 4 * (k // 4))
        H |= (codes[:, k] >> np.uint64(4)) << np.uint64(hb * k)
    for idx in parts:
        hd = rng.integers(0, 1 << 32, n, dtype=np.uint64)  # neighbouring fields: any bits
        w, sh = {4: (0, 0), 5: (8, 8 * idx), 6: (16, 16 * idx), 7: (24, 0)}[B]
        hd = (hd & ~np.uint64(((1 << w) - 1) << sh)) | (H << np.uint64(sh))
        W32, hd32, p = W.astype(np.uint32), hd.astype(np.uint32), np.zeros((n, 4), np.uint32)
        getattr(lib, f"pairs{B}")(*(ctypes.c_void_p(x.ctypes.data) for x in (W32, hd32)), idx, ctypes.c_void_p(p.ctypes.data), n)
        lib_lo, lib_hi = getattr(lib, f"lo{B}"), getattr(lib, f"hi{B}")
        lib_lo.restype = lib_hi.restype = ctypes.c_float
        halves = p.view(np.float16).reshape(n, 4, 2)
        for i in range(4):
            bias = lib_lo() if i < 2 else lib_hi()
            assert np.float16(bias) == bias
            for e in range(2):
                got = halves[:, i, e] - np.float16(bias)
                assert np.array_equal(got.astype(np.int64), codes[:, lib.at(i, e)].astype(np.int64) - (1 << (B - 1))), (idx, i, e)
