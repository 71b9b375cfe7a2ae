"""Host (g++) test of merge_sorted<K, 16>, the merge of a sorted run of 16 into
a sorted list of K slots: every list length the kNN uses, random values, ties,
infinities and the sentinel slots (-1) of lists shorter than K."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

SRC = """
#include "%s"
#define M(K) extern "C" void merge##K(float *A, float *S) { \\
    mhip::oddeven_sort<16>(*reinterpret_cast<float(*)[16]>(S)); \\
    mhip::merge_sorted<K, 16>(*reinterpret_cast<float(*)[K]>(A), *reinterpret_cast<float(*)[16]>(S)); }
M(17) M(21) M(33) M(65)
"""


@pytest.mark.parametrize("K", [17, 21, 33, 65])
def test_merge_keeps_the_smallest(tmp_path, K):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, lib = tmp_path / "m.cpp", tmp_path / "m.so"
    src.write_text(SRC % os.path.join(root, "meshoid_amd", "csrc", "mhip_sortnet.hpp"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, src], check=True)
    f = getattr(ctypes.CDLL(str(lib)), f"merge{K}")
    f.argtypes = [np.ctypeslib.ndpointer(dtype=np.float32, flags="C_CONTIGUOUS")] * 2
    rng = np.random.default_rng(K)
    for trial in range(2000):
        a, s = rng.random(K).astype(np.float32), rng.random(16).astype(np.float32)
        if trial % 3 == 1:
            a, s = np.round(a * 5).astype(np.float32), np.round(s * 5).astype(np.float32)
        if trial % 4 == 2:
            a[rng.integers(1, K):] = np.inf
            s[rng.integers(0, 16):] = np.inf
        if trial % 5 == 3:
            a[: rng.integers(1, K)] = -1
        a.sort()
        want = np.sort(np.concatenate([a, s]))[:K]
        f(a, s)
        assert np.array_equal(a, want), trial
