"""Host (g++) test of knn_wave_serves: a set that the one-wavefront-per-query
kernel takes fits one launch (16 threads a query, fewer than 2^32), and the
lines elsewhere lie where its comment says."""
import ctypes
import os
import subprocess

import pytest

SRC = """
#include "%s"
extern "C" int splits(int64_t n, int64_t nq, int k, int dim, int per) {
    return mhip::knn_splits(n, nq, k, dim, per);
}
extern "C" int serves(int64_t n, int64_t nq, int k, int dim, int per) {
    return mhip::knn_wave_serves(n, nq, k, dim, per);
}
"""


@pytest.fixture(scope="module")
def serves(tmp_path_factory):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    d = tmp_path_factory.mktemp("serves")
    (d / "s.cpp").write_text(SRC % os.path.join(root, "meshoid_amd", "csrc", "mhip_knn_rules.hpp"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", d / "s.so", d / "s.cpp"], check=True)
    L = ctypes.CDLL(str(d / "s.so"))
    for f in (L.serves, L.splits):
        f.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    g = lambda *a: bool(L.serves(*a))
    g.splits = lambda *a: bool(L.splits(*a))
    return g


def test_one_launch_holds_the_set(serves):
    for n in (1, 1000, 100000, 1 << 20, (1 << 28) - 1, 1 << 28, 1 << 31):
        for nq in (1, 32768, 32769, 1 << 20, (1 << 28) - 16, 1 << 28, (1 << 28) + 5, 1 << 30, 1 << 32):
            for k in (2, 32, 33, 64, 65, 128):
                for dim in (1, 2, 3):
                    for per in (0, 1):
                        # (a split set runs both kernels over every slot)
                        if serves(n, nq, k, dim, per) or serves.splits(n, nq, k, dim, per):
                            assert 16 * nq < 1 << 32 and 4 * n < 1 << 32


def test_lines(serves):
    for dim, most in ((3, 100000), (2, 45000), (1, 45000)):
        for k, per, f in ((32, 0, 1), (33, 0, 3), (32, 1, 3), (64, 1, 9)):
            assert serves(most * f, most * f, k, dim, per)
            assert not serves(most * f + 1, most * f + 1, k, dim, per)
    assert serves(1 << 24, 1 << 24, 65, 3, 0) and not serves(1 << 28, 1 << 28, 65, 3, 0)
    # a part of a large set: whole while small, else wavefront by wavefront, and
    # from a quarter on (a fifth for k <= 32) as the set itself
    for k, end in ((32, (1 << 24) // 5), (64, 1 << 22)):
        assert serves(1 << 24, 1 << 20, k, 3, 0) and not serves.splits(1 << 24, 1 << 20, k, 3, 0)
        for nq in ((1 << 20) + 1, end - 1):
            assert not serves(1 << 24, nq, k, 3, 0) and serves.splits(1 << 24, nq, k, 3, 0)
        for nq in (end, 1 << 22, 1 << 24):
            assert not serves(1 << 24, nq, k, 3, 0) and not serves.splits(1 << 24, nq, k, 3, 0)
    assert not serves.splits(1 << 24, 1 << 21, 65, 3, 0) and not serves.splits(1 << 28, 1 << 21, 32, 3, 0)
