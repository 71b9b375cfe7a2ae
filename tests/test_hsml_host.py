"""Host (g++) test of mhip_hsml.hpp, the float64 refinement of the smoothing
length: rows where a few particles near the query carry nearly all of n(h), so
that it is flat at the root and an approximate h is far off, against
bisection.  The tolerance is what the sums can tell: n(h) to 16 eps a term, over
the slope p = h n'(h), and 1e-13 for the last step."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

SRC = """
#include "%s"
extern "C" double refine(double h, int k, int dim, const double *r) {
    return mhip::hsml_refine(
        h, k, dim,
        [&](double x) {
            mhip::HsmlSums s;
            for (int j = 0; j < k; j++) s.add(r[j] * (1.0 / x));
            return s;
        },
        [&] {  // two parts, joined
            mhip::HsmlRange a, b;
            for (int j = 0; j < k; j++) (j %% 3 ? a : b).add(r[j]);
            a.join(b);
            return a;
        });
}
extern "C" double slope(double h, int k, int dim, const double *r) {
    mhip::HsmlSums s;
    for (int j = 0; j < k; j++) s.add(r[j] / h);
    return mhip::hsml_halley(s, k, dim).p;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    d = tmp_path_factory.mktemp("hsml")
    (d / "h.cpp").write_text(SRC % os.path.join(root, "meshoid_amd", "csrc", "mhip_hsml.hpp"))
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-o", d / "h.so", d / "h.cpp"],
                   check=True)
    L = ctypes.CDLL(str(d / "h.so"))
    arr = np.ctypeslib.ndpointer(dtype=np.float64, flags="C_CONTIGUOUS")
    for f in (L.refine, L.slope):
        f.argtypes, f.restype = [ctypes.c_double, ctypes.c_int, ctypes.c_int, arr], ctypes.c_double
    return L


NORM = {1: 8 / 3, 2: 40 / 7, 3: 32 / 3}


def bisect(r, dim):
    r = r.astype(np.longdouble)
    k = len(r)
    lo, hi = r[1], r[-1] / (1 - (2 * np.longdouble(NORM[dim])) ** (np.longdouble(-1) / 3))
    for _ in range(110):
        h = (lo + hi) / 2
        q = r / h
        w = np.where(q <= 0.5, 1 - 6 * q * q * (1 - q), 2 * np.clip(1 - q, 0, None) ** 3)
        lo, hi = (lo, h) if w.sum() * NORM[dim] > k else (h, hi)
    return float((lo + hi) / 2)


# k, dim, particles near the query and how near (over r_k)
CASES = [(32, 3, 0, 0.0), (32, 3, 2, 0.003), (32, 3, 2, 1e-4), (32, 3, 3, 0.003), (64, 3, 5, 0.003), (64, 3, 6, 0.003),
         (64, 3, 5, 1e-4), (20, 2, 2, 0.003), (20, 2, 3, 0.003), (100, 3, 8, 0.003), (4, 1, 0, 0.0), (11, 3, 0, 0.0)]


@pytest.mark.parametrize("k,dim,near,width", CASES)
def test_refined_root(lib, k, dim, near, width):
    rng = np.random.default_rng(k * 10 + near)
    worst = 0.0
    for t in range(300):
        r = rng.random(k) ** (1 / dim)
        r[0] = 0.0
        r[1 : 1 + near] = width * rng.random(near)
        r.sort()
        want = bisect(r, dim)
        tol = 1e-13 + 16 * np.finfo(float).eps * k / max(lib.slope(want, k, dim, r), 1e-300)
        for off in (0.0, 1e-6, -1e-5, 2e-4, -5e-3, 0.2, -0.4):
            h = lib.refine(float(np.float32(want * (1 + off))), k, dim, r)
            assert abs(h - want) <= tol * want, (t, off)
            worst = max(worst, abs(h - want) / want)
    if width != 1e-4:
        assert worst <= 1e-10


@pytest.mark.parametrize("k,dim,near", [(2, 3, 0), (8, 3, 0), (10, 3, 0), (5, 2, 0), (32, 3, 5), (64, 3, 20), (20, 2, 9)])
def test_no_root_ends_at_the_bracket(lib, k, dim, near):
    """n(h) > k throughout: the reference's bisection runs down to the
    distance of the first neighbour."""
    rng = np.random.default_rng(k + near)
    for _ in range(100):
        r = rng.random(k) ** (1 / dim)
        r[0] = 0.0
        r[1 : 1 + near] = 1e-3 * (1 + 1e-3 * rng.random(near))
        r.sort()
        # all of weight 1 at a larger h than r_1 only if n(r_1) > k there
        q = r / r[1]
        w = np.where(q <= 0.5, 1 - 6 * q * q * (1 - q), 2 * np.clip(1 - q, 0, None) ** 3)
        if w.sum() * NORM[dim] < k:
            continue
        for off in (2.5e-7, 0.1, 3.0):
            assert lib.refine(float(np.float32(r[1] * (1 + off))), k, dim, r) == r[1]


def test_flat_stretch_keeps_h(lib):
    """A query and two particles at its place are 32 neighbours for any h below
    the next distance: every such h is a root, and the given one stays."""
    r = np.concatenate([np.zeros(3), np.sort(0.5 + 0.5 * np.random.default_rng(0).random(29))])
    for h in (0.01, 0.3, 0.49):
        assert lib.refine(h, 32, 3, r) == h
