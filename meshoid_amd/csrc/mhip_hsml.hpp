// The smoothing length in float64: HsmlIter's root, norm sum_j W(r_j / h) = k
// (src/meshoid/kernel_density.py:14-57), from an approximate h.
// Header-only and usable from host code (a CPU unit test compiles it with g++).
#pragma once
#include <math.h>

#if !defined(MHIP_HD)
#if defined(__HIPCC__)
#define MHIP_HD __host__ __device__ __forceinline__
#else
#define MHIP_HD inline
#endif
#endif

namespace mhip {

// norm_d of kernel_density.py:26-31 and the bracket factor of :35
MHIP_HD double hsml_norm(int dim) { return dim == 3 ? 32.0 / 3 : (dim == 2 ? 40.0 / 7 : 8.0 / 3); }
MHIP_HD double hsml_bound_coeff(int dim) {
    return dim == 3 ? 1.5638742363463305 : (dim == 2 ? 1.7984058958344455 : 2.33839974837265);
}

// The float32 solve leaves a relative error of ~1e-6 to 1e-5; the
// derivative fits are sensitive to h through the weights of the outermost neighbours (d ln W / d ln h =
// 3q / (1 - q) as q -> 1), so a 2.4e-7 error of h moves second-order
// derivatives by up to ~6e-5.  The spline as truncated powers, W = 2 a^3 - b^3
// with a = (1 - q)_+ and b = (1 - 2q)_+, gives W' = -6 (a^2 - b^2) and
// W'' = 12 a - 24 b without branches, so Halley's step (cubic: third
// derivatives of W are bounded) costs two more operations per neighbour than
// Newton's and leaves h at the rounding level of the float64 sums.
struct HsmlSums {
    double w = 0.0, d1 = 0.0, d2 = 0.0;  // sums of W / 2, -W' q / 6, W'' q^2 / 12
    MHIP_HD void add(double q) {
        const double a = fmax(1.0 - q, 0.0), b = fmax(fma(-2.0, q, 1.0), 0.0);
        const double aa = a * a, bb = b * b, qc = fmin(q, 1.0);
        w += fma(-0.5 * b, bb, a * aa);
        const double t = (aa - bb) * qc;
        d1 += t;
        d2 = fma(fma(-2.0, b, a) * qc, qc, d2);
    }
};

struct HsmlStep {
    double f, p, rel;  // n(h) - k, h n'(h), the step over h
};

MHIP_HD HsmlStep hsml_halley(const HsmlSums &s, int k, int dim) {
    const double norm = hsml_norm(dim);
    // n(h) = norm sum W(r_j / h) grows with h; c = h^2 n''(h)
    HsmlStep r;
    r.f = norm * (2.0 * s.w) - (double)k;
    r.p = norm * 6.0 * s.d1;
    const double c = norm * 12.0 * (s.d2 - s.d1);
    r.rel = 2.0 * r.f * r.p / (2.0 * r.p * r.p - r.f * c);
    return r;
}

// Whether the step is the last.  It leaves about rel^3 h^3 n''' / (6 p), and
// h^3 |n'''| <= 12 norm k: at most 1e-13 h.  One step from the float32 solve is
// enough in all rows of a random set; where nearly all of n comes from a few
// particles close to the query, as a pair within 0.3% of r_k for k = 32 in
// 3D, n is flat at the root, p is small and float32 cannot tell h: one step from
// there left errors to 6e-4, and to 0.2 with the pair within 1e-4.
MHIP_HD bool hsml_last(const HsmlStep &s, int k, int dim) {
    const double x = fabs(s.rel);
    return s.p > 0.0 && x <= 1e-4 && x * x * x * (2.0 * hsml_norm(dim) * k) <= 1e-13 * s.p;
}

// The root within the reference's bracket [lo, hi] = [r_1, c_d r_(k-1)], from h:
// Halley's steps, halving the bracket where they leave it or converge
// slowly; lo where n(lo) > k already (few neighbours or many coincident ones:
// the reference's bisection ends there).  sums_at(h): the sums over the members.
template <typename S>
MHIP_HD double hsml_bracketed(double lo, double hi, double h, int k, int dim, S sums_at) {
    if (lo > 0.0 && hsml_halley(sums_at(lo), k, dim).f >= 0.0) return lo;
    if (!(h > lo && h < hi)) h = 0.5 * (lo + hi);
    for (int it = 0; it < 160; it++) {
        const HsmlStep s = hsml_halley(sums_at(h), k, dim);
        if (s.f == 0.0) return h;
        if (s.f > 0.0)
            hi = h;
        else
            lo = h;
        double hn = h - h * s.rel;
        if (hsml_last(s, k, dim)) return fmin(fmax(hn, lo), hi);
        if (!(s.p > 0.0 && hn > lo && hn < hi) || (it >= 8 && (it & 1))) hn = 0.5 * (lo + hi);
        if (!(hn > lo && hn < hi)) return hn;  // the bracket has collapsed
        h = hn;
    }
    return h;
}

// the two smallest and the largest of a row's distances: the bracket
struct HsmlRange {
    double r0 = INFINITY, r1 = INFINITY, rk = 0.0;
    MHIP_HD void add(double r) {
        r1 = fmin(r1, fmax(r0, r));
        r0 = fmin(r0, r);
        rk = fmax(rk, r);
    }
    // with those of other members
    MHIP_HD void join(const HsmlRange &o) {
        r1 = fmin(fmin(r1, o.r1), fmax(r0, o.r0));
        r0 = fmin(r0, o.r0);
        rk = fmax(rk, o.rk);
    }
};

// whether n(h) > k for all h: the query itself, of weight 1, is k neighbours.
// The bracket's lower end r_1 is then the result.
MHIP_HD bool hsml_rootless(int k, int dim) { return (double)k <= hsml_norm(dim); }

// The refinement from an approximate h: one step where that is enough (see
// hsml_last), else within the bracket.  range(): the row's HsmlRange.
template <typename S, typename R>
MHIP_HD double hsml_refine(double h, int k, int dim, S sums_at, R range) {
    if (!hsml_rootless(k, dim)) {
        const HsmlStep s = hsml_halley(sums_at(h), k, dim);
        if (hsml_last(s, k, dim)) return h - h * s.rel;
    }
    const HsmlRange r = range();
    return hsml_bracketed(r.r1, hsml_bound_coeff(dim) * r.rk, h, k, dim, sums_at);
}

}  // namespace mhip
