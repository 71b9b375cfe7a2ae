// Exact k-nearest-neighbour search with one wavefront per query, the smoothing
// length and the member list (the results of k_knn_main in mhip_knn.hip, for
// the sizes given at knn_wave_serves in mhip_knn_rules.hpp).
//
// The main kernel gives each lane a query and keeps its k + 1 smallest
// distances in registers: a list insertion costs k + 1 instructions, and few
// queries leave most of the chip idle while one wavefront's dependent loads
// run one after another.  Here the 64 lanes share one query:
//   fill    the leaves around the query's own leaf, 64 particles at a time;
//   bound   candidates (float32 d2, sorted index) are appended to a buffer in
//           LDS; the bound, at least the (k+1)-th smallest distance so far,
//           comes from bisecting the float bits with one ballot per 64
//           candidates and step (no sorting, no list), and the buffer is
//           compacted to the candidates below it;
//   walk    inside out from the query's leaf: the ancestor two levels up, its
//           ancestor two levels up, ...; a node's 64 grandchildren (contiguous
//           in the heap numbering) are tested by the 64 lanes at once, and
//           surviving leaves are scanned four at a time, nearest first;
//   result  the k-th and (k+1)-th distances by the same bisection, members
//           compacted, smoothing length with one neighbour (two for k > 64)
//           per lane and wave-wide sums.
// The same float32 distances, box tests and ambiguity rule as the main
// kernel, so the member sets are the same; ambiguous rows go to the resolver.
#include <float.h>

#include <algorithm>
#include <type_traits>

#include "mhip_knn.hpp"

namespace mhip {

constexpr int KW_WAVES = 4;  // wavefronts per block
constexpr int64_t KW_LIST_OPEN = 2048, KW_LIST_PER = 65536;  // grids over deferred wavefronts
constexpr int KW_LEAFQ = 68;  // leaf queue: a block of 64 and up to 3 left over

// ---- reductions over each row of 16 lanes by DPP rotations, result in every
// lane of the row
template <int N>
MHIP_DEV float ror_f(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + N, 0xf, 0xf, true));
}
template <int N>
MHIP_DEV double ror_d(double x) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x120 + N, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x120 + N, 0xf, 0xf, true));
}
MHIP_DEV float row_sum(float x) {
    x += ror_f<8>(x);
    x += ror_f<4>(x);
    x += ror_f<2>(x);
    x += ror_f<1>(x);
    return x;
}
MHIP_DEV double row_sum(double x) {
    x += ror_d<8>(x);
    x += ror_d<4>(x);
    x += ror_d<2>(x);
    x += ror_d<1>(x);
    return x;
}
MHIP_DEV float row_min(float x) {
    x = fminf(x, ror_f<8>(x));
    x = fminf(x, ror_f<4>(x));
    x = fminf(x, ror_f<2>(x));
    return fminf(x, ror_f<1>(x));
}

MHIP_DEV void row_join(HsmlRange &r) {
    r.join(HsmlRange{ror_d<8>(r.r0), ror_d<8>(r.r1), ror_d<8>(r.rk)});
    r.join(HsmlRange{ror_d<4>(r.r0), ror_d<4>(r.r1), ror_d<4>(r.rk)});
    r.join(HsmlRange{ror_d<2>(r.r0), ror_d<2>(r.r1), ror_d<2>(r.rk)});
    r.join(HsmlRange{ror_d<1>(r.r0), ror_d<1>(r.r1), ror_d<1>(r.rk)});
}

MHIP_DEV int lane_rank(uint64_t m) {  // set bits of m below this lane
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// element p of a float array: with fewer than 2^30 of them (OFF = uint32_t)
// through a 32-bit byte offset from a scalar base
template <typename OFF>
MHIP_DEV float ld32(const float *b, uint32_t p) {
    return *(const float *)((const char *)b + (size_t)((OFF)p << 2));
}

template <int NR>
MHIP_DEV int count_le(const float (&v)[NR], float t, int nr) {
    int c = __popcll(__ballot(v[0] <= t)) + __popcll(__ballot(v[1] <= t));
    if (nr > 2) c += __popcll(__ballot(v[2] <= t)) + __popcll(__ballot(v[3] <= t));
    if (NR > 4 && nr > 4) c += __popcll(__ballot(v[NR - 2] <= t)) + __popcll(__ballot(v[NR - 1] <= t));
    return c;
}

// A threshold t with lo_n <= count(v <= t) <= hi_n, from count(v <= top) = n
// >= lo_n; when float32 ties leave no such t, the smallest t with count >=
// lo_n.  The count grows as t^(dim/2) in a locally uniform density: the first
// guess follows that, the next ones interpolate, and after a few the float
// bits are bisected.
template <int NR>
MHIP_DEV float threshold(const float (&v)[NR], float top, int n, int nr, int lo_n, int hi_n, int dim, int &got) {
    got = n;
    if (n <= hi_n) return top;
    uint32_t hi = uniform(__float_as_uint(top)), lo = 0u;
    int cl = 0, ch = n;
    if (count_le<NR>(v, 0.f, nr) >= lo_n) {
        got = count_le<NR>(v, 0.f, nr);
        return 0.f;
    }
    const float aim = 0.5f * (float)(lo_n + hi_n);
    float g = top * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(aim / (float)n) * (2.0f / (float)dim));
    for (int it = 0; hi - lo > 1u; it++) {
        uint32_t mid = uniform(__float_as_uint(g));
        if (it >= 6 || !(mid > lo && mid < hi)) mid = lo + (hi - lo) / 2u;
        const int c = count_le<NR>(v, __uint_as_float(mid), nr);
        if (c < lo_n) {
            lo = mid;
            cl = c;
        } else {
            hi = mid;
            ch = c;
            if (c <= hi_n) break;
        }
        const float fl = __uint_as_float(lo), fh = __uint_as_float(hi);
        g = fl + (fh - fl) * ((aim - (float)cl) * __builtin_amdgcn_rcpf((float)(ch - cl)));
    }
    got = ch;
    return __uint_as_float(hi);
}

// Search for one query.  s_c: the wavefront's candidate buffer (64 NR entries
// of squared distance and sorted index); s_lq: its leaf queue; s_stk: its walk stack.  Members go to
// s_out[j * ncol + col], j < k; returns the row's status bits, tau and tau1 =
// the k-th and (k+1)-th squared distance.
template <int NR, bool PER, bool P64, typename OFF>
MHIP_DEV int32_t wave_search(const KnnArgs &a, int64_t slot, uint32_t qp, uint2 *s_c, uint32_t *s_lq,
                             uint32_t (*s_stk)[4], uint32_t *s_out, int col, int ncol, float &tau_out, float &tau1_out) {
    constexpr int CAP = 64 * NR;
    const int lane = threadIdx.x & (WAVE - 1);
    const TreeView &t = a.t;
    const int k = a.k;
    const QPos q = load_q<P64>(t, qp);
    const uint32_t first_leaf = (uint32_t)t.first_leaf, nleaf = (uint32_t)t.nleaf;
    const uint32_t lc = qp / LEAF;
    int m = 0;               // candidates in the buffer
    int next = 0;            // buffer fill at which the bound is tightened
    // at least the (k+1)-th smallest d2 found so far.  Squared distances that
    // overflow float32 are no candidates (as in the main kernel): a row with
    // fewer than k others goes to the resolver
    float bound = FLT_MAX;

    auto load = [&](float (&v)[NR], uint32_t (&ix)[NR], int nr) {
        lds_order();
#pragma unroll
        for (int r = 0; r < NR; r++) v[r] = INFINITY;
#pragma unroll
        for (int r = 0; r < NR; r += 2) {
            if (r < nr) {
                const uint2 x = s_c[r * 64 + lane], y = s_c[r * 64 + 64 + lane];
                v[r] = r * 64 + lane < m ? __uint_as_float(x.x) : INFINITY;
                v[r + 1] = r * 64 + 64 + lane < m ? __uint_as_float(y.x) : INFINITY;
                ix[r] = x.y;
                ix[r + 1] = y.y;
            }
        }
        lds_order();
    };
    // candidates that pass move to the buffer's entries from, from + 1, ...
    // (in order, entries below cap only)
    auto compact = [&](const float (&v)[NR], const uint32_t (&ix)[NR], int nr, int from, auto pass, int cap) {
        int c = from;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            if (r >= nr) break;
            const bool keep = pass(v[r]);
            const uint64_t b = __ballot(keep);
            const int pos = c + lane_rank(b);
            if (keep && pos < cap) s_c[pos] = make_uint2(__float_as_uint(v[r]), ix[r]);
            c += __popcll(b);
        }
        lds_order();
        return c;
    };
    // a bound that keeps at least k + 1 candidates (m >= k + 1) and few more;
    // the buffer is compacted to them when it could not take another 64
    auto tighten = [&]() {
        float v[NR];
        uint32_t ix[NR];
        const int nr = (m + 63) >> 6;
        load(v, ix, nr);
        float top = bound;
        int n = m;
        if (top < FLT_MAX) {
            n = count_le<NR>(v, top, nr);
        } else {
            top = 0.f;
#pragma unroll
            for (int r = 0; r < NR; r++) top = fmaxf(top, v[r] < INFINITY ? v[r] : 0.f);
            top = wave_max_f(top);
        }
        int got;
        bound = threshold<NR>(v, top, n, nr, k + 1, k + 1 + k / 4, a.dim, got);
        if (m > CAP - 128) {
            if (got <= CAP - 64) {
                m = compact(v, ix, nr, 0, [&](float x) { return x <= bound; }, CAP);
            } else {
                // float32 ties at the bound fill the buffer: the (at most k)
                // closer ones first, then ties while another 64 still fit
                // (the row is ambiguous, and the resolver rebuilds it)
                const int c = compact(v, ix, nr, 0, [&](float x) { return x < bound; }, CAP);
                compact(v, ix, nr, c, [&](float x) { return x == bound; }, CAP - 64);
                m = CAP - 64;
            }
        }
        next = m + 40;
    };
    // 64 particles, one per lane
    auto append = [&](float d2, uint32_t p, bool in) {
        const bool pass = in && d2 <= bound;  // never the NaN of padding
        const uint64_t b = __ballot(pass);
        const int pos = m + lane_rank(b);
        if (pass) s_c[pos] = make_uint2(__float_as_uint(d2), p);
        m += __popcll(b);
    };
    auto dist = [&](uint32_t p, auto per) {
        constexpr bool WRAP = decltype(per)::value;
        return dist2<WRAP, P64>(t, q, ld32<OFF>(t.sx, p), ld32<OFF>(t.sy, p), ld32<OFF>(t.sz, p),
                                P64 ? ld32<OFF>(t.lx, p) : 0.f, P64 ? ld32<OFF>(t.ly, p) : 0.f,
                                P64 ? ld32<OFF>(t.lz, p) : 0.f);
    };

    // fill: the leaves around the query's own (more than k + 1 candidates)
    const uint32_t want = k < 48 ? 8u : (k <= 64 ? 12u : 16u);
    const uint32_t ninit = min(want, nleaf);
    const uint32_t i0 = min(lc > ninit / 2 ? lc - ninit / 2 : 0u, nleaf - ninit);
    for (uint32_t l = 0; l < ninit; l += 4) {
        const uint32_t e = l * LEAF + lane;
        const bool in = e < ninit * LEAF;
        const uint32_t p = i0 * LEAF + (in ? e : 0u);
        append(dist(p, std::integral_constant<bool, PER>()), p, in);
    }
    next = k + 1;
    if (m > k) tighten();

    // the rest of the tree.  per: whether offsets need the periodic image.
    auto walk = [&](auto per) {
        constexpr bool WRAP = decltype(per)::value;
        int nl = 0;  // leaves in the queue
        // scans queued leaves four at a time, one per row of 16 lanes; fewer
        // than four stay queued unless all is set
        auto scan = [&](bool all) {
            int at = 0;
            lds_order();
            while (nl - at >= 4 || (all && at < nl)) {
                if (m > CAP - 64 || m >= next) {
                    if (m > k) tighten();
                }
                const int e = at + (lane >> 4);
                const uint32_t p = s_lq[min(e, nl - 1)] * LEAF + (lane & (LEAF - 1));
                append(dist(p, per), p, e < nl);
                at += 4;
            }
            nl = max(nl - at, 0);
            if (at > 0 && nl > 0) {
                const uint32_t x = s_lq[at + min(lane, nl - 1)];
                lds_order();
                if (lane < nl) s_lq[lane] = x;
            }
        };
        auto queue = [&](bool sel, uint32_t li) {
            const uint64_t b = __ballot(sel);
            if (sel) s_lq[nl + lane_rank(b)] = li;
            nl += __popcll(b);
        };
        auto test = [&](uint32_t base, int cnt) {
            const bool ok =
                lane < cnt && node_d2<WRAP>(t, q, base + (lane < cnt ? lane : 0)) <= bound * PRUNE_REL;
            return __ballot(ok);
        };
        // leaves base .. base + cnt - 1 (heap numbers) into the queue; near:
        // the nearer ones are scanned before the others are chosen
        auto leaves = [&](uint32_t base, int cnt, bool near) {
            const uint32_t li = base + lane - first_leaf;
            bool ok = lane < cnt && li < nleaf && li - i0 >= ninit;
            const float g = ok ? node_d2<WRAP>(t, q, base + lane) : INFINITY;
            if (near) {
                const bool sel = ok && g <= 0.25f * bound;
                queue(sel, li);
                scan(true);
                if (m > next - 24 && m > k) tighten();
                ok = ok && !sel;
            }
            queue(ok && g <= bound * PRUNE_REL, li);
            scan(false);
        };
        uint32_t own = first_leaf + lc;
        int lev = t.depth;
        while (lev > 0) {
            const int step = lev >= 2 ? 2 : 1;
            const uint32_t par = (own - 1) >> 3;
            const uint32_t top = step == 2 ? (par - 1) >> 3 : par;
            const uint32_t base0 = step == 2 ? 64u * top + 9u : 8u * top + 1u;
            const int cnt = step == 2 ? 64 : 8;
            if (lev == t.depth) {
                leaves(base0, cnt, true);
            } else {
                uint32_t base = base0;
                uint64_t mask = test(base, cnt) & ~(1ull << (own - base));
                int flev = lev, f = 0;
                while (true) {
                    if (mask == 0) {
                        if (f == 0) break;
                        f--;
                        flev -= 2;
                        lds_order();
                        base = uniform(s_stk[f][0]);
                        mask = (uint64_t)uniform(s_stk[f][1]) | (uint64_t)uniform(s_stk[f][2]) << 32;
                        continue;
                    }
                    const uint32_t node = base + __builtin_ctzll(mask);
                    mask &= mask - 1;
                    const uint32_t sub = 64u * node + 9u;
                    if (flev + 2 == t.depth) {
                        leaves(sub, 64, false);
                        continue;
                    }
                    if (lane == 0) {
                        s_stk[f][0] = base;
                        s_stk[f][1] = (uint32_t)mask;
                        s_stk[f][2] = (uint32_t)(mask >> 32);
                    }
                    f++;
                    flev += 2;
                    base = sub;
                    mask = test(base, 64);
                }
            }
            own = top;
            lev -= step;
        }
        scan(true);
    };
    if (PER) {
        // a ball that does not reach the box's faces meets no image: offsets
        // beyond half the box are then beyond the bound either way
        const float r = __builtin_sqrtf(bound) * 1.001f + t.slack;
        const float qx[3] = {q.x, q.y, q.z};
        bool inner = r < t.half;
#pragma unroll
        for (int c = 0; c < 3; c++) inner = inner && (c >= a.dim || (qx[c] - r > 0.f && qx[c] + r < t.box));
        if (__any(!inner)) walk(std::true_type());
        else walk(std::false_type());
    } else {
        walk(std::false_type());
    }

    // the k-th and (k+1)-th distances
    float v[NR];
    uint32_t ix[NR];
    const int nr = (m + 63) >> 6;
    load(v, ix, nr);
    float tau = INFINITY, tau1 = INFINITY;
    int32_t st = 0;
    if (m >= k) {
        float top = 0.f;
#pragma unroll
        for (int r = 0; r < NR; r++) top = fmaxf(top, v[r] <= bound && v[r] < INFINITY ? v[r] : 0.f);
        top = wave_max_f(top);
        int got;
        const float lim = threshold<NR>(v, top, count_le<NR>(v, top, nr), nr, k, k, a.dim, got);
        float below = 0.f, above = INFINITY;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const bool in = v[r] <= lim;
            below = fmaxf(below, in ? v[r] : 0.f);
            above = fminf(above, in ? INFINITY : v[r]);
        }
        tau = wave_max_f(below);
        tau1 = got > k ? tau : wave_min_f(above);  // more than k at or below: a float32 tie at the k-th
    }
    if (tau1 <= tau * (1.0f + AMBIG_REL)) st |= ST_AMBIGUOUS;
    int cnt;
    if (tau1 > tau) {
        cnt = min(compact(v, ix, nr, 0, [&](float x) { return x <= tau; }, CAP), k);
    } else {
        // float32 ties at the k-th: every closer one, then ties up to k (with
        // fewer than k candidates tau is +inf, which fills the empty places)
        const int c = compact(v, ix, nr, 0, [&](float x) { return x < tau; }, k);
        cnt = min(compact(v, ix, nr, min(c, k), [&](float x) { return x == tau && x < INFINITY; }, k), k);
    }
    if (cnt != k) st |= ST_COUNT;
    for (int j = lane; j < k; j += 64) {
        const uint2 x = s_c[j];
        s_out[j * ncol + col] = j < cnt ? x.y : qp;
        if (a.nl_d2) a.nl_d2[(int64_t)j * a.nq + slot] = j < cnt ? __uint_as_float(x.x) : INFINITY;
    }
    lds_order();
    if (lane == 0) a.tau[slot] = tau;
    tau_out = tau;
    tau1_out = tau1;
    return st;
}

// Smoothing lengths of the wavefront's up to four queries, one per row of 16
// lanes, MPL members per lane (16 MPL >= k): float64 distances of the members,
// safeguarded float32 Newton, one float64 step.  The same
// control flow as the main kernel's solve.
// SEED: a Newton seed per row (a.seed_h) may be given.
template <int MPL, bool PER, bool P64, bool SEED>
MHIP_DEV void row_hsml(const KnnArgs &a, bool on, int64_t slot, uint32_t qp, float tau, int32_t st,
                       const uint32_t *s_out, int col, int ncol) {
    const int rl = threadIdx.x & 15;
    const TreeView &t = a.t;
    const int k = a.k;
    const QPos q = load_q<P64>(t, qp);
    double r64[MPL];
    float mn = 3e38f;
#pragma unroll
    for (int u = 0; u < MPL; u++) {
        const int j = u * 16 + rl;
        r64[u] = 1e300;
        if (j < k) r64[u] = member_dist<PER, P64, false>(t, q, s_out[j * ncol + col]);
        mn = fminf(mn, fminf((float)r64[u], 3e38f));
    }
    // bracket [r_1, c_d r_(k-1)] of the reference: r_1 is the second smallest
    const float r0 = row_min(mn);
    float sec = 3e38f, eq = 0.f;
#pragma unroll
    for (int u = 0; u < MPL; u++) {
        const float r = fminf((float)r64[u], 3e38f);
        eq += r == r0 ? 1.f : 0.f;
        sec = fminf(sec, r == r0 ? 3e38f : r);
    }
    eq = row_sum(eq);
    sec = row_min(sec);
    float lo = eq > 1.f ? r0 : sec;
    const float rmax = __builtin_sqrtf(tau);
    const float norm = (float)hsml_norm(a.dim), kf = (float)k;
    float hi = (float)hsml_bound_coeff(a.dim) * rmax;
    bool run = on && !(st & ST_COUNT) && hi > 0.f;
    // (no k-th distance: as the main kernel)
    float h = run ? fmaxf(HSML_START * rmax, lo) : (rmax < INFINITY ? 0.f : INFINITY);
    if (SEED && run && a.seed_h) {
        const float seed = a.seed_h[a.qrow ? a.qrow[slot] : a.perm[slot]];
        if (seed > lo && seed < hi) h = seed;
        else if (seed > 0.f) st |= ST_SEED_MISS;
    }
    for (int it = 0; it < 40 && __any(run); it++) {
        const float ih = __builtin_amdgcn_rcpf(h);
        float s = 0.f, ds = 0.f;
#pragma unroll
        for (int u = 0; u < MPL; u++) {
            // W = 2 a^3 - b^3, a = (1 - q)_+, b = (1 - 2q)_+
            const float qq = fminf((float)r64[u] * ih, 1.0f);
            const float aa = 1.0f - qq, bb = fmaxf(fmaf(-2.0f, qq, 1.0f), 0.f);
            const float a2 = aa * aa, b2 = bb * bb;
            s += fmaf(2.0f * aa, a2, -(bb * b2));
            ds = fmaf(a2 - b2, qq, ds);
        }
        s = row_sum(s);
        ds = row_sum(ds);
        const float n = norm * s;
        if (n > kf) hi = h;
        else lo = h;
        float hn = hsml_step(h, n, norm * 6.0f * ds, kf);
        bool done = n == kf;
        if (done) {
            hn = h;
        } else if (fabsf(hn - h) <= HSML_STEP * h) {  // as the main kernel: a step this small ends the solve
            hn = fminf(fmaxf(hn, lo), hi);
            done = true;
        } else {
            if (!(hn > lo && hn < hi)) hn = 0.5f * (lo + hi);
            done = hi - lo <= 2.5e-7f * h;
        }
        if (run) h = hn;
        run = run && !done;
    }
    if (run) st |= ST_HSML_NOCONV;
    double h64 = (double)h;
    const bool fine = on && h > 0.f && !(st & (ST_HSML_NOCONV | ST_AMBIGUOUS | ST_COUNT));
    bool flat = false;  // (refine_h64)
    if (hsml_rootless(k, a.dim)) {
        HsmlRange r;
#pragma unroll
        for (int u = 0; u < MPL; u++)
            if (u * 16 + rl < k) r.add(member_dist<PER, P64, true>(t, q, s_out[(u * 16 + rl) * ncol + col]));
        row_join(r);
        if (fine) h64 = r.r1;
    } else {
        const double ih = fine ? 1.0 / h64 : 0.0;
        HsmlSums s;
#pragma unroll
        for (int u = 0; u < MPL; u++) s.add(r64[u] * ih);
        s.w = row_sum(s.w);
        s.d1 = row_sum(s.d1);
        s.d2 = row_sum(s.d2);
        const HsmlStep step = hsml_halley(s, k, a.dim);
        flat = fine && !hsml_last(step, k, a.dim);
        if (fine && !flat) h64 = h64 - h64 * step.rel;
    }
    if (on && rl == 0) {
        write_h(a, slot, h64);
        a.st_slot[slot] = st;
        if ((st & ST_AMBIGUOUS) || flat) a.amb[1 + atomicAdd(a.amb, 1u)] = (uint32_t)slot;
    }
}

// each wavefront serves PW consecutive slots; the block's rows of the member
// list (4 PW slots wide) are staged in LDS and written together.  The slots
// are all slots (KW_ALL) or those of the wavefronts in a.defer, whose number
// only the device knows: block b serves part first + b of the list (KW_LIST),
// or every gridDim.x-th from there (KW_LOOP: the compiler keeps the loop's
// invariants in registers, 4 wavefronts a SIMD instead of 7).
enum { KW_ALL, KW_LIST, KW_LOOP };
template <int NR, bool PER, bool P64, int PW, int MODE, typename OFF>
__global__ __launch_bounds__(64 * KW_WAVES) void k_knn_wave(KnnArgs a, uint32_t first) {
    constexpr bool LIST = MODE != KW_ALL;
    constexpr int NCOL = KW_WAVES * PW;
    constexpr int KMAX = NR > 4 ? 128 : 64;
    static_assert(WAVE % NCOL == 0, "a deferred wavefront's slots are whole blocks of them");
    __shared__ uint2 s_c[KW_WAVES][64 * NR];
    __shared__ uint32_t s_lq[KW_WAVES][KW_LEAFQ];
    __shared__ uint32_t s_stk[KW_WAVES][MAX_DEPTH / 2 + 1][4];
    __shared__ uint32_t s_out[KMAX * NCOL];
    __shared__ uint32_t s_mine[LIST ? NCOL : 1];  // the rows this launch finishes
    const int w = threadIdx.x >> 6, row = (threadIdx.x & 63) >> 4;
    auto serve = [&](int64_t slot0) {
        // the slot of this lane's row in the smoothing-length stage
        float tau = 0.f;
        int32_t st = 0;
        uint32_t qr = 0;
        bool on = false;
        for (int i = 0; i < PW; i++) {
            const int col = w * PW + i;
            const int64_t slot = slot0 + col;
            if (slot >= a.nq) break;
            if (LIST) {
                const bool mine = row_was_deferred((int32_t)uniform((uint32_t)a.st_slot[slot]));
                if ((threadIdx.x & 63) == 0) s_mine[col] = mine;
                if (!mine) continue;
            }
            const uint32_t qp = uniform(a.qsorted ? a.qsorted[slot] : (uint32_t)slot);
            float tq, tq1;
            int32_t sq = wave_search<NR, PER, P64, OFF>(a, slot, qp, s_c[w], s_lq[w], s_stk[w], s_out, col, NCOL, tq,
                                                        tq1);
            if (LIST && a.seed_r) {
                const float bound = radius_bound(a.seed_r[a.qrow ? a.qrow[slot] : a.perm[slot]]);
                if (bound < INFINITY && tq1 >= bound) sq |= ST_RADIUS_MISS;
            }
            if (row == i) {
                tau = tq;
                st = sq;
                qr = qp;
                on = true;
            }
        }
        const int col = w * PW + min(row, PW - 1);
        const int64_t slot = slot0 + col;
        if (__any(on)) {
            // rows without a query repeat the wavefront's first that has one
            const int some = (int)__builtin_ctzll(__ballot(on));
            const uint32_t q0 = (uint32_t)__shfl((int)qr, some);
            const int c0 = __shfl(col, some);
            if (!on) qr = q0;
            const int c = on ? col : c0;
            if (a.k <= 32) row_hsml<2, PER, P64, LIST>(a, on, slot, qr, tau, st, s_out, c, NCOL);
            else row_hsml<(NR > 4 ? 8 : 4), PER, P64, LIST>(a, on, slot, qr, tau, st, s_out, c, NCOL);
        }
        __syncthreads();
        for (int e = threadIdx.x; e < a.k * NCOL; e += 64 * KW_WAVES) {
            const int64_t s = slot0 + e % NCOL;
            if (s < a.nq && (!LIST || s_mine[e % NCOL])) a.nl_idx[(int64_t)(e / NCOL) * a.nq + s] = s_out[e];
        }
    };
    constexpr uint32_t PARTS = WAVE / NCOL;
    auto part = [&](uint32_t b) { return (int64_t)a.defer[1 + b / PARTS] * WAVE + b % PARTS * NCOL; };
    if constexpr (MODE == KW_ALL) {
        const int64_t slot0 = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * NCOL;
        if (a.split) {  // (qsorted is given then)
            const int64_t s0 = slot0 & ~(int64_t)(WAVE - 1);
            if (a.qsorted[min(s0 + WAVE - 1, a.nq - 1)] - a.qsorted[s0] <= KNN_SPREAD) return;
        }
        serve(slot0);
    } else if constexpr (MODE == KW_LIST) {
        const uint32_t b = first + blockIdx.x;
        if (b < a.defer[0] * PARTS) serve(part(b));
    } else {
        const uint32_t total = a.defer[0] * PARTS;
        for (uint32_t b = first + blockIdx.x; b < total; b += gridDim.x) {
            serve(part(b));
            __syncthreads();  // the next slots reuse s_out
        }
    }
}

template <int NR, int PW, int MODE, typename OFF>
static void launch_wave(const KnnArgs &a, bool per, bool p64, int64_t blocks, int64_t first, hipStream_t s) {
    const dim3 g((unsigned)blocks), b(64 * KW_WAVES);
    const uint32_t f = (uint32_t)first;
    if (per && p64) hipLaunchKernelGGL((k_knn_wave<NR, true, true, PW, MODE, OFF>), g, b, 0, s, a, f);
    else if (per) hipLaunchKernelGGL((k_knn_wave<NR, true, false, PW, MODE, OFF>), g, b, 0, s, a, f);
    else if (p64) hipLaunchKernelGGL((k_knn_wave<NR, false, true, PW, MODE, OFF>), g, b, 0, s, a, f);
    else hipLaunchKernelGGL((k_knn_wave<NR, false, false, PW, MODE, OFF>), g, b, 0, s, a, f);
}

template <int NR>
static void launch_wave_k(const KnnArgs &a, bool per, bool p64, bool deferred, hipStream_t s) {
    if (deferred) {
        // most of the list on a grid that needs no loop: in an open set it is
        // short and a query a wavefront ends sooner than four (2^22 clustered
        // points: 0.135 ms against 0.281), in a periodic one it holds the
        // wavefronts near the faces
        const int64_t waves = (a.nq + WAVE - 1) / WAVE;
        constexpr int64_t P1 = WAVE / KW_WAVES, P4 = P1 / 4;  // blocks per wavefront of the list
        if (a.n >= (int64_t)1 << 30) {
            launch_wave<NR, 4, KW_LOOP, uint64_t>(a, per, p64, std::min(waves * P4, KW_LIST_OPEN), 0, s);
        } else if (per) {
            const int64_t n1 = std::min(waves * P4, KW_LIST_PER);
            launch_wave<NR, 4, KW_LIST, uint32_t>(a, per, p64, n1, 0, s);
            if (waves * P4 > n1)
                launch_wave<NR, 4, KW_LOOP, uint32_t>(a, per, p64, std::min(waves * P4 - n1, KW_LIST_OPEN), n1, s);
        } else {
            const int64_t n1 = std::min(waves * P1, 4 * KW_LIST_OPEN);
            launch_wave<NR, 1, KW_LIST, uint32_t>(a, per, p64, n1, 0, s);
            if (waves * P1 > n1)
                launch_wave<NR, 1, KW_LOOP, uint32_t>(a, per, p64, std::min(waves * P1 - n1, KW_LIST_OPEN), n1, s);
        }
    } else if (a.nq <= 32768) {
        // one slot per wavefront while there are fewer wavefronts than the
        // chip holds, else four
        launch_wave<NR, 1, KW_ALL, uint32_t>(a, per, p64, (a.nq + KW_WAVES - 1) / KW_WAVES, 0, s);
    } else {
        launch_wave<NR, 4, KW_ALL, uint32_t>(a, per, p64, (a.nq + 4 * KW_WAVES - 1) / (4 * KW_WAVES), 0, s);
    }
}

int knn_wave_launch(mhip_ctx *ctx, const KnnArgs &a, bool per, bool p64, bool deferred) {
    if (a.k <= 64) launch_wave_k<4>(a, per, p64, deferred, ctx->stream);
    else launch_wave_k<6>(a, per, p64, deferred, ctx->stream);
    return check_hip(ctx, hipGetLastError(), "knn launch");
}

}  // namespace mhip
