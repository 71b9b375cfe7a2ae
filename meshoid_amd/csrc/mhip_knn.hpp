// Shared by the kNN kernels (mhip_knn.hip: one lane per query; mhip_knn_wave.hip:
// one wavefront per query): tree view, float32 distances and box gaps, float64
// refinement of the smoothing length.
#pragma once
#include "mhip_internal.hpp"
#include "mhip_knn_rules.hpp"

namespace mhip {

constexpr float U32 = 5.9604645e-8f;         // 2^-24
constexpr float AMBIG_REL = 12.0f * U32;     // fp32 vs fp64 ordering ambiguity of d^2
constexpr float BAND_REL = 16.0f * U32;      // resolver band half-width
constexpr float HSML_STEP = 2e-3f;           // a relative float32 step that ends the solve for h
constexpr float HSML_START = 0.92f;          // first guess of h / r_k (its median is 0.91)
constexpr float PRUNE_REL = 1.0f + 1e-5f;    // box-test safety factor

struct TreeView {
    const float *sx, *sy, *sz, *lx, *ly, *lz;
    const float *nodes;
    int64_t first_leaf, nleaf;
    float box, half;  // periodic box length and half of it (0: open)
    float slack;      // absolute box-test slack: 0 for float32 inputs, covers
                      // the float32 residuals of float64 inputs otherwise
    int depth;        // level of the leaves (root = level 0)
};

struct QPos {
    float x, y, z, lx, ly, lz;
};

template <bool P64>
MHIP_DEV QPos load_q(const TreeView &t, uint32_t p) {
    QPos q;
    q.x = t.sx[p];
    q.y = t.sy[p];
    q.z = t.sz[p];
    q.lx = P64 ? t.lx[p] : 0.f;
    q.ly = P64 ? t.ly[p] : 0.f;
    q.lz = P64 ? t.lz[p] : 0.f;
    return q;
}

// Offset c - q along one axis.  Periodic: the nearest image is formed by
// moving whichever coordinate lies in the far half by one box length; that
// subtraction (x - box with box/2 <= x < box) is exact (Sterbenz), so the
// wrapped offset carries a single rounding, like an unwrapped one.
template <bool PER>
MHIP_DEV float axis_off(float c, float q, float box, float half) {
    const float d = c - q;
    if (!PER) return d;
    const float up = (c - box) - q;  // image of c one box lower (c in the far half)
    const float dn = c - (q - box);  // image of c one box higher (q in the far half)
    return d > half ? up : (d < -half ? dn : d);
}

// squared distance, float32, fixed operation order (shared by every pass so
// that the same pair always yields the same bits)
template <bool PER, bool P64>
MHIP_DEV float dist2(const TreeView &t, const QPos &q, float cx, float cy, float cz, float clx,
                     float cly, float clz) {
    float dx = axis_off<PER>(cx, q.x, t.box, t.half);
    float dy = axis_off<PER>(cy, q.y, t.box, t.half);
    float dz = axis_off<PER>(cz, q.z, t.box, t.half);
    if (P64) {
        dx = dx + (clx - q.lx);
        dy = dy + (cly - q.ly);
        dz = dz + (clz - q.lz);
    }
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

template <bool PER>
MHIP_DEV float axis_gap(float q, float lo, float hi, float box, float slack) {
    float g = fmaxf(lo - q, q - hi);
    if (PER) {
        // the box one period lower / higher
        g = fminf(g, fmaxf((lo - box) - q, q - (hi - box)));
        g = fminf(g, fmaxf(lo - (q - box), (q - box) - hi));
    }
    return fmaxf(g - slack, 0.f);
}

// lower bound of the squared distance from q to any particle under node x
template <bool PER>
MHIP_DEV float node_d2(const TreeView &t, const QPos &q, uint32_t x) {
    const float4 *nb = (const float4 *)(t.nodes + (int64_t)x * 8);
    const float4 a = nb[0], b = nb[1];  // lo xyz, hi x | hi yz
    const float dx = axis_gap<PER>(q.x, a.x, a.w, t.box, t.slack);
    const float dy = axis_gap<PER>(q.y, a.y, b.x, t.box, t.slack);
    const float dz = axis_gap<PER>(q.z, a.z, b.y, t.box, t.slack);
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// next node in depth-first order after the subtree of x is finished; false
// at the end of the traversal (children of p are 8p+1..8p+8)
MHIP_DEV bool next_after(uint32_t &x) {
    while (x != 0 && (x & (FANOUT - 1)) == 0) x = (x - 1) >> 3;
    if (x == 0) return false;
    x++;
    return true;
}

// one leaf's candidates of this lane (per-lane gathers, 64-byte aligned)
template <bool P64>
MHIP_DEV void load_leaf(const TreeView &t, int64_t leaf, float (&cx)[LEAF], float (&cy)[LEAF],
                        float (&cz)[LEAF], float (&clx)[LEAF], float (&cly)[LEAF], float (&clz)[LEAF]) {
    const int64_t base = leaf * LEAF;
#pragma unroll
    for (int v = 0; v < LEAF / 4; v++) {
        const float4 X = ((const float4 *)(t.sx + base))[v];
        const float4 Y = ((const float4 *)(t.sy + base))[v];
        const float4 Z = ((const float4 *)(t.sz + base))[v];
        cx[4 * v] = X.x, cx[4 * v + 1] = X.y, cx[4 * v + 2] = X.z, cx[4 * v + 3] = X.w;
        cy[4 * v] = Y.x, cy[4 * v + 1] = Y.y, cy[4 * v + 2] = Y.z, cy[4 * v + 3] = Y.w;
        cz[4 * v] = Z.x, cz[4 * v + 1] = Z.y, cz[4 * v + 2] = Z.z, cz[4 * v + 3] = Z.w;
        if (P64) {
            const float4 LX = ((const float4 *)(t.lx + base))[v];
            const float4 LY = ((const float4 *)(t.ly + base))[v];
            const float4 LZ = ((const float4 *)(t.lz + base))[v];
            clx[4 * v] = LX.x, clx[4 * v + 1] = LX.y, clx[4 * v + 2] = LX.z, clx[4 * v + 3] = LX.w;
            cly[4 * v] = LY.x, cly[4 * v + 1] = LY.y, cly[4 * v + 2] = LY.z, cly[4 * v + 3] = LY.w;
            clz[4 * v] = LZ.x, clz[4 * v + 1] = LZ.y, clz[4 * v + 2] = LZ.z, clz[4 * v + 3] = LZ.w;
        } else {
            clx[4 * v] = clx[4 * v + 1] = clx[4 * v + 2] = clx[4 * v + 3] = 0.f;
            cly[4 * v] = cly[4 * v + 1] = cly[4 * v + 2] = cly[4 * v + 3] = 0.f;
            clz[4 * v] = clz[4 * v + 1] = clz[4 * v + 2] = clz[4 * v + 3] = 0.f;
        }
    }
}

// orders this wavefront's LDS accesses (they execute in program order; this
// keeps the compiler from moving them across)
MHIP_DEV void lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// wavefront minimum / maximum on the DPP network: rows of 16, then the row
// broadcasts; the result is in lane 63
template <int CTRL, int ROWS>
MHIP_DEV float dpp_f(float old, float x) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), CTRL, ROWS, 0xf, false));
}
MHIP_DEV float wave_min_f(float x) {
    x = fminf(x, dpp_f<0x111, 0xf>(x, x));
    x = fminf(x, dpp_f<0x112, 0xf>(x, x));
    x = fminf(x, dpp_f<0x114, 0xf>(x, x));
    x = fminf(x, dpp_f<0x118, 0xf>(x, x));
    x = fminf(x, dpp_f<0x142, 0xa>(x, x));
    x = fminf(x, dpp_f<0x143, 0xc>(x, x));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
MHIP_DEV float wave_max_f(float x) { return -wave_min_f(-x); }

MHIP_DEV int wave_max(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
    return (int)uniform((uint32_t)v);
}

MHIP_DEV uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

struct KnnArgs {
    TreeView t;
    const uint32_t *qsorted;  // null: slot q is sorted particle q
    const uint32_t *qrow;     // null: row = perm[q]
    const uint32_t *perm;
    int64_t nq, n;
    int k, dim;
    const float *seed_h;   // Newton seed per output row, null = none
    const float *seed_r;   // search-radius bound per output row, null = none
    int redo;              // 1: second launch, redo waves with a radius-seed miss
    int32_t *status_out;
    // per slot state
    float *tau;
    float *h_slot;
    double *h64_slot;
    int32_t *st_slot;
    uint32_t *nl_idx;
    float *nl_d2;
    unsigned long long *stats;  // work counters, may be null
    uint32_t *amb;              // [0] count, [1..] slots for the resolver: ambiguous, or h not refined
    uint32_t *defer;            // [0] count, [1..] wavefronts (64 slots) left to the one-wavefront-per-query kernel
    bool split;                 // wavefronts shared out between the kernels (knn_splits)
    uint32_t wlcap;             // leaf-record capacity used (<= WLCAP; smaller only as a test hook)
};

// square of a radius seed, +inf for none (0): a row whose (k+1)-th squared
// distance is not below it missed (ST_RADIUS_MISS)
MHIP_DEV float radius_bound(float sr) { return sr > 0.f && sr < 3e18f ? sr * sr : INFINITY; }

MHIP_DEV void pad_list(const KnnArgs &a, int cnt, uint32_t qp, int64_t slot) {
    // never leave undefined indices behind: pad with the query itself
    for (int j = cnt; j < a.k; j++) {
        a.nl_idx[(int64_t)j * a.nq + slot] = qp;
        if (a.nl_d2) a.nl_d2[(int64_t)j * a.nq + slot] = INFINITY;
    }
}

// |d| from r2 = |d|^2 (float64): the hardware reciprocal square root (5.2e-8 off
// at most) and one third-order step, without the scaling and fix-up
// instructions of the correctly rounded root: 1.7e-16 off at most over 2^22
// values.  Tiny r2 (float64 inputs at pathological scales, where the estimate
// would meet denormals) take sqrt.
MHIP_DEV double pair_dist(double r2) {
    if (r2 < 1e-280) return sqrt(r2);
    const double y = __builtin_amdgcn_rsq(r2);
    const double r = r2 * y;
    const double e = fma(-r, y, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}
// The same by one Newton step on the root, 4.1e-15 off at most: the weights of a
// fit, whose results are float32, and the one step of the smoothing length,
// which moves by no more than its distances do.  (Against sqrt, apply_D1 2.27 ->
// 2.05 ms at 2^24 with four lanes per query.)
MHIP_DEV double fit_dist(double r2) {
    if (r2 < 1e-280) return sqrt(r2);
    const double y = __builtin_amdgcn_rsq(r2);
    const double r = r2 * y;
    const double res = fma(-r, r, r2);
    return fma(0.5 * y, res, r);
}

// float64 distance of member p from the query: exact offsets for float32
// positions, hi + lo for float64 inputs, minimum image when periodic.  FINE: the
// root by pair_dist (a row's bracket, and rows where n(h) is flat)
template <bool PER, bool P64, bool FINE>
MHIP_DEV double member_dist(const TreeView &t, const QPos &q, uint32_t p) {
    double d[3] = {(double)t.sx[p] - ((double)q.x + (double)q.lx), (double)t.sy[p] - ((double)q.y + (double)q.ly),
                   (double)t.sz[p] - ((double)q.z + (double)q.lz)};
    if (P64) {
        d[0] += (double)t.lx[p];
        d[1] += (double)t.ly[p];
        d[2] += (double)t.lz[p];
    }
    if (PER) {
        const double box = (double)t.box;
#pragma unroll
        for (int c = 0; c < 3; c++) d[c] = wrap<double>(d[c], box);
    }
    const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    return FINE ? pair_dist(r2) : fit_dist(r2);
}

// The float64 smoothing length by one lane, member(j) giving the sorted index of
// member j < k: one step from the float32 solve.  flat: a step is not enough
// (hsml_last); the row then goes to the resolver kernel, by the same list as the
// ambiguous ones, which has a wavefront for it.
template <bool PER, bool P64, typename F>
MHIP_DEV double refine_h64(const KnnArgs &a, const QPos &q, double hd, bool &flat, F member) {
    if (hsml_rootless(a.k, a.dim)) {
        HsmlRange r;
        for (int j = 0; j < a.k; j++) r.add(member_dist<PER, P64, true>(a.t, q, member(j)));
        return r.r1;
    }
    const double ih = 1.0 / hd;
    HsmlSums s;
    for (int j = 0; j < a.k; j++) s.add(member_dist<PER, P64, false>(a.t, q, member(j)) * ih);
    const HsmlStep st = hsml_halley(s, a.k, a.dim);
    flat = !hsml_last(st, a.k, a.dim);
    return flat ? hd : hd - hd * st.rel;
}

// Newton's step in the logarithms, ln n against ln h (n(h) is close to a power
// law between neighbours): p = h n'(h)
MHIP_DEV float hsml_step(float h, float n, float p, float kf) {
    return h * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(kf * __builtin_amdgcn_rcpf(n)) * n *
                                      __builtin_amdgcn_rcpf(p));
}

// smoothing length of one query slot (float32 copy and float64); the
// row-order h, density and volume are formed from it by k_rows_rec
MHIP_DEV void write_h(const KnnArgs &a, int64_t slot, double h) {
    a.h_slot[slot] = (float)h;
    a.h64_slot[slot] = h;
}

// one wavefront per query (mhip_knn_wave.hip): its launch over every slot, or
// (deferred) over the wavefronts in a.defer
int knn_wave_launch(mhip_ctx *ctx, const KnnArgs &a, bool per, bool p64, bool deferred);

}  // namespace mhip
