// Exact k-nearest-neighbour search, smoothing length and density on the GPU.
//
// Replaces, for the hot path, the reference's
//   cKDTree.query(pos[mask], des_ngb)           src/meshoid/Meshoid.py:157
//   HsmlIter(ngbdist, error_norm=1e-13, dim)     src/meshoid/Meshoid.py:165,
//                                                src/meshoid/kernel_density.py:14-57
//   density = des_ngb*m/(volnorm*h^dim)          src/meshoid/Meshoid.py:169-170
//
// Two kernels: one lane per query (here) and one wavefront per query
// (mhip_knn_wave.hip); knn_wave_serves there says which takes a set.
//
// One lane per query (64 consecutive queries in Hilbert order per wavefront;
// the tree is a complete 8-ary tree in heap numbering, root 0, children of x
// at 8x+1..8x+8, leaves of 16 particles on the last level).  Every lane keeps
// the k+1 smallest float32 squared distances of its query sorted in VGPRs.
//   (1) The leaves holding the wave's own queries and two on either side are
//       scanned first; then a walk inside out over groups of 64 nodes.
//   (2) A leaf's 16 candidates (scalar loads) go to each lane's LDS queue
//       row, which advances when the candidate is under the lane's (k+1)-th
//       distance.  Queues drain 16 rows at a time through sorting networks
//       (few rows: one in-place v_med3 per slot and row).  Leaves where some
//       lane queued a candidate are recorded, with the lanes that did.
//   (3) Epilogue: smoothing length (safeguarded float32 Newton, then one
//       float64 step over the final members), density, volume, and the member
//       set {d2 <= tau}: each lane scans the recorded leaves that it queued
//       from and that its final radius reaches, one leaf per lane per step
//       (per-lane loads); the indices are staged in LDS and written as whole
//       rows.  Queries whose k-th and (k+1)-th distances float32 cannot order
//       are re-ranked with float64 distances from the caller's positions, so
//       neighbour sets equal the float64 kNN except for float64 ties.
//       The same kernel finishes smoothing lengths that one float64 step does
//       not give (rows where n(h) is flat at the root, see hsml_last).
//   Wavefronts whose queries spread over a large region, and in periodic sets
//   those whose balls reach a face of the box, are left to the other kernel.
// It is bound by vector instructions: 28.1k a wavefront at 2^24 clustered
// particles, k = 32 (70 leaves x 143, 20 runs of 16 through the networks x
// 306, 3.5 smoothing-length iterations x 415, 16 member steps x 157), the
// vector units 79% busy; 14.3 ms, against 20.0 ms and 43.3k with one insertion
// step per queued row, 8 child boxes tested by all lanes per node and
// compensated branches in the smoothing length.
#include "../../include/meshoid_hip.h"
#include "mhip_internal.hpp"
#include "mhip_knn.hpp"
#include "mhip_sortnet.hpp"

namespace mhip {

constexpr int KNN_BLOCK = 256;
constexpr int KNN_WAVES = KNN_BLOCK / WAVE;
constexpr int QCAP = 32;                     // per-lane pending-candidate queue
constexpr int WLCAP = 128;                   // per-wave record of candidate leaves
constexpr int WLWORDS = WLCAP / 32;
static_assert(WLWORDS == 4, "the member pass reads the masks as two pairs");
// leaves after which a wavefront gives up (its queries lie far apart; ~70 are
// scanned by one whose queries do not)
constexpr uint32_t LEAFMAX = 224;
constexpr uint32_t INF_BITS = 0x7f800000u;   // +inf
constexpr int BAND_CAP = 32;
constexpr int64_t RESOLVE_WAVES = 8192;      // resolver grid (one wavefront per ambiguous slot)


// Inserts x into the ascending list A, dropping the largest entry: slot j
// becomes med3(A[j-1], x, A[j]).  The slots are updated in place from the top
// down (each instruction's destination is its own old value), so the list
// keeps its registers across loop iterations instead of alternating between
// two register sets joined by copies.  x is never NaN.
template <int KCAP>
MHIP_DEV void insert_sorted(float (&A)[KCAP], float x) {
#pragma unroll
    for (int j = KCAP - 1; j > 0; --j)
        asm volatile("v_med3_f32 %0, %1, %2, %0" : "+v"(A[j]) : "v"(A[j - 1]), "v"(x));
    asm volatile("v_min_f32 %0, %1, %0" : "+v"(A[0]) : "v"(x));
}


// LDS rows are ROW_STEP bytes apart (one float per lane)
constexpr uint32_t ROW_STEP = WAVE * 4;

// LDS byte address of a shared variable, and a store there
MHIP_DEV uint32_t lds_address(uint32_t *p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)p; }
MHIP_DEV void lds_store(uint32_t addr, uint32_t v) { *(__attribute__((address_space(3))) uint32_t *)(uintptr_t)addr = v; }

// row address ra of the lanes with a < b (or a <= b) moves on by one row: the
// compare writes EXEC, the addition runs under it, and the wavefront's EXEC
// (all) comes back.  Two vector instructions per candidate; a compare into a
// mask, a select and an addition are three, and a row counter with the
// address formed from it four.
MHIP_DEV void advance_lt(uint32_t &ra, float a, float b, uint64_t all) {
    asm volatile("v_cmpx_lt_f32 vcc, %1, %2\n\tv_add_u32 %0, %3, %0\n\ts_mov_b64 exec, %4"
                 : "+v"(ra)
                 : "v"(a), "v"(b), "s"(ROW_STEP), "s"(all)
                 : "vcc");
}
MHIP_DEV void advance_le(uint32_t &ra, float a, float b, uint64_t all) {
    asm volatile("v_cmpx_le_f32 vcc, %1, %2\n\tv_add_u32 %0, %3, %0\n\ts_mov_b64 exec, %4"
                 : "+v"(ra)
                 : "v"(a), "v"(b), "s"(ROW_STEP), "s"(all)
                 : "vcc");
}

MHIP_DEV int64_t slot_of_lane(int64_t *first) {
    const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
    const int64_t wave0 = ((int64_t)b * KNN_WAVES + (threadIdx.x >> 6)) * WAVE;
    *first = wave0;
    return wave0 + (threadIdx.x & (WAVE - 1));
}


// ---------------------------------------------------------------------------
// smoothing length on the k nearest distances (kernel_density.py:36-56 root):
// norm * sum_j W(r_j/h) = k, bracket [r_1, c_d r_{k-1}].  Safeguarded Newton in
// float32; the bracket is the fallback.  On return A[0..KCAP-2] hold the
// distances (sentinel slots: larger than any), not their squares: the list is
// not needed afterwards, and reusing its registers keeps the kernel's register
// count at that of the traversal.  W as truncated powers (see HsmlSums): 11
// instructions per neighbour and iteration, against ~30 with the two branches
// of the spline and compensated sums.  The float64 step that follows is cubic,
// so h needs to be good to ~1e-5 only: a step below HSML_STEP h ends the solve
// (n(h) is C^2, the error left is about twice the step squared).
// ---------------------------------------------------------------------------
template <int KCAP>
MHIP_DEV float hsml_solve(float (&A)[KCAP], int k, int dim, float seed, int32_t &st, int &iters) {
    const int e = KCAP - 1 - k;  // first real slot
    const float norm = (float)hsml_norm(dim);
    float(&r)[KCAP] = A;
    float lo = 0.f, rmax = 0.f;
#pragma unroll
    for (int j = 0; j < KCAP - 1; j++) {
        r[j] = A[j] >= 0.f ? __builtin_amdgcn_sqrtf(A[j]) : 3e38f;
        if (j == e + 1) lo = r[j];
        if (j == KCAP - 2) rmax = r[j];
    }
    float hi = (float)hsml_bound_coeff(dim) * rmax;
    iters = 0;
    if (!(hi > 0.f)) return 0.f;  // all k at distance 0: the reference returns 0
    float h = fmaxf(HSML_START * rmax, lo);
    if (seed > 0.f) {
        if (seed > lo && seed < hi)
            h = seed;
        else
            st |= ST_SEED_MISS;
    }
    const float kf = (float)k;
    int it = 0;
    for (; it < 40; it++) {
        const float ih = __builtin_amdgcn_rcpf(h);
        float s = 0.f, ds = 0.f;  // sums of W / 2 and of -W' q / 6
#pragma unroll
        for (int j = 0; j < KCAP - 1; j++) {
            const float q = fminf(r[j] * ih, 1.0f);
            const float a = 1.0f - q, b = fmaxf(fmaf(-2.0f, q, 1.0f), 0.f);
            const float aa = a * a, bb = b * b;
            s = fmaf(a, aa, s);
            s = fmaf(-0.5f * b, bb, s);
            ds = fmaf(aa - bb, q, ds);
            // keep the terms in order: evaluating all k kernel values ahead
            // of the sums would hold them all in registers at once
            asm volatile("" : "+v"(s), "+v"(ds));
        }
        const float n = 2.0f * norm * s;
        if (n == kf) break;
        if (n > kf)
            hi = h;
        else
            lo = h;
        float hn = hsml_step(h, n, norm * 6.0f * ds, kf);
        // such a step ends the solve even when it rounds onto the bracket end
        // that h itself has just become (otherwise a converged lane would
        // bisect the whole bracket again and hold its wavefront).  A collapsed
        // bracket also ends it.
        if (fabsf(hn - h) <= HSML_STEP * h) {
            h = fminf(fmaxf(hn, lo), hi);
            break;
        }
        if (!(hn > lo && hn < hi)) hn = 0.5f * (lo + hi);
        if (hi - lo <= 2.5e-7f * h) {
            h = hn;
            break;
        }
        h = hn;
    }
    if (it >= 40) st |= ST_HSML_NOCONV;
    iters = min(it + 1, 40);
    return h;
}

// Read-only data read at wave-uniform addresses goes through the constant
// address space, which the compiler serves with scalar (SMEM) loads into
// SGPRs: one load per wavefront instead of 64 lanes, and no VGPRs.
typedef const float __attribute__((address_space(4))) cfloat;
MHIP_DEV float ldc(const float *p, int64_t i) { return ((cfloat *)p)[i]; }

// one leaf's candidates, wave-uniform address (scalar loads)
template <bool P64>
MHIP_DEV void load_leaf_uniform(const float *sx, const float *sy, const float *sz, const float *lx,
                                const float *ly, const float *lz, int64_t leaf, float (&cx)[LEAF],
                                float (&cy)[LEAF], float (&cz)[LEAF], float (&clx)[LEAF],
                                float (&cly)[LEAF], float (&clz)[LEAF]) {
    const int64_t base = leaf * LEAF;
#pragma unroll
    for (int i = 0; i < LEAF; i++) {
        cx[i] = ldc(sx, base + i);
        cy[i] = ldc(sy, base + i);
        cz[i] = ldc(sz, base + i);
        clx[i] = P64 ? ldc(lx, base + i) : 0.f;
        cly[i] = P64 ? ldc(ly, base + i) : 0.f;
        clz[i] = P64 ? ldc(lz, base + i) : 0.f;
    }
}


// squared gap from a lane's query to a box read at wave-uniform addresses
// (scalar loads); the query interval [ql, qh] per axis is the position widened
// by the float64-residual slack (ql = qh for float32 inputs); zero inside
template <bool PER>
MHIP_DEV float axis_gap_u(float ql, float qh, float lo, float hi, float box) {
    float g = fmaxf(lo - qh, ql - hi);
    if (PER) {
        g = fminf(g, fmaxf((lo - box) - qh, ql - (hi - box)));  // the box one period lower
        g = fminf(g, fmaxf(lo - (qh - box), (ql - box) - hi));  // the box one period higher
    }
    return fmaxf(g, 0.f);
}

struct QBox {
    float lx, ly, lz, hx, hy, hz;
};

template <bool PER>
MHIP_DEV float box_gap2_u(const TreeView &t, const QBox &b, uint32_t x) {
    const int64_t o = (int64_t)x * 8;
    const float gx = axis_gap_u<PER>(b.lx, b.hx, ldc(t.nodes, o), ldc(t.nodes, o + 3), t.box);
    const float gy = axis_gap_u<PER>(b.ly, b.hy, ldc(t.nodes, o + 1), ldc(t.nodes, o + 4), t.box);
    const float gz = axis_gap_u<PER>(b.lz, b.hz, ldc(t.nodes, o + 2), ldc(t.nodes, o + 5), t.box);
    return fmaf(gz, gz, fmaf(gy, gy, gx * gx));
}

// bit c set: child 8x+1+c lies within bound of some lane's query
template <bool PER>
MHIP_DEV uint32_t expand_mask(const TreeView &t, const QBox &b, uint32_t x, float bound) {
    uint32_t m = 0;
    const uint32_t c0 = FANOUT * x + 1;
#pragma unroll
    for (int c = 0; c < FANOUT; c++)
        if (__any(box_gap2_u<PER>(t, b, c0 + c) <= bound)) m |= 1u << c;
    return m;
}

// the set bit of m nearest to position o <= 63 (m != 0); ties go upwards
MHIP_DEV uint32_t pick_nearest64(uint64_t m, int o) {
    const uint64_t up = m >> o, down = m & ((1ull << o) - 1ull);
    if (!down) return o + __builtin_ctzll(up);
    const uint32_t cd = 63u - __builtin_clzll(down);
    if (!up) return cd;
    const uint32_t cu = o + __builtin_ctzll(up);
    return cu - o <= o - cd ? cu : cd;
}

// 8-bit child masks of the traversal path, levels 0..7 and 8..15
struct MaskStack {
    uint64_t lo = 0, hi = 0;
    MHIP_DEV uint32_t get(int l) const {
        return l < 8 ? (uint32_t)(lo >> (8 * l)) & 0xffu : (uint32_t)(hi >> (8 * (l - 8))) & 0xffu;
    }
    MHIP_DEV void put(int l, uint32_t m) {
        if (l < 8)
            lo |= (uint64_t)m << (8 * l);
        else
            hi |= (uint64_t)m << (8 * (l - 8));
    }
    MHIP_DEV void clear(int l, uint32_t c) {
        if (l < 8)
            lo &= ~(1ull << (8 * l + c));
        else
            hi &= ~(1ull << (8 * (l - 8) + c));
    }
};

constexpr int LROWS = 33;                          // staged member rows (k <= 32)
constexpr int QROWS = QCAP > LROWS ? QCAP : LROWS;  // per-lane LDS rows

// SPLIT: wavefronts whose queries lie far apart are the other kernel's
// (knn_splits).  An instantiation of its own: the test alone, through the
// allocation of scalar registers, made whole sets 3.4% slower (2^24, k = 32).
template <int KCAP, bool P64, bool SPLIT>
__global__ __launch_bounds__(KNN_BLOCK) void k_knn_main(KnnArgs a) {
    // members are staged in LDS and written as whole rows when they fit
    constexpr bool STAGE = KCAP <= LROWS;
    __shared__ uint32_t s_buf[KNN_WAVES][QROWS][WAVE];
    __shared__ uint32_t s_wl[KNN_WAVES][WLCAP];
    __shared__ uint32_t s_stk[KNN_WAVES][MAX_DEPTH / 2 + 1][3];
    __shared__ uint32_t s_walk[KNN_WAVES][8];
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x >> 6;
    int64_t wave0;
    const int64_t slot = slot_of_lane(&wave0);
    if (wave0 >= a.nq) return;
    const bool live = slot < a.nq;
    const int64_t qs_slot = min<int64_t>(slot, a.nq - 1);
    // redo launch: only waves where some lane missed its radius seed
    const bool missed = a.redo && live && (a.st_slot[qs_slot] & ST_RADIUS_MISS);
    if (a.redo && !__any(missed)) return;
    const uint32_t qp = a.qsorted ? a.qsorted[qs_slot] : (uint32_t)qs_slot;
    if (SPLIT && uniform(__shfl(qp, WAVE - 1)) - uniform(__shfl(qp, 0)) > KNN_SPREAD) return;
    const uint32_t row = a.qrow ? a.qrow[qs_slot] : a.perm[qs_slot];
    // a radius seed starts the k+1 slots at (seed radius)^2 instead of +inf: a
    // lane whose (k+1)-th slot still holds that bound at the end missed
    const float tau0 = radius_bound((a.seed_r && !a.redo) ? a.seed_r[row] : 0.f);
    const TreeView &t = a.t;
    const float *__restrict__ sx = t.sx;
    const float *__restrict__ sy = t.sy;
    const float *__restrict__ sz = t.sz;
    const float *__restrict__ lx = t.lx;
    const float *__restrict__ ly = t.ly;
    const float *__restrict__ lz = t.lz;
    const QPos q = load_q<P64>(t, qp);
    QBox qb;
    qb.lx = P64 ? q.x - t.slack : q.x;
    qb.ly = P64 ? q.y - t.slack : q.y;
    qb.lz = P64 ? q.z - t.slack : q.z;
    qb.hx = P64 ? q.x + t.slack : q.x;
    qb.hy = P64 ? q.y + t.slack : q.y;
    qb.hz = P64 ? q.z + t.slack : q.z;

    // sorted k+1 smallest squared distances; slots below e are -1 sentinels
    // when k + 1 < KCAP, so A[KCAP-2] is the k-th and A[KCAP-1] the (k+1)-th
    float A[KCAP];
    const int e = KCAP - 1 - a.k;
#pragma unroll
    for (int j = 0; j < KCAP; j++) A[j] = j < e ? -1.0f : tau0;
    float cx[LEAF], cy[LEAF], cz[LEAF], clx[LEAF], cly[LEAF], clz[LEAF];
    uint32_t n_ins = 0, n_leaf = 0, n_nodes = 0;  // work counters

    // lists of at least LEAF slots take whole runs of LEAF candidates through
    // sorting networks
    // (longer lists have no registers left for it: k = 100 gains nothing, k =
    // 128 spills)
    constexpr bool NET = KCAP >= LEAF && KCAP <= 65;
    // fewer queued rows than this are inserted one by one: a step costs about
    // KCAP + 8 instructions, sorting and merging a run of 16 about 300 (KCAP
    // 33) or 230 (KCAP 17, 21)
    constexpr int NETMIN = 8;
    float t1 = tau0;               // this lane's (k+1)-th distance when its queue was last drained
    float bound = t1 * PRUNE_REL;  // of it: box tests
    float bmax = INFINITY;         // the wavefront's largest bound
    // this lane's queue: LDS byte addresses of its first and next row
    const uint32_t rows0 = lds_address(&s_buf[w][0][lane]);
    uint32_t qa = rows0;
    bool pad = false;              // the last, NaN-padded leaf has been scanned since the last drain
    uint32_t nwl = 0;              // recorded leaves
    uint32_t mw[WLWORDS];          // bit r: this lane queued a candidate of recorded leaf r
#pragma unroll
    for (int i = 0; i < WLWORDS; i++) mw[i] = 0u;
    const uint32_t first_leaf = (uint32_t)t.first_leaf, nleaf = (uint32_t)t.nleaf;
    const uint32_t last_leaf = nleaf - 1;
    const int depth = t.depth;

    // (1) the leaves holding the wave's own queries, and EXT more on either
    // side along the curve, fill the lists (two leaves more than that take
    // tighten the outer queries' bounds, which decide how many rows the later
    // drains insert); then (2) the rest of the tree, inside out from the
    // middle query's leaf: its ancestor two levels up, then the rest of that
    // node's ancestor two levels up, ...  A node's 64 grandchildren
    // (contiguous in the heap numbering) are tested by the 64 lanes at once
    // against the box of all queries and the largest bound; the survivors are
    // then tested one by one by every lane against its own bound of the
    // moment.  A block's leaves go in three classes of distance to the
    // queries' box, each from the curve's position outwards.
    // One loop holds every stage, so that the scan and the drain exist once.
    const uint32_t p_first = uniform(__shfl(qp, 0));
    const uint32_t p_last = uniform(__shfl(qp, WAVE - 1));
    constexpr uint32_t EXT = NET ? 2 : 0;
    uint32_t l0 = p_first / LEAF;
    const uint32_t l1 = min(min(p_last / LEAF, l0 + 7) + EXT, last_leaf);
    l0 = l0 > EXT ? l0 - EXT : 0;
    uint32_t L = l0;  // next of these leaves
    float wlo[3] = {qb.lx, qb.ly, qb.lz}, whi[3] = {qb.hx, qb.hy, qb.hz};
#pragma unroll
    for (int c = 0; c < 3; c++) {
        wlo[c] = wave_min_f(wlo[c]);
        whi[c] = wave_max_f(whi[c]);
    }
    const uint32_t lc = uniform(__shfl(qp, WAVE / 2 - 1)) / LEAF;
    uint32_t lbase = 0;               // current block of leaves (heap number),
    uint64_t lmask = 0;               // those of the current class still to visit,
    float g = NAN;                    // this lane's leaf's distance (NaN: none, or visited)
    int cls = 3, lpos = 0;            // next class; the curve's position in the block
    // the walk above the leaves is needed once per block of leaves: it lives
    // in LDS, the scalar registers being short (48 hold a leaf's candidates).
    // Lane 0 writes it, and what is read is lane 0's own value (uniform), so no
    // fence is needed
    struct Walk {
        uint32_t own;        // ancestor of the middle leaf whose subtree is done,
        int lev;             // its level
        uint32_t base, mlo, mhi;  // current group of inner nodes, those still to visit,
        int flev, f;         // their level, stacked groups
    };
    if (lane == 0) {
        s_walk[w][0] = first_leaf + lc;
        s_walk[w][1] = (uint32_t)depth;
        s_walk[w][2] = s_walk[w][3] = s_walk[w][4] = s_walk[w][5] = s_walk[w][6] = 0u;
    }
    __builtin_amdgcn_wave_barrier();
    for (int r = 0; r < QROWS; r++) s_buf[w][r][lane] = INF_BITS;
    bool done = false, fill = true, defer = false;
    while (!done) {
        uint32_t li = 0;
        if (L <= l1) {
            li = L++;
        } else {
            while (true) {
                if (lmask) {
                    const uint32_t b = pick_nearest64(lmask, lpos);
                    lmask &= ~(1ull << b);
                    if (!__any(box_gap2_u<false>(t, qb, lbase + b) <= bound)) continue;
                    li = lbase + b - first_leaf;
                    break;
                }
                if (cls < 3) {
                    const float part = cls == 0 ? 0.06f : (cls == 1 ? 0.25f : 1.0f);
                    const bool sel = g <= part * bmax;
                    lmask = __ballot(sel);
                    g = sel ? NAN : g;
                    cls++;
                    continue;
                }
                // the next group of nodes
                __builtin_amdgcn_wave_barrier();
                Walk k;
                k.own = uniform(s_walk[w][0]);
                k.lev = (int)uniform(s_walk[w][1]);
                k.base = uniform(s_walk[w][2]);
                uint64_t fmask = (uint64_t)uniform(s_walk[w][3]) | (uint64_t)uniform(s_walk[w][4]) << 32;
                k.flev = (int)uniform(s_walk[w][5]);
                k.f = (int)uniform(s_walk[w][6]);
                uint32_t y = 0;  // inner node to expand
                while (true) {
                    if (fmask) {
                        y = k.base + __builtin_ctzll(fmask);
                        fmask &= fmask - 1;
                        if (__any(box_gap2_u<false>(t, qb, y) <= bound)) break;
                        y = 0;
                    } else if (k.f > 0) {
                        k.f--;
                        k.flev -= 2;
                        k.base = uniform(s_stk[w][k.f][0]);
                        fmask = (uint64_t)uniform(s_stk[w][k.f][1]) | (uint64_t)uniform(s_stk[w][k.f][2]) << 32;
                    } else {
                        break;
                    }
                }
                if (y == 0 && k.lev == 0) {
                    done = true;
                    break;
                }
                if (n_leaf > LEAFMAX) {
                    defer = true;
                    break;
                }
                uint32_t eb;  // group to expand, its nodes, their level
                int ecnt = 64, elev;
                uint64_t skip = 0;
                if (y != 0) {
                    eb = 64u * y + 9u;
                    elev = k.flev + 2;
                    if (elev != depth) {
                        if (lane == 0) {
                            s_stk[w][k.f][0] = k.base;
                            s_stk[w][k.f][1] = (uint32_t)fmask;
                            s_stk[w][k.f][2] = (uint32_t)(fmask >> 32);
                        }
                        k.f++;
                    }
                } else {
                    // up: the group that holds own
                    const uint32_t par = (k.own - 1) >> 3;
                    const bool two = k.lev >= 2;
                    const uint32_t top = two ? (par - 1) >> 3 : par;
                    eb = two ? 64u * top + 9u : 8u * top + 1u;
                    ecnt = two ? 64 : 8;
                    elev = k.lev;
                    skip = 1ull << (k.own - eb);
                    k.own = top;
                    k.lev -= two ? 2 : 1;
                }
                // the group's boxes against the box of all queries
                n_nodes += WAVE;
                const float4 *nb = (const float4 *)(t.nodes + (int64_t)(eb + min(lane, ecnt - 1)) * 8);
                const float4 u = nb[0], v = nb[1];  // lo xyz, hi x | hi yz
                const float gx = axis_gap_u<false>(wlo[0], whi[0], u.x, u.w, t.box);
                const float gy = axis_gap_u<false>(wlo[1], whi[1], u.y, v.x, t.box);
                const float gz = axis_gap_u<false>(wlo[2], whi[2], u.z, v.y, t.box);
                const float gap = fmaf(gz, gz, fmaf(gy, gy, gx * gx));
                if (elev == depth) {
                    const uint32_t l = eb + lane - first_leaf;
                    g = lane < ecnt && l < nleaf && !(l >= l0 && l <= l1) ? gap : NAN;
                    cls = 0;
                    lbase = eb;
                    const int o = (int)min<int64_t>(63, max<int64_t>(0, (int64_t)lc - (int64_t)(eb - first_leaf)));
                    lpos = o;
                } else {
                    k.base = eb;
                    k.flev = elev;
                    fmask = __ballot(lane < ecnt && gap <= bmax) & ~skip;
                }
                if (lane == 0) {
                    s_walk[w][0] = k.own;
                    s_walk[w][1] = (uint32_t)k.lev;
                    s_walk[w][2] = k.base;
                    s_walk[w][3] = (uint32_t)fmask;
                    s_walk[w][4] = (uint32_t)(fmask >> 32);
                    s_walk[w][5] = (uint32_t)k.flev;
                    s_walk[w][6] = (uint32_t)k.f;
                }
                __builtin_amdgcn_wave_barrier();
            }
            if (defer) break;
        }
        if (!done) {
            // every candidate of the leaf is written to its lane's next queue
            // row, and the row advances when it is under the lane's (k+1)-th
            // distance; leaves where some lane queued a candidate are recorded
            n_leaf++;
            load_leaf_uniform<P64>(sx, sy, sz, lx, ly, lz, li, cx, cy, cz, clx, cly, clz);
            const uint32_t before = qa;
            const uint64_t all = __builtin_amdgcn_read_exec();
#pragma unroll
            for (int i = 0; i < LEAF; i++) {
                const float d2 = dist2<false, P64>(t, q, cx[i], cy[i], cz[i], clx[i], cly[i], clz[i]);
                // at most QCAP - LEAF rows are in use when a leaf starts, so
                // the row stays in range
                lds_store(qa, __float_as_uint(d2));
                advance_lt(qa, d2, t1, all);
            }
            if (li == last_leaf) pad = true;
            if (__any(qa > before)) {
                if (nwl == a.wlcap) {
                    defer = true;
                    break;
                }
                if (lane == 0) s_wl[w][nwl] = li;
                const uint32_t bit = qa > before ? 1u << (nwl & 31u) : 0u;
#pragma unroll
                for (int i = 0; i < WLWORDS; i++)
                    if ((nwl >> 5) == (uint32_t)i) mw[i] |= bit;
                nwl++;
            }
        }
        // the queues drain when one may not take another leaf, after the fill
        // and at the end.  Rows past a lane's qn hold +inf, or at row qn a
        // candidate that was not under the lane's (k+1)-th distance: neither
        // changes a list.
        if (done || (fill && L > l1) || __any(qa > rows0 + (QCAP - LEAF) * ROW_STEP)) {
            const bool filled = fill && L > l1;
            const int nd = wave_max((int)(qa - rows0)) / (int)ROW_STEP;
            if (pad) {
                for (int i = 0; i < QROWS; i++)
                    s_buf[w][i][lane] = __float_as_uint(fminf(__uint_as_float(s_buf[w][i][lane]), INFINITY));
                pad = false;
            }
            int i = 0;
            if constexpr (NET) {
                while (nd - i >= NETMIN && i + LEAF <= QROWS) {
                    float S[LEAF];
#pragma unroll
                    for (int r = 0; r < LEAF; r++) S[r] = __uint_as_float(s_buf[w][i + r][lane]);
#pragma unroll
                    for (int r = 0; r < LEAF; r++) s_buf[w][i + r][lane] = INF_BITS;
                    oddeven_sort<LEAF>(S);
                    merge_sorted<KCAP, LEAF>(A, S);
                    i += LEAF;
                    n_ins += LEAF;
                }
            }
            for (; i < nd; i++) {
                const float v = __uint_as_float(s_buf[w][i][lane]);
                s_buf[w][i][lane] = INF_BITS;
                // rows that no lane's list takes any more are skipped
                if (__any(v < A[KCAP - 1])) {
                    insert_sorted<KCAP>(A, v);
                    n_ins++;
                }
            }
            s_buf[w][min(nd, QROWS - 1)][lane] = INF_BITS;
            qa = rows0;
            t1 = A[KCAP - 1];
            bound = t1 * PRUNE_REL;
            bmax = wave_max_f(bound);
            if (filled) {
                fill = false;
                if (t.box > 0.f) {
                    // Periodic: no query's ball may reach a face of the box
                    // (no neighbour is then an image, and plain offsets and
                    // box gaps serve)
                    const float r = __builtin_amdgcn_sqrtf(t1) * 1.001f + t.slack;
                    const float qx[3] = {q.x, q.y, q.z};
                    bool inner = r < t.half;
#pragma unroll
                    for (int c = 0; c < 3; c++)
                        inner = inner && (c >= a.dim || (qx[c] - r > 0.f && qx[c] + r < t.box));
                    if (__any(!inner)) {
                        defer = true;
                        break;
                    }
                }
            }
        }
    }
    if (defer) {
        // queries spread over a large region (more leaves than the record
        // holds, or than a wavefront should scan), or near a periodic face:
        // left to the one-wavefront-per-query kernel
        if (lane == 0) {
            a.defer[1 + atomicAdd(a.defer, 1u)] = (uint32_t)(wave0 / WAVE);
            if (a.stats) {
                atomicAdd(a.stats + STAT_OVERFLOW_WAVES, 1ull);
                atomicAdd(a.stats + STAT_WAVES, 1ull);
            }
        }
        if (live && row_is_new(a.redo, missed)) a.st_slot[slot] = ROW_DEFERRED;
        return;
    }
    lds_order();  // lane 0 wrote the leaf record that every lane reads
    if (a.stats && lane == 0) {
        atomicAdd(a.stats + STAT_P1_LEAVES, (unsigned long long)n_leaf);
        atomicAdd(a.stats + STAT_P1_NODES, (unsigned long long)n_nodes);
        atomicAdd(a.stats + STAT_P1_INSERTS, (unsigned long long)n_ins);
        atomicAdd(a.stats + STAT_P2_LEAVES, (unsigned long long)nwl);
        atomicAdd(a.stats + STAT_WAVES, 1ull);
    }

    // (3) epilogue
    int32_t st = missed ? ST_RADIUS_MISS : 0;
    const float tau = A[KCAP - 2], tau1 = A[KCAP - 1];
    if (tau0 < INFINITY && tau1 >= tau0) {
        // radius seed missed: the redo launch recomputes this wave plainly
        if (live) a.st_slot[slot] = ST_RADIUS_MISS;
        return;
    }
    if (tau1 <= tau * (1.0f + AMBIG_REL)) st |= ST_AMBIGUOUS;
    const float seed = a.seed_h ? a.seed_h[row] : 0.f;
    int n_newton = 0;
    const float h = hsml_solve<KCAP>(A, a.k, a.dim, seed, st, n_newton);
    if (a.stats) {
        // a redo launch counts only the lanes it recomputes for a miss
        const bool cnt = live && (!a.redo || missed);
        const uint32_t tot = wave_sum(cnt ? (uint32_t)n_newton : 0u);
        const uint32_t mx = (uint32_t)wave_max(cnt ? n_newton : 0);
        if (lane == 0) {
            atomicAdd(a.stats + STAT_NEWTON, (unsigned long long)tot);
            atomicAdd(a.stats + STAT_NEWTON_WMAX, (unsigned long long)mx);
        }
    }
    if (live) {
        a.tau[slot] = tau;
    }
    double h64 = (double)h;
    bool flat = false;  // h is left to the resolver
    // members: a candidate at or below tau passed its lane's queue filter
    // when its leaf was scanned, so it lies in a recorded leaf; leaves no
    // final ball reaches are skipped
    {
        // Unless the row is ambiguous, exactly k particles have d2 <= tau
        // (the (k+1)-th distance is strictly larger), so "d2 <= tau" selects
        // the members.  Ambiguous rows (float32 ties at tau included) are
        // rebuilt by the float64 resolver; for them the count is only capped.
        // Each lane scans only the recorded leaves its own final ball reaches,
        // 64 recorded leaves at a time: a step scans one leaf per lane (its
        // particles loaded by the lane itself), so the wave pays for the
        // busiest lane, not for every leaf some lane needs.
        // Ambiguous lanes take nothing: the resolver writes their rows.
        int cnt = 0;
        uint32_t ra = rows0;  // staged rows: LDS address of the next
        uint32_t nscan = 0;
        const float tb = tau * PRUNE_REL;
        const float take = st & ST_AMBIGUOUS ? -1.0f : tau;
#pragma unroll 1
        for (uint32_t r0 = 0; r0 < nwl; r0 += 64) {
            const uint32_t nr = min(64u, nwl - r0);
            uint32_t nlo = 0, nhi = 0;
            for (uint32_t r = 0; r < nr; r++) {
                const uint32_t li = uniform(s_wl[w][r0 + r]);
                if (box_gap2_u<false>(t, qb, first_leaf + li) <= tb) {
                    if (r < 32)
                        nlo |= 1u << r;
                    else
                        nhi |= 1u << (r - 32);
                }
            }
            // a lane that queued no candidate of a leaf has no member there
            nlo &= r0 == 0 ? mw[0] : mw[2];
            nhi &= r0 == 0 ? mw[1] : mw[3];
            while (__any((nlo | nhi) != 0u)) {
                const bool act = (nlo | nhi) != 0u;
                const uint32_t r =
                    nlo ? (uint32_t)__builtin_ctz(nlo) : (nhi ? 32u + (uint32_t)__builtin_ctz(nhi) : 0u);
                if (nlo)
                    nlo &= nlo - 1u;
                else
                    nhi &= nhi - 1u;
                const uint32_t li = s_wl[w][r0 + r];
                nscan++;
                load_leaf<P64>(t, li, cx, cy, cz, clx, cly, clz);
                const float lim = act ? take : -1.0f;
                if (STAGE) {
                    const uint64_t all = __builtin_amdgcn_read_exec();
#pragma unroll
                    for (int i = 0; i < LEAF; i++) {
                        const float d2 = dist2<false, P64>(t, q, cx[i], cy[i], cz[i], clx[i], cly[i], clz[i]);
                        // at most k members, so at most row k < LROWS; a
                        // row is kept only on a hit
                        lds_store(ra, li * LEAF + i);
                        advance_le(ra, d2, lim, all);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < LEAF; i++) {
                        const float d2 = dist2<false, P64>(t, q, cx[i], cy[i], cz[i], clx[i], cly[i], clz[i]);
                        const bool hit = d2 <= lim;
                        if (hit && live) {
                            a.nl_idx[(int64_t)cnt * a.nq + slot] = li * LEAF + i;
                            if (a.nl_d2) a.nl_d2[(int64_t)cnt * a.nq + slot] = d2;
                        }
                        cnt += hit;
                    }
                }
            }
        }
        if (STAGE) cnt = (int)((ra - rows0) / ROW_STEP);
        if (a.stats && lane == 0) atomicAdd(a.stats + STAT_P2_NODES, (unsigned long long)nscan);
        if (STAGE && live) {
            for (int j = 0; j < a.k; j++) a.nl_idx[(int64_t)j * a.nq + slot] = j < cnt ? s_buf[w][j][lane] : qp;
            if (a.nl_d2) {
                for (int j = 0; j < a.k; j++) {
                    const uint32_t p = j < cnt ? s_buf[w][j][lane] : qp;
                    const float d2 = dist2<false, P64>(t, q, sx[p], sy[p], sz[p], P64 ? lx[p] : 0.f, P64 ? ly[p] : 0.f,
                                                     P64 ? lz[p] : 0.f);
                    a.nl_d2[(int64_t)j * a.nq + slot] = j < cnt ? d2 : INFINITY;
                }
            }
        }
        if (live && cnt != a.k) {
            st |= ST_COUNT;  // (the resolver takes it back from rows it completes)
            if (!STAGE) pad_list(a, cnt, qp, slot);
        }
        // float64 refinement over the members just collected; ambiguous rows
        // (whose capped collection may hold the wrong ties) are refined by
        // the resolver once it has rebuilt them
        if (live && cnt == a.k && h > 0.f && !(st & (ST_HSML_NOCONV | ST_AMBIGUOUS))) {
            if (STAGE)
                h64 = refine_h64<false, P64>(a, q, h64, flat, [&](int j) { return s_buf[w][j][lane]; });
            else
                h64 = refine_h64<false, P64>(a, q, h64, flat, [&](int j) { return a.nl_idx[(int64_t)j * a.nq + slot]; });
        }
    }
    if (live) {
        write_h(a, slot, h64);
        a.st_slot[slot] = st;
    }
    // ambiguous and flat queries for the resolver, one vector atomic per wavefront by
    // its lowest active lane (lanes that missed a radius seed left earlier;
    // in the redo launch only the recomputed lanes are new)
    const bool amb = live && ((st & ST_AMBIGUOUS) || flat) && row_is_new(a.redo, missed);
    const uint64_t am = __ballot(amb);
    if (am) {
        const int leader = __ffsll((long long)__ballot(1)) - 1;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(a.amb, (uint32_t)__popcll(am));
        base = __shfl(base, leader);
        if (amb) a.amb[1 + base + __popcll(am & ((1ull << lane) - 1ull))] = (uint32_t)slot;
    }
}

// the float64 smoothing length of a slot by one wavefront, from its present one;
// the list's members are in memory, up to two of them a lane (k <= 128)
template <bool PER, bool P64>
MHIP_DEV void refine_slot(const KnnArgs &a, const QPos &q, int64_t slot) {
    const int lane = threadIdx.x;
    double r[2] = {1e300, 1e300};  // (no member: no weight)
#pragma unroll
    for (int u = 0; u < 2; u++)
        if (u * WAVE + lane < a.k)
            r[u] = member_dist<PER, P64, true>(a.t, q, a.nl_idx[(int64_t)(u * WAVE + lane) * a.nq + slot]);
    const double h = hsml_refine(
        a.h64_slot[slot], a.k, a.dim,
        [&](double x) {
            const double ix = 1.0 / x;
            HsmlSums s;
            s.add(r[0] * ix);
            s.add(r[1] * ix);
#pragma unroll
            for (int o = WAVE / 2; o > 0; o >>= 1) {
                s.w += __shfl_xor(s.w, o);
                s.d1 += __shfl_xor(s.d1, o);
                s.d2 += __shfl_xor(s.d2, o);
            }
            return s;
        },
        [&] {
            HsmlRange g;
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (u * WAVE + lane < a.k) g.add(r[u]);
#pragma unroll
            for (int o = WAVE / 2; o > 0; o >>= 1)
                g.join(HsmlRange{__shfl_xor(g.r0, o), __shfl_xor(g.r1, o), __shfl_xor(g.rk, o)});
            return g;
        });
    if (lane == 0) write_h(a, slot, h);
}

// float64 squared distance between original particles i and j
template <typename PT, bool PER>
MHIP_DEV double exact_d2(const PT *pos, int dim, uint32_t i, uint32_t j, double box) {
    double s = 0.0;
    for (int c = 0; c < dim; c++) {
        double d = (double)pos[(int64_t)j * dim + c] - (double)pos[(int64_t)i * dim + c];
        if (PER) d = wrap<double>(d, box);
        s = __dadd_rn(s, __dmul_rn(d, d));
    }
    return s;
}

// one ambiguous slot (from the main kernel's list), served by a whole
// wavefront.  The walk is the depth-first one of a single lane (children in
// index order; a node is entered when its box lies within the band's outer
// radius), with a node's 8 children tested by 8 lanes at once and a leaf's
// particles classified by 16 lanes at once: members and band entries are
// taken in the order a lone lane would take them.  The band (at most BAND_CAP
// entries, in LDS) is then ordered and completed by lane 0.
template <bool PER, bool P64, typename PT>
MHIP_DEV void resolve_slot(const KnnArgs &a, const PT *__restrict__ pos_in, int64_t slot, double *s_bd,
                           uint32_t *s_bi) {
    const int lane = threadIdx.x;  // one wavefront per block
    const TreeView &t = a.t;
    const uint32_t qp = a.qsorted ? a.qsorted[slot] : (uint32_t)slot;
    const QPos q = load_q<P64>(t, qp);
    const float tau = a.tau[slot];
    const float band_lo = tau * (1.0f - BAND_REL), band_hi = tau * (1.0f + BAND_REL);
    const float thr = band_hi * PRUNE_REL;
    const uint32_t qo = a.perm[qp];
    const int64_t nq = a.nq;
    const uint64_t below = (1ull << lane) - 1ull;
    int nb = 0, cnt = 0;
    int32_t st = a.st_slot[slot];
    const uint32_t first_leaf = (uint32_t)t.first_leaf;
    // children of internal node x whose boxes pass, as a bit mask
    auto expand = [&](uint32_t x) -> uint32_t {
        const bool pass = lane < FANOUT && node_d2<PER>(t, q, FANOUT * x + 1 + lane) <= thr;
        return (uint32_t)__ballot(pass) & 0xffu;
    };
    auto leaf = [&](uint32_t x) {
        const int64_t li = (int64_t)(x - first_leaf);
        if (li >= t.nleaf) return;
        const int64_t p = li * LEAF + lane;
        float d2 = INFINITY;
        if (lane < LEAF)
            d2 = dist2<PER, P64>(t, q, t.sx[p], t.sy[p], t.sz[p], P64 ? t.lx[p] : 0.f, P64 ? t.ly[p] : 0.f,
                                 P64 ? t.lz[p] : 0.f);
        const bool mem = lane < LEAF && d2 < band_lo;
        const bool inb = lane < LEAF && !mem && d2 <= band_hi && p < a.n;
        const uint64_t bm = __ballot(mem);
        if (mem) {
            const int pos = cnt + __popcll(bm & below);
            if (pos < a.k) {
                a.nl_idx[(int64_t)pos * nq + slot] = (uint32_t)p;
                if (a.nl_d2) a.nl_d2[(int64_t)pos * nq + slot] = d2;
            }
        }
        cnt += __popcll(bm);
        const uint64_t bb = __ballot(inb);
        if (!bb) return;
        const double e = inb ? exact_d2<PT, PER>(pos_in, a.dim, qo, a.perm[p], (double)t.box) : 0.0;
        const int nbb = __popcll(bb);
        if (nb + nbb <= BAND_CAP) {
            if (inb) {
                const int i = nb + __popcll(bb & below);
                s_bd[i] = e;
                s_bi[i] = (uint32_t)p;
            }
            nb += nbb;
            __syncthreads();
            return;
        }
        // entry by entry: appended while there is room, then replacing the
        // largest entry when smaller
        __syncthreads();
        uint64_t rem = bb;
        while (rem) {
            const int l = __ffsll((long long)rem) - 1;
            rem &= rem - 1ull;
            const double el = __shfl(e, l);
            const uint32_t pl = (uint32_t)__shfl((int)p, l);
            if (lane == 0) {
                if (nb < BAND_CAP) {
                    s_bd[nb] = el;
                    s_bi[nb] = pl;
                } else {
                    int wmax = 0;
                    for (int m = 1; m < BAND_CAP; m++)
                        if (s_bd[m] > s_bd[wmax]) wmax = m;
                    if (el < s_bd[wmax]) {
                        s_bd[wmax] = el;
                        s_bi[wmax] = pl;
                    }
                }
            }
            if (nb < BAND_CAP)
                nb++;
            else
                st |= ST_BAND_OVERFLOW;
            __syncthreads();
        }
    };
    if (node_d2<PER>(t, q, 0) <= thr) {
        if (first_leaf == 0) {
            leaf(0);
        } else {
            MaskStack ms;
            ms.put(0, expand(0));
            int lvl = 0;
            uint32_t x = 0;
            while (true) {
                const uint32_t m = ms.get(lvl);
                if (m == 0u) {
                    if (lvl == 0) break;
                    lvl--;
                    x = (x - 1) >> 3;
                    continue;
                }
                const uint32_t c = (uint32_t)__builtin_ctz(m);
                ms.clear(lvl, c);
                const uint32_t y = FANOUT * x + 1 + c;
                if (y >= first_leaf) {
                    leaf(y);
                    continue;
                }
                lvl++;
                x = y;
                ms.put(lvl, expand(y));
            }
        }
    }
    __syncthreads();
    // where float32 distances overflowed there was no solve yet
    const float h0 = a.h_slot[slot];
    if (!(h0 < INFINITY)) st &= ~ST_HSML_NOCONV;
    // (cnt, nb and st are the same in every lane)
    const int have = cnt, total = cnt < a.k ? min(cnt + nb, a.k) : cnt;
    if (total != a.k)
        st |= ST_COUNT;
    else
        st &= ~ST_COUNT;
    if (lane == 0) {
        // order the band by (exact d^2, original index) and take what is missing
        for (int i = 1; i < nb; i++) {
            const double v = s_bd[i];
            const uint32_t vi = s_bi[i];
            int j = i - 1;
            while (j >= 0 && (s_bd[j] > v || (s_bd[j] == v && a.perm[s_bi[j]] > a.perm[vi]))) {
                s_bd[j + 1] = s_bd[j];
                s_bi[j + 1] = s_bi[j];
                j--;
            }
            s_bd[j + 1] = v;
            s_bi[j + 1] = vi;
        }
        for (int i = 0; have + i < total; i++) {
            a.nl_idx[(int64_t)(have + i) * nq + slot] = s_bi[i];
            if (a.nl_d2) a.nl_d2[(int64_t)(have + i) * nq + slot] = (float)s_bd[i];
        }
        if (total != a.k) pad_list(a, min(total, a.k), qp, slot);
        a.st_slot[slot] = st;
    }
    bool flat = false;
    if (lane == 0 && total == a.k && h0 > 0.f && !(st & ST_HSML_NOCONV))
        write_h(a, slot, refine_h64<PER, P64>(a, q, (double)h0, flat,
                                              [&](int j) { return a.nl_idx[(int64_t)j * nq + slot]; }));
    __syncthreads();
    if (__any(flat)) refine_slot<PER, P64>(a, q, slot);
}

// empties the lists of ambiguous slots and of deferred wavefronts (a kernel,
// so graph capture records no memset node)
__global__ void k_lists_reset(uint32_t *__restrict__ amb, uint32_t *__restrict__ defer) {
    if (threadIdx.x == 0) amb[0] = defer[0] = 0u;
}

// the list of ambiguous slots and of those whose smoothing length one step does
// not give, one wavefront per slot (a grid-stride loop over the list, whose
// length only the device knows)
template <bool PER, bool P64, typename PT>
__global__ __launch_bounds__(64) void k_knn_resolve(KnnArgs a, const PT *__restrict__ pos_in) {
    __shared__ double s_bd[BAND_CAP];
    __shared__ uint32_t s_bi[BAND_CAP];
    const uint32_t count = a.amb[0];
    for (int64_t i = blockIdx.x; i < count; i += gridDim.x) {
        const int64_t slot = a.amb[1 + i];
        if (slot >= a.nq) continue;
        if (a.st_slot[slot] & ST_AMBIGUOUS)
            resolve_slot<PER, P64, PT>(a, pos_in, slot, s_bd, s_bi);
        else
            refine_slot<PER, P64>(a, load_q<P64>(a.t, a.qsorted ? a.qsorted[slot] : (uint32_t)slot), slot);
        __syncthreads();  // the next slot reuses the band arrays
    }
}

__global__ void k_qsetup_mask(const int64_t *__restrict__ qidx, int64_t nq,
                              const uint32_t *__restrict__ iperm, uint64_t *__restrict__ keys,
                              uint32_t *__restrict__ vals) {
    int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r >= nq) return;
    keys[r] = iperm[qidx[r]];
    vals[r] = (uint32_t)r;
}

__global__ void k_qsetup_finish(const uint64_t *__restrict__ keys, const uint32_t *__restrict__ vals,
                                int64_t nq, uint32_t *__restrict__ qsorted, uint32_t *__restrict__ qrow) {
    int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= nq) return;
    qsorted[s] = (uint32_t)keys[s];
    qrow[s] = vals[s];
}

// inverse of the index's sorted -> original map (built on first use: only
// queries on a subset of the particles need it)
__global__ __launch_bounds__(256) void k_iperm(const uint32_t *__restrict__ perm, int64_t n,
                                              uint32_t *__restrict__ iperm) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p < n) iperm[perm[p]] = (uint32_t)p;
}

static int ensure_iperm(mhip_ctx *ctx, const mhip_index *ix) {
    if (ix->iperm_ok) return 0;
    hipLaunchKernelGGL(k_iperm, dim3((unsigned)((ix->n + 255) / 256)), dim3(256), 0, ctx->stream, ix->perm, ix->n,
                       ix->iperm);
    ix->iperm_ok = 1;
    return check_hip(ctx, hipGetLastError(), "inverse permutation");
}

// Row-order outputs from the slot-ordered results.  One thread per query
// slot forms h, density = k m / (V_d h^d), volume = m / density
// (Meshoid.py:165-170) and the status bits, and writes them as one 16-byte
// record to its output row (row = srow[slot]: one scattered write per row);
// a second pass copies the records, in row order, into the four output
// arrays (coalesced).  The slot arrays are read in order, so no inverse of
// the sort order is needed.
__global__ __launch_bounds__(256) void k_rows_rec(const uint32_t *__restrict__ srow, int64_t nq, int k, int dim,
                                                 const double *__restrict__ h64, const int32_t *__restrict__ st,
                                                 const double *__restrict__ m_rows, RowRec *__restrict__ rec) {
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= nq) return;
    const uint32_t r = srow[s];
    const double h = h64[s];
    const double vn = dim == 3 ? 4.18879020478639098 : (dim == 2 ? 3.14159265358979324 : 2.0);
    const double m = m_rows ? m_rows[r] : 1.0;
    const double hp = dim == 3 ? h * h * h : (dim == 2 ? h * h : h);
    const double rho = (double)k * m / (vn * hp);
    rec[r] = RowRec{(float)h, (float)rho, (float)(m / rho), st[s]};
}

__global__ __launch_bounds__(256) void k_rows_split(const RowRec *__restrict__ rec, int64_t nq,
                                                   float *__restrict__ h_out, float *__restrict__ rho_out,
                                                   float *__restrict__ vol_out, int32_t *__restrict__ status_out) {
    const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r >= nq) return;
    const RowRec v = rec[r];
    if (h_out) h_out[r] = v.h;
    if (rho_out) rho_out[r] = v.rho;
    if (vol_out) vol_out[r] = v.vol;
    if (status_out) status_out[r] = v.status;
}

template <int KCAP>
static void launch_main(const KnnArgs &a, bool p64, dim3 g, hipStream_t s) {
    // (larger k of a split set are the other kernel's altogether)
    constexpr bool MAY = KCAP <= 65;
    if (p64 && MAY && a.split)
        hipLaunchKernelGGL((k_knn_main<KCAP, true, MAY>), g, dim3(KNN_BLOCK), 0, s, a);
    else if (MAY && a.split)
        hipLaunchKernelGGL((k_knn_main<KCAP, false, MAY>), g, dim3(KNN_BLOCK), 0, s, a);
    else if (p64)
        hipLaunchKernelGGL((k_knn_main<KCAP, true, false>), g, dim3(KNN_BLOCK), 0, s, a);
    else
        hipLaunchKernelGGL((k_knn_main<KCAP, false, false>), g, dim3(KNN_BLOCK), 0, s, a);
}

static void launch_main_k(const KnnArgs &a, bool p64, dim3 g, hipStream_t s) {
    const int need = a.k + 1;
    if (need <= 5) launch_main<5>(a, p64, g, s);
    else if (need <= 9) launch_main<9>(a, p64, g, s);
    else if (need <= 17) launch_main<17>(a, p64, g, s);
    else if (need <= 21) launch_main<21>(a, p64, g, s);
    else if (need <= 33) launch_main<33>(a, p64, g, s);
    else if (need <= 65) launch_main<65>(a, p64, g, s);
    else if (need <= 101) launch_main<101>(a, p64, g, s);
    else launch_main<129>(a, p64, g, s);
}

size_t nlist_layout(mhip_nlist *nl, int64_t nq, int k, bool masked, bool d2, char *base) {
    Carve c{base};
    nl->idx = c.take<uint32_t>(nq * k);
    nl->h64 = c.take<double>(nq);
    nl->rowrec = c.take<RowRec>(nq);
    nl->tau = c.take<float>(nq);
    nl->h = c.take<float>(nq);
    nl->status = c.take<int32_t>(nq);
    nl->amb = c.take<uint32_t>(nq + 1);
    nl->defer = c.take<uint32_t>(nq / WAVE + 2);
    nl->qsorted = masked ? c.take<uint32_t>(nq) : nullptr;
    nl->qrow = masked ? c.take<uint32_t>(nq) : nullptr;
    nl->d2 = d2 ? c.take<float>(nq * k) : nullptr;
    return c.off;
}

static int nl_reserve(mhip_ctx *ctx, mhip_nlist *nl, int64_t nq, int k, bool masked, bool d2) {
    const int rc = block_reserve(ctx, nl->mem, nlist_layout(nl, nq, k, masked, d2, nullptr), "neighbour list");
    if (rc) {
        nl->nq = 0;
        return rc;
    }
    nlist_layout(nl, nq, k, masked, d2, nl->mem.p);
    return 0;
}

// slots of the query rows qidx in sorted (Hilbert) order: qsorted[s] is the
// sorted-space particle of slot s, qrow[s] its row in qidx
static int query_setup(mhip_ctx *ctx, const mhip_index *ix, const int64_t *qidx, int64_t nq, mhip_nlist *nl) {
    ProfRegion pr(ctx, "knn_query_setup");
    int rc = 0;
    size_t cw = radix_counts_words(nq);
    char *s = (char *)scratch(ctx, nq * 24 + cw * 4, &rc);
    if (!s) return rc;
    uint64_t *k0 = (uint64_t *)s, *k1 = k0 + nq;
    uint32_t *v0 = (uint32_t *)(k1 + nq), *v1 = v0 + nq, *counts = v1 + nq;
    if ((rc = ensure_iperm(ctx, ix))) return rc;
    hipLaunchKernelGGL(k_qsetup_mask, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, ctx->stream, qidx, nq,
                       ix->iperm, k0, v0);
    int bits = 1;
    while (bits < 32 && ((int64_t)1 << bits) < ix->n) bits++;
    uint64_t *ks;
    uint32_t *vs;
    if ((rc = radix_sort_pairs(ctx, k0, v0, k1, v1, counts, nq, bits, &ks, &vs))) return rc;
    hipLaunchKernelGGL(k_qsetup_finish, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, ctx->stream, ks, vs,
                       nq, nl->qsorted, nl->qrow);
    return 0;
}

static TreeView tree_view(const mhip_index *ix) {
    TreeView t;
    t.sx = ix->sx;
    t.sy = ix->sy;
    t.sz = ix->sz;
    t.lx = ix->lx;
    t.ly = ix->ly;
    t.lz = ix->lz;
    t.nodes = ix->nodes;
    t.first_leaf = ix->first_leaf;
    t.nleaf = ix->nleaf;
    t.depth = ix->depth;
    const bool per = ix->box > 0;
    t.box = per ? (float)ix->box : 0.f;
    t.half = per ? 0.5f * (float)ix->box : 0.f;
    float m = per ? (float)ix->box : 0.f;
    for (int c = 0; c < 6; c++) m = fmaxf(m, fabsf(ix->bbox[c]));
    t.slack = ix->pos_f64 ? 2.4e-7f * m : 0.f;  // 4 ulp of the largest |coordinate|
    return t;
}

int knn_run(mhip_ctx *ctx, const mhip_index *ix, const int64_t *qidx, int64_t nq, int k,
            const double *m_rows, const float *seed_h, const float *seed_r, float *h_out,
            float *rho_out, float *vol_out, int32_t *status_out, int flags, mhip_nlist *nl) {
    if (k < 2) return fail(ctx, -1, "des_ngb must be at least 2");
    if (k > 128) return fail(ctx, -4, "des_ngb above 128 is not supported by the GPU kNN");
    if (k > ix->n) return fail(ctx, -1, "des_ngb exceeds the number of particles");
    if (!qidx) nq = ix->n;
    if (nq < 1) return fail(ctx, -1, "no query rows");
    int rc = 0;
    if ((rc = nl_reserve(ctx, nl, nq, k, qidx != nullptr, (flags & 1) != 0))) return rc;
    nl->nq = nq;
    nl->k = k;
    nl->index = ix;
    nl->has_d2 = (flags & 1) != 0;
    // query slots in Hilbert order
    const bool masked = qidx != nullptr;
    nl->masked = masked;
    if (masked && (rc = query_setup(ctx, ix, qidx, nq, nl))) {
        nl->nq = 0;
        return rc;
    }
    KnnArgs a;
    a.t = tree_view(ix);
    const bool per = ix->box > 0;
    a.qsorted = masked ? nl->qsorted : nullptr;
    a.qrow = masked ? nl->qrow : nullptr;
    a.perm = ix->perm;
    a.nq = nq;
    a.n = ix->n;
    a.k = k;
    a.dim = ix->dim;
    a.seed_h = seed_h;
    a.seed_r = seed_r;
    a.redo = 0;
    a.status_out = status_out;
    a.tau = nl->tau;
    a.h_slot = nl->h;
    a.h64_slot = nl->h64;
    a.st_slot = nl->status;
    a.nl_idx = nl->idx;
    a.nl_d2 = nl->has_d2 ? nl->d2 : nullptr;
    a.stats = ctx->prof >= 2 ? ctx->stats : nullptr;
    a.amb = nl->amb;
    a.defer = nl->defer;
    a.split = false;
    a.wlcap = (flags & MHIP_KNN_SMALL_RECORD) ? 8u : (uint32_t)WLCAP;
    const bool p64 = ix->pos_f64 != 0;
    const dim3 g((unsigned)((nq + KNN_BLOCK - 1) / KNN_BLOCK));
    hipStream_t s = ctx->stream;
    hipLaunchKernelGGL(k_lists_reset, dim3(1), dim3(64), 0, s, nl->amb, nl->defer);
    ProfRegion pr1(ctx, "knn_main");
    // seeds and the test hooks belong to the main kernel
    const bool wave = !seed_h && !seed_r && !(flags & (MHIP_KNN_SMALL_RECORD | MHIP_KNN_LANE)) &&
                      knn_wave_serves(ix->n, nq, k, ix->dim, per);
    if (wave) {
        if ((rc = knn_wave_launch(ctx, a, per, p64, false))) return rc;
    } else {
        if (!seed_h && !seed_r && !(flags & (MHIP_KNN_SMALL_RECORD | MHIP_KNN_LANE)))
            a.split = knn_splits(ix->n, nq, k, ix->dim, per);
        launch_main_k(a, p64, g, s);
        if (a.split && (rc = knn_wave_launch(ctx, a, per, p64, false))) return rc;
        if (seed_r) {
            // second launch: waves with a radius-seed miss are recomputed plainly
            KnnArgs r = a;
            r.redo = 1;
            launch_main_k(r, p64, g, s);
        }
        if ((rc = knn_wave_launch(ctx, a, per, p64, true))) return rc;
    }
    pr1.end();
    ProfRegion pr3(ctx, "knn_resolve");
    const dim3 gr((unsigned)std::min<int64_t>(RESOLVE_WAVES, (nq + 63) / 64));
    if (per) {
        if (p64)
            hipLaunchKernelGGL((k_knn_resolve<true, true, double>), gr, dim3(64), 0, s, a,
                               (const double *)ix->pos_in);
        else
            hipLaunchKernelGGL((k_knn_resolve<true, false, float>), gr, dim3(64), 0, s, a,
                               (const float *)ix->pos_in);
    } else {
        if (p64)
            hipLaunchKernelGGL((k_knn_resolve<false, true, double>), gr, dim3(64), 0, s, a,
                               (const double *)ix->pos_in);
        else
            hipLaunchKernelGGL((k_knn_resolve<false, false, float>), gr, dim3(64), 0, s, a,
                               (const float *)ix->pos_in);
    }
    pr3.end();
    if (status_out || h_out || rho_out || vol_out) {
        ProfRegion pr4(ctx, "knn_rows_out");
        const dim3 gq((unsigned)((nq + 255) / 256));
        hipLaunchKernelGGL(k_rows_rec, gq, dim3(256), 0, s, masked ? nl->qrow : ix->perm, nq, k, ix->dim, nl->h64,
                           nl->status, m_rows, nl->rowrec);
        hipLaunchKernelGGL(k_rows_split, gq, dim3(256), 0, s, nl->rowrec, nq, h_out, rho_out, vol_out, status_out);
    }
    return check_hip(ctx, hipGetLastError(), "knn launch");
}

// ---------------------------------------------------------------------------
// export: rows in output-row order, ascending (distance, original index),
// original particle indices -- the layout cKDTree.query returns.  A block
// holds EXP_ROWS consecutive slots: their distances and indices go to LDS
// once (the list's columns are read in 128-byte runs), then every entry
// counts the entries of its row that come before it (LDS reads that a row's
// lanes share) and is written there; a row's entries are contiguous, so the
// writes of a wavefront fall into a few whole lines.  One thread per row that
// formed every distance k times from global memory took 4.3 ms for 250000
// rows of 32 float64 distances; this takes 0.13 ms.
// ---------------------------------------------------------------------------
constexpr int EXP_ROWS = 32;

// dist2_of(slot, particle): squared distance of an entry (T: float or double)
template <typename T, typename F>
MHIP_DEV void export_rows(const uint32_t *__restrict__ idx, const uint32_t *__restrict__ qrow,
                          const uint32_t *__restrict__ perm, int64_t nq, int k, int32_t *__restrict__ ngb_out,
                          T *__restrict__ dist_out, char *lds, F dist2_of) {
    const int kp = k + 1;  // rows one entry apart: no common LDS bank
    T *s_d = (T *)lds;
    uint32_t *s_o = (uint32_t *)(s_d + EXP_ROWS * kp);
    for (int64_t slot0 = blockIdx.x * (int64_t)EXP_ROWS; slot0 < nq; slot0 += (int64_t)gridDim.x * EXP_ROWS) {
        for (int e = threadIdx.x; e < k * EXP_ROWS; e += 256) {
            const int r = e % EXP_ROWS, j = e / EXP_ROWS;
            const int64_t s = slot0 + r;
            if (s >= nq) continue;
            const uint32_t o = perm[idx[(int64_t)j * nq + s]];
            s_o[r * kp + j] = o;
            s_d[r * kp + j] = dist2_of(s, j, o);
        }
        __syncthreads();
        for (int e = threadIdx.x; e < k * EXP_ROWS; e += 256) {
            const int r = e / k, j = e % k;
            const int64_t s = slot0 + r;
            if (s >= nq) break;
            const T *d = s_d + r * kp;
            const uint32_t *o = s_o + r * kp;
            const T dj = d[j];
            const uint32_t oj = o[j];
            int rank = 0;
            for (int l = 0; l < k; l++) {
                const T dl = d[l];
                rank += dl < dj;
                // equal distances by index; repeated entries (padded rows) by place
                if (dl == dj) rank += o[l] < oj || (o[l] == oj && l < j);
            }
            const int64_t row = qrow ? qrow[s] : perm[s];
            if (ngb_out) ngb_out[row * k + rank] = (int32_t)oj;
            if (dist_out) dist_out[row * k + rank] = sqrt(dj);
        }
        __syncthreads();  // the next rows reuse the LDS
    }
}

static unsigned export_blocks(int64_t nq) {
    return (unsigned)std::min<int64_t>((nq + EXP_ROWS - 1) / EXP_ROWS, 1 << 20);
}

template <typename T>
static size_t export_lds(int k) { return (size_t)EXP_ROWS * (k + 1) * (sizeof(T) + sizeof(uint32_t)); }

__global__ __launch_bounds__(256) void k_export(const uint32_t *__restrict__ idx, const float *__restrict__ d2,
                                               const uint32_t *__restrict__ qrow,
                                               const uint32_t *__restrict__ perm, int64_t nq, int k,
                                               int32_t *__restrict__ ngb_out, float *__restrict__ dist_out) {
    extern __shared__ char s_exp[];
    export_rows<float>(idx, qrow, perm, nq, k, ngb_out, dist_out, s_exp,
                       [&](int64_t s, int j, uint32_t) { return d2[(int64_t)j * nq + s]; });
}

// ---------------------------------------------------------------------------
// rows of a full-set list for a subset of query rows.  A particle's k nearest
// neighbours, their distances and its smoothing length do not depend on
// which other particles are queried, so TreeUpdate with a particle_mask
// (src/meshoid/Meshoid.py:147-170) equals these rows of the unmasked list;
// density and volume use the subset's masses (Meshoid.py:169-170).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_nl_subset(
    const uint32_t *__restrict__ fidx, const float *__restrict__ fd2, const float *__restrict__ ftau,
    const float *__restrict__ fh, const double *__restrict__ fh64,
    const int32_t *__restrict__ fst, int64_t nfull, const uint32_t *__restrict__ qsorted,
    const uint32_t *__restrict__ qrow, int64_t nq, int k, int dim, const double *__restrict__ m_rows,
    uint32_t *__restrict__ idx, float *__restrict__ d2, float *__restrict__ tau,
    float *__restrict__ hs, double *__restrict__ hs64, int32_t *__restrict__ st, float *__restrict__ h_out,
    float *__restrict__ rho_out, float *__restrict__ vol_out, int32_t *__restrict__ status_out) {
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= nq) return;
    const uint32_t f = qsorted[s], row = qrow[s];
    for (int j = 0; j < k; j++) {
        idx[(int64_t)j * nq + s] = fidx[(int64_t)j * nfull + f];
        if (d2) d2[(int64_t)j * nq + s] = fd2[(int64_t)j * nfull + f];
    }
    const double h = fh64[f];
    tau[s] = ftau[f];
    hs[s] = fh[f];
    hs64[s] = h;
    st[s] = fst[f];
    // the main kernel's density and volume arithmetic
    const double vn = dim == 3 ? 4.18879020478639098 : (dim == 2 ? 3.14159265358979324 : 2.0);
    const double m = m_rows ? m_rows[row] : 1.0;
    const double hp = dim == 3 ? h * h * h : (dim == 2 ? h * h : h);
    const double rho = (double)k * m / (vn * hp);
    if (h_out) h_out[row] = (float)h;
    if (rho_out) rho_out[row] = (float)rho;
    if (vol_out) vol_out[row] = (float)(m / rho);
    if (status_out) status_out[row] = fst[f];
}

int nlist_subset(mhip_ctx *ctx, const mhip_nlist *full, const int64_t *qidx, int64_t nq, const double *m_rows,
                 float *h_out, float *rho_out, float *vol_out, int32_t *status_out, mhip_nlist *nl) {
    const mhip_index *ix = full->index;
    if (!ix || ix->n < 1 || full->nq < 1) return fail(ctx, -1, "neighbour list is empty");
    if (full->masked || full->nq != ix->n) return fail(ctx, -1, "the source list must cover every particle");
    if (nl == full) return fail(ctx, -1, "the subset needs a list of its own");
    if (nq < 1) return fail(ctx, -1, "no query rows");
    const int k = full->k;
    int rc = 0;
    if ((rc = nl_reserve(ctx, nl, nq, k, true, full->has_d2 != 0))) return rc;
    nl->nq = nq;
    nl->k = k;
    nl->index = ix;
    nl->has_d2 = full->has_d2;
    nl->masked = true;
    if ((rc = query_setup(ctx, ix, qidx, nq, nl))) {
        nl->nq = 0;
        return rc;
    }
    ProfRegion pr(ctx, "nlist_subset");
    hipLaunchKernelGGL(k_nl_subset, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, ctx->stream, full->idx,
                       full->has_d2 ? full->d2 : nullptr, full->tau, full->h, full->h64, full->status,
                       full->nq, nl->qsorted, nl->qrow, nq, k, ix->dim, m_rows, nl->idx,
                       full->has_d2 ? nl->d2 : nullptr, nl->tau, nl->h, nl->h64, nl->status, h_out, rho_out,
                       vol_out, status_out);
    return check_hip(ctx, hipGetLastError(), "subset launch");
}

// The same rows with float64 distances recomputed from the caller's
// positions (original indices), the distance cKDTree.query returns
// (src/meshoid/Meshoid.py:157): d = sqrt((dx^2 + dy^2) + dz^2) of the float64
// offsets, minimum image when periodic; rows ascending by (distance, index).
template <typename PT, bool PER>
__global__ __launch_bounds__(256) void k_export64(const uint32_t *__restrict__ idx, const uint32_t *__restrict__ qsorted,
                                                 const uint32_t *__restrict__ qrow, const uint32_t *__restrict__ perm,
                                                 const PT *__restrict__ pos, int dim, double box, int64_t nq, int k,
                                                 int32_t *__restrict__ ngb_out, double *__restrict__ dist_out) {
    extern __shared__ char s_exp[];
    export_rows<double>(idx, qrow, perm, nq, k, ngb_out, dist_out, s_exp, [&](int64_t s, int, uint32_t o) {
        return exact_d2<PT, PER>(pos, dim, perm[qsorted ? qsorted[s] : (uint32_t)s], o, box);
    });
}

int nlist_export64(mhip_ctx *ctx, const mhip_nlist *nl, int32_t *ngb_out, double *dist_out) {
    const mhip_index *ix = nl->index;
    if (!ix || ix->n < 1 || nl->nq < 1) return fail(ctx, -1, "neighbour list is empty");
    if (!ix->pos_in) return fail(ctx, -1, "the index holds no positions");
    ProfRegion pr(ctx, "nlist_export64");
    const dim3 g(export_blocks(nl->nq)), b(256);
    const size_t lds = export_lds<double>(nl->k);
    const uint32_t *qs = nl->masked ? nl->qsorted : nullptr, *qr = nl->masked ? nl->qrow : nullptr;
    const bool per = ix->box > 0;
#define MHIP_EXP(PT, P)                                                                                        \
    hipLaunchKernelGGL((k_export64<PT, P>), g, b, lds, ctx->stream, nl->idx, qs, qr, ix->perm, (const PT *)ix->pos_in, \
                       ix->dim, ix->box, nl->nq, nl->k, ngb_out, dist_out)
    if (ix->pos_f64) {
        if (per) MHIP_EXP(double, true);
        else MHIP_EXP(double, false);
    } else {
        if (per) MHIP_EXP(float, true);
        else MHIP_EXP(float, false);
    }
#undef MHIP_EXP
    return check_hip(ctx, hipGetLastError(), "export launch");
}

// the list's float64 smoothing lengths in output-row order
__global__ __launch_bounds__(256) void k_rows_h64(const double *__restrict__ h64, const uint32_t *__restrict__ qrow,
                                                 const uint32_t *__restrict__ perm, int64_t nq,
                                                 double *__restrict__ out) {
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= nq) return;
    out[qrow ? qrow[s] : perm[s]] = h64[s];
}

int nlist_hsml(mhip_ctx *ctx, const mhip_nlist *nl, double *h_out) {
    if (!nl->index || nl->index->n < 1 || nl->nq < 1) return fail(ctx, -1, "neighbour list is empty");
    hipLaunchKernelGGL(k_rows_h64, dim3((unsigned)((nl->nq + 255) / 256)), dim3(256), 0, ctx->stream, nl->h64,
                       nl->masked ? nl->qrow : nullptr, nl->index->perm, nl->nq, h_out);
    return check_hip(ctx, hipGetLastError(), "hsml copy launch");
}

// h, density and volume of the rows in float64 (Meshoid.py:165-170) and their
// status: as k_rows_rec and k_rows_split, one scattered record per row (two
// 16-byte writes to one 32-byte sector), then a coalesced split
struct __align__(16) RowRec64 {
    double h, rho, vol;
    int32_t status, pad;
};
__global__ __launch_bounds__(256) void k_rows64_rec(const uint32_t *__restrict__ srow, int64_t nq, int k, int dim,
                                                   const double *__restrict__ h64, const int32_t *__restrict__ st,
                                                   const double *__restrict__ m_rows, RowRec64 *__restrict__ rec) {
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= nq) return;
    const uint32_t r = srow[s];
    const double h = h64[s];
    const double vn = dim == 3 ? 4.18879020478639098 : (dim == 2 ? 3.14159265358979324 : 2.0);
    const double m = m_rows ? m_rows[r] : 1.0;
    const double hp = dim == 3 ? h * h * h : (dim == 2 ? h * h : h);
    const double rho = (double)k * m / (vn * hp);
    rec[r] = RowRec64{h, rho, m / rho, st[s], 0};
}

__global__ __launch_bounds__(256) void k_rows64_split(const RowRec64 *__restrict__ rec, int64_t nq,
                                                     double *__restrict__ h, double *__restrict__ rho,
                                                     double *__restrict__ vol, int32_t *__restrict__ status) {
    const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r >= nq) return;
    const RowRec64 v = rec[r];
    if (h) h[r] = v.h;
    if (rho) rho[r] = v.rho;
    if (vol) vol[r] = v.vol;
    if (status) status[r] = v.status;
}

int nlist_rows64(mhip_ctx *ctx, const mhip_nlist *nl, const double *m_rows, double *h, double *rho, double *vol,
                 int32_t *status) {
    const mhip_index *ix = nl->index;
    if (!ix || ix->n < 1 || nl->nq < 1) return fail(ctx, -1, "neighbour list is empty");
    int rc = 0;
    RowRec64 *rec = (RowRec64 *)scratch(ctx, (size_t)nl->nq * sizeof(RowRec64), &rc);
    if (!rec) return rc;
    ProfRegion pr(ctx, "nlist_rows64");
    const dim3 g((unsigned)((nl->nq + 255) / 256));
    hipLaunchKernelGGL(k_rows64_rec, g, dim3(256), 0, ctx->stream, nl->masked ? nl->qrow : ix->perm, nl->nq, nl->k,
                       ix->dim, nl->h64, nl->status, m_rows, rec);
    hipLaunchKernelGGL(k_rows64_split, g, dim3(256), 0, ctx->stream, rec, nl->nq, h, rho, vol, status);
    return check_hip(ctx, hipGetLastError(), "row output launch");
}

int nlist_export(mhip_ctx *ctx, const mhip_nlist *nl, int32_t *ngb_out, float *dist_out) {
    const mhip_index *ix = nl->index;
    if (!ix || ix->n < 1 || nl->nq < 1) return fail(ctx, -1, "neighbour list is empty");
    if (!nl->has_d2) return fail(ctx, -1, "neighbour list was built without distances");
    ProfRegion pr(ctx, "nlist_export");
    hipLaunchKernelGGL(k_export, dim3(export_blocks(nl->nq)), dim3(256),
                       export_lds<float>(nl->k), ctx->stream,
                       nl->idx, nl->d2, nl->masked ? nl->qrow : nullptr, ix->perm, nl->nq, nl->k,
                       ngb_out, dist_out);
    return check_hip(ctx, hipGetLastError(), "export launch");
}

// ---------------------------------------------------------------------------
// nearest particle of arbitrary float64 points: cKDTree.query(x)[1], k = 1
// (src/meshoid/Meshoid.py:409).  The points are first put in the index's
// Hilbert order, so that a wavefront's 64 lanes serve a compact block of
// points.  (1) Each lane finds, by binary search over the leaves' first
// sort keys, the leaf where its point's key falls, and scans it and its
// two neighbours (in Hilbert order these usually hold the nearest particle):
// every lane starts with a tight bound.  (2) A wave-uniform walk, inside out
// from the middle lane's leaf (its siblings, then the rest of the
// grandparent's subtree, ... up to the root), tests each node once for all
// lanes and scans the leaves some lane's bound (widened by the float32
// rounding band) reaches; it keeps the nearest and the second-nearest
// float32 d2.  (3) Where those two lie closer than float32 rounding can
// order, the band is re-ranked with float64 distances from the caller's
// positions (the distance cKDTree computes), ties to the lowest original
// index.  The point is split into float32 hi + lo parts, so its float32
// distances are as accurate as those between two particles.
// ---------------------------------------------------------------------------
struct NearestArgs {
    TreeView t;
    const uint32_t *order;  // point of each thread (Hilbert order), null = identity
    const uint32_t *perm;
    const void *pos_in;
    int64_t n;
    int dim;
    double box;        // > 0: periodic in [0, box)
    float org[3], scale;  // the index's key quantisation frame
    const double *tg;  // (nt, dim) row-major
    int64_t nt;
    int64_t *out;      // original particle index per point, -1 for a non-finite point
    unsigned long long *stats;  // work counters, may be null
    const uint64_t *leaf_key;   // first key of each leaf, on the bits the index is sorted on
};

template <typename PT, bool PER>
MHIP_DEV double exact_d2_point(const PT *pos, int dim, uint32_t j, const double (&tp)[3], double box) {
    double s = 0.0;
    for (int c = 0; c < dim; c++) {
        double d = (double)pos[(int64_t)j * dim + c] - tp[c];
        if (PER) d = wrap<double>(d, box);
        s = __dadd_rn(s, __dmul_rn(d, d));
    }
    return s;
}

// sort key of each point in the index's quantisation frame (as the
// particles' keys are formed), periodic points wrapped into the box first
__global__ __launch_bounds__(256) void k_point_keys(const double *__restrict__ tg, int64_t nt, int dim,
                                                    double box, float ox, float oy, float oz, float scale,
                                                    uint64_t *__restrict__ keys, uint32_t *__restrict__ vals) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= nt) return;
    const float org[3] = {ox, oy, oz};
    uint32_t cc[3] = {0u, 0u, 0u};
    for (int c = 0; c < dim; c++) {
        double v = tg[i * dim + c];
        if (box > 0.0 && (v < 0.0 || v >= box)) v -= floor(v / box) * box;
        cc[c] = key_cell((float)v, org[c], scale);
    }
    keys[i] = hilbert_key(cc[0], cc[1], cc[2], dim);
    vals[i] = (uint32_t)i;
}

// sort key of sorted particle p, formed as the index build forms it
MHIP_DEV uint64_t particle_key(const TreeView &t, const float (&org)[3], float scale, int dim, int64_t p) {
    const float v[3] = {t.sx[p], t.sy[p], t.sz[p]};
    uint32_t cc[3] = {0u, 0u, 0u};
    for (int c = 0; c < dim; c++) cc[c] = key_cell(v[c], org[c], scale);
    return hilbert_key(cc[0], cc[1], cc[2], dim);
}

// first sort key of every leaf (on the bits the index is sorted on), for the
// points' first-leaf search
__global__ __launch_bounds__(256) void k_leaf_keys(TreeView t, float ox, float oy, float oz, float scale, int dim,
                                                  uint64_t *__restrict__ out) {
    const int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (l >= t.nleaf) return;
    const float org[3] = {ox, oy, oz};
    out[l] = particle_key(t, org, scale, dim, l * LEAF) >> key_sort_lo_bit(dim);
}

template <bool PER, bool P64, typename PT>
__global__ __launch_bounds__(256) void k_nearest(NearestArgs a) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t wave0 = tid - lane;
    if (wave0 >= a.nt) return;
    const bool live = tid < a.nt;
    // lanes past the end take the wave's first point (never written)
    const int64_t slot = live ? tid : wave0;
    const int64_t i = a.order ? (int64_t)a.order[slot] : slot;
    double tp[3] = {0.0, 0.0, 0.0};
    for (int c = 0; c < a.dim; c++) {
        double v = a.tg[i * a.dim + c];
        if (PER && (v < 0.0 || v >= a.box)) {
            v -= floor(v / a.box) * a.box;
            if (!(v >= 0.0 && v < a.box)) v = 0.0;  // rounded onto the upper edge
        }
        tp[c] = v;
    }
    QPos q;
    q.x = (float)tp[0];
    q.y = (float)tp[1];
    q.z = (float)tp[2];
    q.lx = (float)(tp[0] - (double)q.x);
    q.ly = (float)(tp[1] - (double)q.y);
    q.lz = (float)(tp[2] - (double)q.z);
    // box tests use the hi parts: the slack covers the point's lo parts and
    // (float64 particles) the particles' lo parts
    TreeView t = a.t;
    t.slack = a.t.slack + fmaxf(fabsf(q.lx), fmaxf(fabsf(q.ly), fabsf(q.lz)));
    QBox qb;
    qb.lx = q.x - t.slack;
    qb.ly = q.y - t.slack;
    qb.lz = q.z - t.slack;
    qb.hx = q.x + t.slack;
    qb.hy = q.y + t.slack;
    qb.hz = q.z + t.slack;
    const uint32_t first_leaf = (uint32_t)t.first_leaf;
    // (1) this lane's leaf: the last leaf whose first key is at most the
    // point's key (on the bits the index is sorted on); it and its neighbours
    // give the lane a first bound
    const int kshift = key_sort_lo_bit(a.dim);
    uint64_t kq = 0;
    {
        uint32_t cc[3] = {0u, 0u, 0u};
        for (int c = 0; c < a.dim; c++) cc[c] = key_cell((float)tp[c], a.org[c], a.scale);
        kq = hilbert_key(cc[0], cc[1], cc[2], a.dim) >> kshift;
    }
    uint32_t lo = 0, hi = (uint32_t)t.nleaf;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a.leaf_key[mid] <= kq)
            lo = mid;
        else
            hi = mid;
    }
    const uint32_t own_lo = lo > 0 ? lo - 1 : 0, own_hi = min(lo + 1, (uint32_t)t.nleaf - 1);
    float best = INFINITY, second = INFINITY;
    uint32_t bp = 0xffffffffu;
    float cx[LEAF], cy[LEAF], cz[LEAF], clx[LEAF], cly[LEAF], clz[LEAF];
    // candidates of one leaf; skip: this lane has the leaf already
    auto take = [&](int64_t leaf, bool skip) {
#pragma unroll
        for (int j = 0; j < LEAF; j++) {
            // padding particles carry NaN coordinates: never below a bound
            const float d2 = dist2<PER, true>(t, q, cx[j], cy[j], cz[j], clx[j], cly[j], clz[j]);
            const bool nb = !skip && d2 < best;
            second = nb ? best : (skip ? second : fminf(second, d2));
            best = nb ? d2 : best;
            bp = nb ? (uint32_t)(leaf * LEAF + j) : bp;
        }
    };
    auto scan = [&](uint32_t node) {
        const int64_t leaf = node - first_leaf;
        load_leaf_uniform<P64>(t.sx, t.sy, t.sz, t.lx, t.ly, t.lz, leaf, cx, cy, cz, clx, cly, clz);
        take(leaf, leaf >= own_lo && leaf <= own_hi);
    };
    for (uint32_t l = own_lo; l <= own_hi; l++) {
        load_leaf<P64>(t, l, cx, cy, cz, clx, cly, clz);
        take(l, false);
    }
    // the middle lane's leaf, for every lane
    const uint32_t x = first_leaf + uniform(__shfl(lo, WAVE / 2));
    uint32_t n_nodes = 0, n_leaves = 1;
    scan(x);
    // (2) wave-uniform walk, inside out: the subtree of each ancestor of the
    // middle lane's leaf in turn (parent, grandparent, ... root), minus the
    // subtree already done, depth first (children in index order) and pruned
    // by every lane's bound.  A node's 8 children are tested together (their
    // boxes loaded at once) into a mask; a leaf is tested again with the
    // bound of the moment before it is scanned.  A leaf inside a child that
    // the bound of the moment would have pruned lies in that child's box, so
    // the leaf test prunes it too: the leaves scanned, and their order, are
    // those of a walk that tests each node just before entering it.
    const float F = (1.0f + BAND_REL) * PRUNE_REL;
    uint32_t done = x;  // scanned
    while (done != 0) {
        const uint32_t top = (done - 1) >> 3;
        MaskStack ms;
        ms.put(0, expand_mask<PER>(t, qb, top, best * F) & ~(1u << (done - (FANOUT * top + 1))));
        n_nodes += FANOUT;
        int lvl = 0;
        uint32_t cur = top;
        while (true) {
            const uint32_t m = ms.get(lvl);
            if (m == 0u) {
                if (lvl == 0) break;
                lvl--;
                cur = (cur - 1) >> 3;
                continue;
            }
            const uint32_t c = (uint32_t)__builtin_ctz(m);
            ms.clear(lvl, c);
            const uint32_t y = FANOUT * cur + 1 + c;
            if (y >= first_leaf) {
                if (y - first_leaf < t.nleaf && __any(box_gap2_u<PER>(t, qb, y) <= best * F)) {
                    scan(y);
                    n_leaves++;
                }
                continue;
            }
            lvl++;
            cur = y;
            ms.put(lvl, expand_mask<PER>(t, qb, y, best * F));
            n_nodes += FANOUT;
        }
        done = top;
    }
    if (a.stats) {
        const bool ex = live && bp != 0xffffffffu && second <= best * (1.0f + AMBIG_REL);
        const uint32_t nex = (uint32_t)__popcll(__ballot(ex));
        if (lane == 0) {
            atomicAdd(a.stats + STAT_NN_WAVES, 1ull);
            atomicAdd(a.stats + STAT_NN_NODES, (unsigned long long)n_nodes);
            atomicAdd(a.stats + STAT_NN_LEAVES, (unsigned long long)n_leaves);
            atomicAdd(a.stats + STAT_NN_EXACT, (unsigned long long)nex);
        }
    }
    if (!live) return;
    int64_t res = -1;
    if (bp != 0xffffffffu) {
        res = a.perm[bp];
        if (second <= best * (1.0f + AMBIG_REL)) {
            // (3) float64 re-rank of this point's rounding band (rare; per lane)
            const PT *pos = (const PT *)a.pos_in;
            const float lim = best * (1.0f + BAND_REL);
            double be = INFINITY;
            uint32_t bo = 0xffffffffu;
            uint32_t y = 0;
            bool more = true;
            while (more) {
                if (node_d2<PER>(t, q, y) <= lim * PRUNE_REL) {
                    if (y < first_leaf) {
                        y = FANOUT * y + 1;
                        continue;
                    }
                    if (y - first_leaf < t.nleaf) {
                        const int64_t leaf = y - first_leaf;
                        load_leaf<P64>(t, leaf, cx, cy, cz, clx, cly, clz);
                        for (int j = 0; j < LEAF; j++) {
                            const int64_t p = leaf * LEAF + j;
                            const float d2 = dist2<PER, true>(t, q, cx[j], cy[j], cz[j], clx[j], cly[j], clz[j]);
                            if (d2 <= lim && p < a.n) {
                                const uint32_t o = a.perm[p];
                                const double e = exact_d2_point<PT, PER>(pos, a.dim, o, tp, a.box);
                                if (e < be || (e == be && o < bo)) {
                                    be = e;
                                    bo = o;
                                }
                            }
                        }
                    }
                }
                more = next_after(y);
            }
            res = bo;
        }
    }
    a.out[i] = res;
}

int nearest_run(mhip_ctx *ctx, const mhip_index *ix, const double *targets, int64_t nt, int dim,
                int64_t *out) {
    if (!ix || ix->n < 1) return fail(ctx, -1, "the index holds no particles");
    if (dim != ix->dim) return fail(ctx, -1, "point dimension differs from the particles'");
    if (nt < 0) return fail(ctx, -1, "negative point count");
    if (nt == 0) return 0;
    NearestArgs a;
    a.t = tree_view(ix);
    a.order = nullptr;
    a.perm = ix->perm;
    a.pos_in = ix->pos_in;
    a.n = ix->n;
    a.dim = ix->dim;
    a.box = ix->box > 0 ? ix->box : 0.0;
    for (int c = 0; c < 3; c++) a.org[c] = ix->frame[c];
    a.scale = ix->frame[3];
    a.tg = targets;
    a.nt = nt;
    a.out = out;
    a.stats = ctx->prof >= 2 ? ctx->stats : nullptr;
    const bool per = ix->box > 0, p64 = ix->pos_f64 != 0;
    const dim3 g((unsigned)((nt + 255) / 256));
    hipStream_t s = ctx->stream;
    // scratch: the points' sort (large sets), then the leaves' first keys
    const bool sort_pts = nt >= 4096 && nt <= 0xffffffffll;
    const size_t cw = sort_pts ? radix_counts_words(nt) : 0;
    const size_t pts_bytes = sort_pts ? (((size_t)nt * 24 + cw * 4 + 255) & ~(size_t)255) : 0;
    int rc = 0;
    char *sc = (char *)scratch(ctx, pts_bytes + (size_t)ix->nleaf * sizeof(uint64_t), &rc);
    if (!sc) return rc;
    uint64_t *lkey = (uint64_t *)(sc + pts_bytes);
    a.leaf_key = lkey;
    if (sort_pts) {
        // points in the index's Hilbert order
        ProfRegion pk(ctx, "nearest_sort");
        uint64_t *k0 = (uint64_t *)sc, *k1 = k0 + nt;
        uint32_t *v0 = (uint32_t *)(k1 + nt), *v1 = v0 + nt, *counts = v1 + nt;
        hipLaunchKernelGGL(k_point_keys, g, dim3(256), 0, s, targets, nt, dim, a.box, ix->frame[0], ix->frame[1],
                           ix->frame[2], ix->frame[3], k0, v0);
        uint64_t *ks;
        uint32_t *vs;
        if ((rc = radix_sort_pairs(ctx, k0, v0, k1, v1, counts, nt, KEY_BITS_PER_AXIS * dim, &ks, &vs,
                                   key_sort_lo_bit(dim))))
            return rc;
        a.order = vs;
    }
    ProfRegion pr(ctx, "nearest");
    hipLaunchKernelGGL(k_leaf_keys, dim3((unsigned)((ix->nleaf + 255) / 256)), dim3(256), 0, s, a.t, a.org[0],
                       a.org[1], a.org[2], a.scale, a.dim, lkey);
    if (per) {
        if (p64)
            hipLaunchKernelGGL((k_nearest<true, true, double>), g, dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_nearest<true, false, float>), g, dim3(256), 0, s, a);
    } else {
        if (p64)
            hipLaunchKernelGGL((k_nearest<false, true, double>), g, dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_nearest<false, false, float>), g, dim3(256), 0, s, a);
    }
    return check_hip(ctx, hipGetLastError(), "nearest launch");
}

}  // namespace mhip
