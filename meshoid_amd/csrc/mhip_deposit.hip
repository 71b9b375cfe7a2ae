// Surface density of a particle quantity on a grid of sightlines.
//
// Replaces
//   Meshoid.SurfaceDensity                   src/meshoid/Meshoid.py:595-643
//   GridSurfaceDensity (parallel split/sum)  src/meshoid/grid_deposition.py:123-184
//   GridSurfaceDensity_core                  src/meshoid/grid_deposition.py:187-229
//   GridSurfaceDensity_conservative_core     src/meshoid/grid_deposition.py:232-295
//   kernel2d                                 src/meshoid/kernel_density.py:60-68
//   Meshoid.DepositToGrid                    src/meshoid/Meshoid.py:557-593
//   GridDensity                              src/meshoid/grid_deposition.py:534-603
//   kernel3d                                 src/meshoid/kernel_density.py:71-79
//
// Each particle adds kernel2d(r/h) f / h^2 to every grid point (spacing
// size/(res-1), point 0 at center - size/2) within h of its projected
// position; the conservative variant divides each particle's weights by
// their sum and scales the grid by 1/dx^2 at the end.  Accumulation is
// float64.  Up to res = 128 every block keeps a private copy of the whole
// map in LDS (float64 LDS atomics, 128 KB) for an interleaved share of the
// particles and adds it to the HBM map once at the end: the many particles
// of a clump that land on the same few cells contend in LDS, not in L2.
// Larger maps (and every GridDensity volume) are binned: particles are
// sorted by the brick (32^2 map cells, 8^3 volume cells) that holds the
// first cell of their footprint, and each block takes a run of the sorted
// particles; a brick's run of at least BIN_DENSE particles accumulates in an
// LDS window (the brick plus the footprint reach above it, 4096 cells) that
// is added to the HBM map once, shorter runs take float64 atomics in HBM.  In
// the window a footprint below WAVE_CELLS cells is one lane's work and a larger
// one a wavefront's, a cell per lane.  Footprints wider than the window are
// deposited tile by tile of the map, again a wavefront each.
//
// float64 arithmetic bounds all of it, about 45 vector instructions a cell, 21
// of them float64.  2^22 clustered particles, radii of 32 neighbours: the
// 1024^2 map 9.8 -> 2.6 ms (windows 2.25 -> 0.64, wide footprints 7.16 -> 1.77:
// one block per particle ran at the rate of float64 atomics in L2), the 128^3
// volume 4.3 -> 1.1 ms.
#include "mhip_internal.hpp"

namespace mhip {

constexpr int DEP_THREADS = 256;
constexpr int64_t BIG_CELLS = 1024;           // footprint handled by one thread at most
constexpr int DEP_TILE = 128;                 // map side held whole in LDS (128 KB of float64)
constexpr double KERNEL2D_NORM = 1.8189136353359467;  // 40 / (7 pi)

// binned deposition
// sorted particles per block: a block of large footprints is the launch's tail
// (2048 a block: 1.5 and 1.6 ms for map and volume, 512: 0.70 and 1.07, 256:
// 0.64 and 0.90)
constexpr int BIN_CHUNK = 256;
// a brick's run of this many particles in a block uses the window (64, 32, 16:
// 1.15, 1.13, 1.11 ms of the volume)
constexpr int BIN_DENSE = 16;
constexpr int WIN_CELLS = 4096;   // LDS window, float64 cells (32 KB)
constexpr int BRICK2 = 32, WIN2 = 64;  // maps: brick side, window side (footprint span <= 33)
constexpr int BRICK3 = 8, WIN3 = 16;   // volumes: brick side, window side (span <= 9)
static_assert(WIN2 * WIN2 == WIN_CELLS && WIN3 * WIN3 * WIN3 == WIN_CELLS, "window size");
// sort keys: brick << SIZE_BITS | (SIZE_MAX_RANK - min(footprint cells,
// SIZE_MAX_RANK)), so a brick's particles come widest first and the small
// ones in order: a wavefront's 64 lanes finish together (from WAVE_CELLS on
// the order no longer matters)
constexpr int SIZE_BITS = 6;
constexpr uint32_t SIZE_MAX_RANK = (1u << SIZE_BITS) - 1;
// conservative footprints up to this many cells (4^2, 2^3: the narrowest, h of
// two spacings on a map and one in a volume) keep their weights in registers
// between the total and the deposit; at 27 cells the registers halved the
// wavefronts in flight (volume 1.24 ms against 1.16)
constexpr int WCACHE2 = 16, WCACHE3 = 8;
// in the window, footprints of at least this many cells are deposited by a
// whole wavefront, a cell per lane (up to WAVE_CACHE turns of it keep their
// weights in registers); smaller ones by one lane each.  By one lane all, a
// background particle's ~340 cells kept a few lanes of one block busy at the end
// (volume 3.5 ms against 1.9); 32 and 64 measure alike.
constexpr int WAVE_CELLS = 64;
constexpr int WAVE_CACHE = 8;
static_assert(WAVE_CELLS <= SIZE_MAX_RANK + 1, "footprints one lane deposits are told apart by size");

struct DepArgs {
    const void *f, *pos, *h;
    int f_f64, pos_f64, h_f64, dim;
    int64_t n;
    double smooth, hmin;  // h used = min(max(smooth h, hmin), 1e100)
    double ox, oy;        // center - size/2: the position of grid point 0
    double dx;            // size / (res - 1)
    int res, conservative;
    double *grid;           // (res, res), [gx][gy]
    uint32_t *big, *nbig;   // wide particles and their number (whole-map path)
    int nb;                 // bricks per axis (binned path)
};

// The cubic spline of r^2 at 1/h: 2 (1-q)_+^3 - (1-2q)_+^3, q = r / h, the same
// function as its two branches (and 0 beyond q = 1) without them; r from the
// reciprocal square root and one Newton step (a correctly rounded root gives
// the same errors of the maps).  18 float64 instructions, where sqrt's own
// expansion and both branches took about 40; r^2 below 1e-300 counts as 1e-300
// (q = 0 to rounding).  Offsets and r^2 are rounded as the reference rounds
// them: where a footprint's few points all lie near r = h, 1 - q multiplies a
// last-place difference by ten.
MHIP_DEV double spline_r2(double r2, double hinv) {
    r2 = fmax(r2, 1e-300);
    const double y = __builtin_amdgcn_rsq(r2);
    double r = r2 * y;
    r = fma(0.5 * y, fma(-r, r, r2), r);
    const double q = r * hinv, a = fmax(1.0 - q, 0.0), b = fmax(fma(-2.0, q, 1.0), 0.0);
    return fma(a + a, a * a, -(b * b * b));
}

template <typename T>
MHIP_DEV double ld(const void *p, int64_t i) {
    return (double)((const T *)p)[i];
}

struct Foot {
    double xs0, xs1, hinv, w;  // projected position, 1/h, factor of the spline's value
    int gx0, gx1, gy0, gy1;
};

// grid index range of int((x -/+ h) / dx (+ 1)) as the reference forms it
// (truncation toward zero, then clipped to the grid)
MHIP_DEV int lo_index(double a, int res) {
    if (!(a > 0.0)) return 0;
    return a >= (double)res ? res : (int)a;
}
MHIP_DEV int hi_index(double b, int res) {
    if (!(b > -1.0)) return -1;
    return b >= (double)(res - 1) ? res - 1 : (int)b;
}

// false: nothing to deposit (non-finite input or footprint off the grid)
MHIP_DEV bool footprint(const DepArgs &a, int64_t i, Foot &fp) {
    const double x0 = a.pos_f64 ? ld<double>(a.pos, i * a.dim) : ld<float>(a.pos, i * a.dim);
    const double x1 = a.pos_f64 ? ld<double>(a.pos, i * a.dim + 1) : ld<float>(a.pos, i * a.dim + 1);
    const double hv = a.h_f64 ? ld<double>(a.h, i) : ld<float>(a.h, i);
    const double fv = a.f_f64 ? ld<double>(a.f, i) : ld<float>(a.f, i);
    fp.xs0 = (x0 - a.ox);
    fp.xs1 = (x1 - a.oy);
    double hs = fmin(fmax(a.smooth * hv, a.hmin), 1e100);
    if (a.conservative) hs = fmax(hs, a.dx);
    if (!(hs > 0.0) || !isfinite(fp.xs0) || !isfinite(fp.xs1) || !isfinite(fv)) return false;
    fp.hinv = 1.0 / hs;
    // conservative: shares of f, in which the kernel's constant cancels
    fp.w = a.conservative ? fv : KERNEL2D_NORM * (fv * fp.hinv * fp.hinv);
    fp.gx0 = lo_index((fp.xs0 - hs) / a.dx + 1.0, a.res);
    fp.gx1 = hi_index((fp.xs0 + hs) / a.dx, a.res);
    fp.gy0 = lo_index((fp.xs1 - hs) / a.dx + 1.0, a.res);
    fp.gy1 = hi_index((fp.xs1 + hs) / a.dx, a.res);
    return fp.gx0 <= fp.gx1 && fp.gy0 <= fp.gy1;
}

// offset of grid line g from the particle, per axis
MHIP_DEV double line_off(double xs, int g, double dx) { return xs - g * dx; }

// kernel weight at grid point (gx, gy) without the kernel's constant, 0 when
// it lies beyond h
MHIP_DEV double cell_weight(const DepArgs &a, const Foot &fp, int gx, int gy) {
    const double x = line_off(fp.xs0, gx, a.dx), y = line_off(fp.xs1, gy, a.dx);
    return spline_r2(x * x + y * y, fp.hinv);
}

// visit(gx, gy, weight) over the cells [gx0, gx1] x [gy0, gy1]
template <typename F>
MHIP_DEV void each_cell(const DepArgs &a, const Foot &fp, int gx0, int gx1, int gy0, int gy1, F visit) {
    for (int gx = gx0; gx <= gx1; gx++)
        for (int gy = gy0; gy <= gy1; gy++) visit(gx, gy, cell_weight(a, fp, gx, gy));
}

// conservative variant: the particle's total weight over its (clipped)
// footprint, by which each weight is divided; 1 for the plain variant
MHIP_DEV double foot_total(const DepArgs &a, const Foot &fp) {
    if (!a.conservative) return 1.0;
    double tot = 0.0;
    each_cell(a, fp, fp.gx0, fp.gx1, fp.gy0, fp.gy1, [&](int, int, double k) { tot += k; });
    return tot;
}

// lane l's value of v in every lane (l uniform)
MHIP_DEV int lane_value(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
MHIP_DEV double lane_value(double v, int l) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
MHIP_DEV Foot lane_foot(const Foot &f, int l) {
    Foot r;
    r.xs0 = lane_value(f.xs0, l);
    r.xs1 = lane_value(f.xs1, l);
    r.hinv = lane_value(f.hinv, l);
    r.w = lane_value(f.w, l);
    r.gx0 = lane_value(f.gx0, l);
    r.gx1 = lane_value(f.gx1, l);
    r.gy0 = lane_value(f.gy0, l);
    r.gy1 = lane_value(f.gy1, l);
    return r;
}

MHIP_DEV double wave_sum(double v) {
    for (int o = WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    return v;
}

// The walk of `stride` lanes (a wavefront, a block) over a box of cells, a cell
// per lane in row-major order: lane l starts at cell l and moves on by `stride`
// cells at a time, rows and planes by carries (one division per box, where a
// division per cell would cost more than the weight).
struct Walk2 {
    int x, y;  // the lane's cell
    int sx, sy, wy, x1, y1;
    MHIP_DEV void start(int lane, int stride, int x0, int y0, int x1_, int y1_) {
        x1 = x1_;
        y1 = y1_;
        wy = y1 - y0 + 1;
        const int row = lane / wy;
        sx = stride / wy;
        sy = stride - sx * wy;
        x = x0 + row;
        y = y0 + (lane - row * wy);
    }
    MHIP_DEV bool inside() const { return x <= x1; }
    MHIP_DEV void next() {
        x += sx;
        y += sy;
        if (y > y1) {
            y -= wy;
            x++;
        }
    }
};

struct Walk3 {
    int x, y, z;
    int sx, sy, sz, wy, wz, x1, y1, z1;
    MHIP_DEV void start(int lane, int stride, const int *lo, const int *hi) {
        x1 = hi[0];
        y1 = hi[1];
        z1 = hi[2];
        wy = y1 - lo[1] + 1;
        wz = z1 - lo[2] + 1;
        const int row = lane / wz, srow = stride / wz, plane = row / wy;
        sz = stride - srow * wz;
        sx = srow / wy;
        sy = srow - sx * wy;
        x = lo[0] + plane;
        y = lo[1] + (row - plane * wy);
        z = lo[2] + (lane - row * wz);
    }
    MHIP_DEV bool inside() const { return x <= x1; }
    MHIP_DEV void next() {
        x += sx;
        y += sy;
        z += sz;
        if (z > z1) {
            z -= wz;
            y++;
        }
        if (y > y1) {
            y -= wy;
            x++;
        }
    }
};

// The cells of one particle by a whole wavefront: weight(walk) is the weight
// of the lane's present cell, add(walk, share) deposits its share.
// Conservative shares are weight / (sum of the weights), plain ones the weight.
template <typename Walk, typename W, typename A>
MHIP_DEV void wave_spread(const Walk &w0, int ncell, bool conservative, W weight, A add) {
    if (!conservative) {
        for (Walk w = w0; w.inside(); w.next()) {
            const double k = weight(w);
            if (k != 0.0) add(w, k);
        }
    } else if (ncell <= WAVE * WAVE_CACHE) {
        double wc[WAVE_CACHE], tot = 0.0;
        Walk w = w0;
#pragma unroll
        for (int t = 0; t < WAVE_CACHE; t++) {
            wc[t] = 0.0;
            if (t * WAVE < ncell) {
                if (w.inside()) wc[t] = weight(w);
                tot += wc[t];
                w.next();
            }
        }
        tot = wave_sum(tot);
        if (!(tot > 0.0)) return;
        const double inv = 1.0 / tot;
        w = w0;
#pragma unroll
        for (int t = 0; t < WAVE_CACHE; t++)
            if (t * WAVE < ncell) {
                if (wc[t] != 0.0) add(w, wc[t] * inv);
                w.next();
            }
    } else {
        double tot = 0.0;
        for (Walk w = w0; w.inside(); w.next()) tot += weight(w);
        tot = wave_sum(tot);
        if (!(tot > 0.0)) return;
        const double inv = 1.0 / tot;
        for (Walk w = w0; w.inside(); w.next()) {
            const double k = weight(w);
            if (k != 0.0) add(w, k * inv);
        }
    }
}

// block b: map tile (b % ntile) (tw x tw cells held in LDS) and particle
// chunk (b / ntile), the chunk being every nchunk-th run of 256 particles
// (interleaved, so that a clump's particles, stored together, spread over
// all chunks instead of piling onto one block's LDS atomics); it deposits the
// cells of its tile only, and adds the tile to the HBM map once at the end
__global__ __launch_bounds__(DEP_THREADS) void k_deposit_tiles(DepArgs a, int tw, int ntx, int nchunk) {
    extern __shared__ double sg[];
    const int ntile = ntx * ntx;
    const int tile = blockIdx.x % ntile, chunk = blockIdx.x / ntile;
    const int tx0 = (tile / ntx) * tw, ty0 = (tile % ntx) * tw;
    const int tx1 = min(tx0 + tw, a.res) - 1, ty1 = min(ty0 + tw, a.res) - 1;
    for (int c = threadIdx.x; c < tw * tw; c += DEP_THREADS) sg[c] = 0.0;
    __syncthreads();
    for (int64_t i = (int64_t)chunk * DEP_THREADS + threadIdx.x; i < a.n; i += (int64_t)nchunk * DEP_THREADS) {
        Foot fp;
        if (!footprint(a, i, fp)) continue;
        const int64_t cells = (int64_t)(fp.gx1 - fp.gx0 + 1) * (fp.gy1 - fp.gy0 + 1);
        if (cells > BIG_CELLS) {
            // listed once, by the tile that holds its first cell; the list
            // holds n entries
            if (fp.gx0 >= tx0 && fp.gx0 <= tx1 && fp.gy0 >= ty0 && fp.gy0 <= ty1)
                a.big[atomicAdd(a.nbig, 1u)] = (uint32_t)i;
            continue;
        }
        if (a.conservative && ntx == 1 && cells <= WCACHE2) {
            // one tile holds the whole map (and footprint): small footprints
            // keep their weights in registers between the total (summed in
            // the order of the loop below) and the deposit
            double wc[WCACHE2];
            double tot = 0.0;
            int gx = fp.gx0, gy = fp.gy0;
#pragma unroll
            for (int c = 0; c < WCACHE2; c++) {
                wc[c] = 0.0;
                if (c < cells) {
                    wc[c] = cell_weight(a, fp, gx, gy);
                    tot += wc[c];
                    if (++gy > fp.gy1) {
                        gy = fp.gy0;
                        gx++;
                    }
                }
            }
            if (tot == 0.0) continue;
            const double inv = 1.0 / tot;
            gx = fp.gx0;
            gy = fp.gy0;
#pragma unroll
            for (int c = 0; c < WCACHE2; c++) {
                if (c < cells) {
                    if (wc[c] != 0.0) atomicAdd(&sg[(gx - tx0) * tw + (gy - ty0)], wc[c] * inv * fp.w);
                    if (++gy > fp.gy1) {
                        gy = fp.gy0;
                        gx++;
                    }
                }
            }
            continue;
        }
        const int gx0 = max(fp.gx0, tx0), gx1 = min(fp.gx1, tx1);
        const int gy0 = max(fp.gy0, ty0), gy1 = min(fp.gy1, ty1);
        if (gx0 > gx1 || gy0 > gy1) continue;
        // conservative: each weight over the particle's total weight (the
        // whole footprint, not only this tile's part)
        double tot = 1.0;
        if (a.conservative) {
            tot = foot_total(a, fp);
            if (tot == 0.0) continue;
        }
        const double inv = 1.0 / tot;
        each_cell(a, fp, gx0, gx1, gy0, gy1, [&](int gx, int gy, double k) {
            if (k != 0.0) atomicAdd(&sg[(gx - tx0) * tw + (gy - ty0)], k * inv * fp.w);
        });
    }
    __syncthreads();
    for (int c = threadIdx.x; c < tw * tw; c += DEP_THREADS) {
        const double v = sg[c];
        if (v != 0.0) atomicAdd(&a.grid[(int64_t)(tx0 + c / tw) * a.res + (ty0 + c % tw)], v);
    }
}

// ---------------------------------------------------------------------------
// Binned deposition.  A policy P gives, for its kind of grid:
//   key(a, i, cells)     the brick of particle i's first footprint cell (and
//                        the footprint's cells); skip(a) + that brick when the
//                        footprint is too large for the window (it goes to the
//                        tiles below), 2 skip(a) when there is none
//   direct(a, i)         deposit particle i with float64 atomics in HBM
//   foot(a, i, fp), cells(fp)   particle i's footprint and its cells
//   window(a, fp, k, w)  deposit a particle (brick k) into the LDS window w
//   window_wave(a, fp, l, k, w)   the same for lane l's, by the wavefront
//   flush(a, k, c, v)    add window cell c of brick k (value v) to the map
// ---------------------------------------------------------------------------
struct Map2 {
    using Args = DepArgs;
    static MHIP_DEV uint32_t skip(const DepArgs &a) { return (uint32_t)a.nb * (uint32_t)a.nb; }
    static MHIP_DEV uint32_t key(const DepArgs &a, int64_t i, uint32_t &cells) {
        Foot fp;
        cells = 0;
        if (!footprint(a, i, fp)) return 2 * skip(a);
        const uint32_t brick = (uint32_t)(fp.gx0 / BRICK2) * (uint32_t)a.nb + (uint32_t)(fp.gy0 / BRICK2);
        const int sx = fp.gx1 - fp.gx0 + 1, sy = fp.gy1 - fp.gy0 + 1;
        if (sx > WIN2 - BRICK2 + 1 || sy > WIN2 - BRICK2 + 1 || (int64_t)sx * sy > BIG_CELLS) {
            cells = SIZE_MAX_RANK;
            return skip(a) + brick;
        }
        cells = (uint32_t)(sx * sy);
        return brick;
    }
    static MHIP_DEV void direct(const DepArgs &a, uint32_t i) {
        Foot fp;
        footprint(a, i, fp);  // keyed, so it has a footprint
        const double tot = foot_total(a, fp);
        if (tot == 0.0) return;
        const double inv = 1.0 / tot;
        each_cell(a, fp, fp.gx0, fp.gx1, fp.gy0, fp.gy1, [&](int gx, int gy, double k) {
            if (k != 0.0) atomicAdd(&a.grid[(int64_t)gx * a.res + gy], k * inv * fp.w);
        });
    }
    // the window holds cells [ox, ox + 64) x [oy, oy + 64) of the brick's
    // origin (ox, oy); a keyed footprint starts inside the brick and spans at
    // most 33 cells per axis, so it stays inside.  A lane goes round its
    // footprint from a cell of its own: the particles of a clump, stored
    // together, cover the same few cells, and lanes in step would add to one
    // address 64 at a time.
    using F = Foot;
    static MHIP_DEV bool foot(const DepArgs &a, uint32_t i, F &fp) { return footprint(a, i, fp); }
    static MHIP_DEV int cells(const F &fp) { return (fp.gx1 - fp.gx0 + 1) * (fp.gy1 - fp.gy0 + 1); }
    // lane l's particle, by the whole wavefront
    static MHIP_DEV void window_wave(const DepArgs &a, const F &mine, int l, uint32_t key, double *win) {
        const F fp = lane_foot(mine, l);
        const int ox = (int)(key / (uint32_t)a.nb) * BRICK2, oy = (int)(key % (uint32_t)a.nb) * BRICK2;
        const int origin = ox * WIN2 + oy;
        Walk2 w;
        w.start(threadIdx.x % WAVE, WAVE, fp.gx0, fp.gy0, fp.gx1, fp.gy1);
        wave_spread(
            w, cells(fp), a.conservative != 0, [&](const Walk2 &c) { return cell_weight(a, fp, c.x, c.y); },
            [&](const Walk2 &c, double k) { atomicAdd(&win[c.x * WIN2 + c.y - origin], k * fp.w); });
    }
    static MHIP_DEV void window(const DepArgs &a, const F &fp, uint32_t key, double *win) {
        const int ox = (int)(key / (uint32_t)a.nb) * BRICK2, oy = (int)(key % (uint32_t)a.nb) * BRICK2;
        const int wx = fp.gx1 - fp.gx0 + 1, wy = fp.gy1 - fp.gy0 + 1, ncell = wx * wy;
        const uint32_t lane = threadIdx.x % WAVE;
        const int gxs = fp.gx0 + (int)(lane / (uint32_t)wy % (uint32_t)wx), gys = fp.gy0 + (int)(lane % (uint32_t)wy);
        int gx = gxs, gy = gys;
        auto next = [&]() {
            if (++gy > fp.gy1) {
                gy = fp.gy0;
                if (++gx > fp.gx1) gx = fp.gx0;
            }
        };
        if (a.conservative && ncell <= WCACHE2) {
            // small footprints: the weights stay in registers between the
            // total and the deposit
            double wc[WCACHE2];
            double tot = 0.0;
#pragma unroll
            for (int c = 0; c < WCACHE2; c++) {
                wc[c] = 0.0;
                if (c < ncell) {
                    wc[c] = cell_weight(a, fp, gx, gy);
                    tot += wc[c];
                    next();
                }
            }
            if (tot == 0.0) return;
            const double inv = 1.0 / tot;
            gx = gxs;
            gy = gys;
#pragma unroll
            for (int c = 0; c < WCACHE2; c++) {
                if (c < ncell) {
                    if (wc[c] != 0.0) atomicAdd(&win[(gx - ox) * WIN2 + (gy - oy)], wc[c] * inv * fp.w);
                    next();
                }
            }
            return;
        }
        const double tot = foot_total(a, fp);
        if (tot == 0.0) return;
        const double inv = 1.0 / tot;
        for (int c = 0; c < ncell; c++) {
            const double k = cell_weight(a, fp, gx, gy);
            if (k != 0.0) atomicAdd(&win[(gx - ox) * WIN2 + (gy - oy)], k * inv * fp.w);
            next();
        }
    }
    static MHIP_DEV void flush(const DepArgs &a, uint32_t key, int c, double v) {
        const int gx = (int)(key / (uint32_t)a.nb) * BRICK2 + c / WIN2;
        const int gy = (int)(key % (uint32_t)a.nb) * BRICK2 + c % WIN2;
        if (gx < a.res && gy < a.res) atomicAdd(&a.grid[(int64_t)gx * a.res + gy], v);
    }

    // ---- tiles of WIN2^2 cells
    static constexpr int SIDE = WIN2;
    // (ms by cells a tile, direct / tiles: 32768^2 630 3.3 / 5.9, 5000 14.0 / 9.5;
    // 16384^2 800 2.1 / 2.6, 2500 2.3 / 2.1)
    static constexpr int TILE_CELLS = 2000;
    // this thread's share (of `stride`) of the cells, straight into the grid
    static MHIP_DEV void spread(const DepArgs &a, const F &fp, double inv, int thread, int stride) {
        const double f = fp.w * inv;
        Walk2 w;
        for (w.start(thread, stride, fp.gx0, fp.gy0, fp.gx1, fp.gy1); w.inside(); w.next()) {
            const double k = cell_weight(a, fp, w.x, w.y);
            if (k != 0.0) atomicAdd(&a.grid[(int64_t)w.x * a.res + w.y], k * f);
        }
    }
    static MHIP_DEV void box(const F &fp, int *lo, int *hi) {
        lo[0] = fp.gx0;
        hi[0] = fp.gx1;
        lo[1] = fp.gy0;
        hi[1] = fp.gy1;
        lo[2] = hi[2] = 0;
    }
    static MHIP_DEV void corner(int64_t tile, int nt, int *t0) {
        t0[0] = (int)(tile / nt) * SIDE;
        t0[1] = (int)(tile % nt) * SIDE;
        t0[2] = 0;
    }
    static MHIP_DEV bool meets(const DepArgs &, const int *lo, const int *hi, const int *t0) {
        return lo[0] < t0[0] + SIDE && hi[0] >= t0[0] && lo[1] < t0[1] + SIDE && hi[1] >= t0[1];
    }
    // this thread's share (of `stride`) of the sum of the weights
    static MHIP_DEV double total(const DepArgs &a, const F &fp, int thread, int stride) {
        Walk2 w;
        double tot = 0.0;
        for (w.start(thread, stride, fp.gx0, fp.gy0, fp.gx1, fp.gy1); w.inside(); w.next())
            tot += cell_weight(a, fp, w.x, w.y);
        return tot;
    }
    static MHIP_DEV void tile_wave(const DepArgs &a, const F &mine, double inv, int l, const int *t0, double *win) {
        const F fp = lane_foot(mine, l);
        const double f = a.conservative ? fp.w * lane_value(inv, l) : fp.w;
        const int origin = t0[0] * SIDE + t0[1];
        Walk2 w;
        w.start(threadIdx.x % WAVE, WAVE, max(fp.gx0, t0[0]), max(fp.gy0, t0[1]), min(fp.gx1, t0[0] + SIDE - 1),
                min(fp.gy1, t0[1] + SIDE - 1));
        for (; w.inside(); w.next()) {
            const double k = cell_weight(a, fp, w.x, w.y);
            if (k != 0.0) atomicAdd(&win[w.x * SIDE + w.y - origin], k * f);
        }
    }
    static MHIP_DEV void tile_flush(const DepArgs &a, const int *t0, int c, double v) {
        const int gx = t0[0] + c / SIDE, gy = t0[1] + c % SIDE;
        atomicAdd(&a.grid[(int64_t)gx * a.res + gy], v);
    }
};

template <class P>
__global__ __launch_bounds__(256) void k_bin_keys(typename P::Args a, uint64_t *__restrict__ keys,
                                                  uint32_t *__restrict__ vals) {
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= a.n) return;
    uint32_t cells;
    const uint32_t b = P::key(a, i, cells);
    keys[i] = (uint64_t)b << SIZE_BITS | (SIZE_MAX_RANK - min(cells, SIZE_MAX_RANK));
    vals[i] = (uint32_t)i;
}

MHIP_DEV int first_not_below(const uint32_t *s, int m, uint32_t k) {
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s[mid] < k)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

MHIP_DEV int first_above(const uint32_t *s, int m, uint32_t k) {
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s[mid] <= k)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// block b: sorted particles [b BIN_CHUNK, (b + 1) BIN_CHUNK).  Their bricks'
// runs (lengths from binary searches of the block's keys in LDS) shorter
// than BIN_DENSE are deposited straight into HBM; each longer run is
// deposited into the LDS window by the whole block and added to the map
// once (cells still zero are skipped), the window cleared as it is read
template <class P>
__global__ __launch_bounds__(DEP_THREADS) void k_bin_deposit(typename P::Args a, const uint64_t *__restrict__ keys,
                                                             const uint32_t *__restrict__ vals) {
    __shared__ double win[WIN_CELLS];
    __shared__ uint32_t skey[BIN_CHUNK];
    __shared__ uint32_t runs[BIN_CHUNK / BIN_DENSE];  // offset | length << 16
    __shared__ uint32_t s_nrun;
    const int64_t cs = (int64_t)blockIdx.x * BIN_CHUNK;
    const int m = (int)min<int64_t>(BIN_CHUNK, a.n - cs);
    const uint32_t skip = P::skip(a);
    for (int c = threadIdx.x; c < WIN_CELLS; c += DEP_THREADS) win[c] = 0.0;
    for (int e = threadIdx.x; e < m; e += DEP_THREADS) skey[e] = (uint32_t)(keys[cs + e] >> SIZE_BITS);
    if (threadIdx.x == 0) s_nrun = 0u;
    __syncthreads();
    for (int e = threadIdx.x; e < m; e += DEP_THREADS) {
        const uint32_t k = skey[e];
        if (k >= skip) break;  // the rest is wider than a window, or nothing
        const int lo = first_not_below(skey, m, k), hi = first_above(skey, m, k);
        if (hi - lo >= BIN_DENSE) {
            // at most BIN_CHUNK / BIN_DENSE runs this long
            if (e == lo) runs[atomicAdd(&s_nrun, 1u)] = (uint32_t)lo | (uint32_t)(hi - lo) << 16;
        } else {
            P::direct(a, vals[cs + e]);
        }
    }
    __syncthreads();
    const uint32_t nrun = s_nrun;
    for (uint32_t r = 0; r < nrun; r++) {
        const int lo = (int)(runs[r] & 0xffffu), len = (int)(runs[r] >> 16);
        const uint32_t k = skey[lo];
        // lane l of wavefront w: particle 4 l + w of each 256 (a brick's
        // particles come largest first, so the four share the large ones)
        const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
        for (int b = 0; b < len; b += DEP_THREADS) {
            const int e = b + lane * (DEP_THREADS / WAVE) + wave;
            typename P::F fp;
            const bool has = e < len && P::foot(a, vals[cs + lo + e], fp);
            const bool wide = has && P::cells(fp) >= WAVE_CELLS;
            for (uint64_t todo = __ballot(wide); todo; todo &= todo - 1)
                P::window_wave(a, fp, __builtin_ctzll(todo), k, win);
            if (has && !wide) P::window(a, fp, k, win);
        }
        __syncthreads();
        for (int c = threadIdx.x; c < WIN_CELLS; c += DEP_THREADS) {
            const double v = win[c];
            if (v != 0.0) {
                P::flush(a, k, c, v);
                win[c] = 0.0;
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Footprints wider than a window.  The grid is cut into tiles of SIDE^dim =
// 4096 cells held in LDS; a block goes over its share of the wide particles,
// keeps those that meet its tile and deposits, a wavefront per particle and a
// cell per lane, the cells inside.  Tile and particle meet by tests on boxes
// of cells, 64 groups of 64 particles at once and then the particles of a
// group, so no list of pairs is made; the particles are in brick order, so a
// group's box is little larger than one footprint.  On large grids a tile would
// meet a vanishing part of the groups, and the tests, tiles times groups, would
// cost more than the deposit: there runs of 64 groups have boxes too, and only
// the groups of those that meet the tile are tested (at least
// WIDE_BLOCKS tiles; 2^22 particles 40 cells wide on a map of 32768^2 114 -> 17
// ms, 12 cells wide in a volume of 1024^3 295 -> 64 ms).
// One block per particle adding each cell to HBM runs at the rate of float64
// atomics in L2, 1.1e11 a second; here they stay in LDS and each tile is added
// once per block.  That rate is the better one only where the tiles of a large
// grid get few cells each (P::TILE_CELLS on average): a tile's tests, clearing and
// reading cost as much as those atomics.  k_wide_boxes sums the footprints,
// k_wide_direct or k_wide_tiles does the work.
// ---------------------------------------------------------------------------
struct Wide {
    const uint32_t *list;  // the particles, count of them from list[range[0]]
    uint32_t *range;       // first, count; then room for cells (binned grids)
    int *boxes;            // (groups, 6): lowest and highest cell on each axis
    int *runs;             // the same of each 64 groups; null: not tested
    double *inv;           // 1 / total weight by place in the list; null: plain shares
    // sum of the footprints' cells (of a particle at most 2^31 counted); null:
    // the tiles in any case
    unsigned long long *cells;
};

// whether the wide particles are few enough to add their cells to HBM
template <class P>
MHIP_DEV bool wide_few(const Wide &wd, int64_t ntile) {
    return wd.cells && *wd.cells < (unsigned long long)ntile * P::TILE_CELLS;
}

// first of the sorted keys (brick << SIZE_BITS | size) with brick >= k, by a
// wavefront: 64 splits of the range at a time
MHIP_DEV int64_t wave_lower_bound(const uint64_t *__restrict__ keys, int64_t n, uint32_t k) {
    const int lane = threadIdx.x % WAVE;
    int64_t lo = 0, hi = n;  // the answer is in [lo, hi]
    while (lo < hi) {
        const int64_t step = (hi - lo + WAVE - 1) / WAVE;
        const int64_t p = lo + lane * step;
        const int below = __popcll(__ballot(p < hi && (uint32_t)(keys[p] >> SIZE_BITS) < k));
        if (below == 0) return lo;
        const int64_t last = lo + (below - 1) * step;  // below k
        hi = min(hi, last + step);
        lo = last + 1;
    }
    return lo;
}

__global__ __launch_bounds__(WAVE) void k_wide_range(const uint64_t *__restrict__ keys, int64_t n, uint32_t skip,
                                                     uint32_t *__restrict__ range) {
    const int64_t lo = wave_lower_bound(keys, n, skip), hi = wave_lower_bound(keys, n, 2 * skip);
    if (threadIdx.x == 0) {
        range[0] = (uint32_t)lo;
        range[1] = (uint32_t)(hi - lo);
        range[2] = range[3] = 0u;  // Wide::cells
    }
}

MHIP_DEV int wave_min_i(int v) {
    for (int o = WAVE / 2; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, WAVE));
    return v;
}
MHIP_DEV int wave_max_i(int v) {
    for (int o = WAVE / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, WAVE));
    return v;
}

// the groups' boxes, a wavefront per group
template <class P>
__global__ __launch_bounds__(DEP_THREADS) void k_wide_boxes(typename P::Args a, Wide wd) {
    const uint32_t first = wd.range[0], count = wd.range[1];
    const int lane = threadIdx.x % WAVE;
    const uint32_t ng = (uint32_t)(((uint64_t)count + WAVE - 1) / WAVE);
    const uint32_t stride = gridDim.x * (DEP_THREADS / WAVE);
    for (uint32_t g = blockIdx.x * (DEP_THREADS / WAVE) + threadIdx.x / WAVE; g < ng; g += stride) {
        const int64_t e = (int64_t)g * WAVE + lane;
        typename P::F fp;
        int lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
        double cells = 0.0;
        if (e < count && P::foot(a, wd.list[first + e], fp)) {
            P::box(fp, lo, hi);
            cells = 1.0;
            for (int c = 0; c < 3; c++) cells *= (double)hi[c] - (double)lo[c] + 1.0;
        }
        if (wd.cells) {
            cells = wave_sum(fmin(cells, 2147483648.0));
            if (lane == 0) atomicAdd(wd.cells, (unsigned long long)cells);
        }
        for (int c = 0; c < 3; c++) {
            const int l = wave_min_i(lo[c]), h = wave_max_i(hi[c]);
            if (lane == 0) {
                wd.boxes[(size_t)g * 6 + c] = l;
                wd.boxes[(size_t)g * 6 + 3 + c] = h;
            }
        }
    }
}

// the boxes of each 64 groups, a wavefront per run
__global__ __launch_bounds__(DEP_THREADS) void k_wide_runs(Wide wd) {
    const int lane = threadIdx.x % WAVE;
    const int64_t ng = ((int64_t)wd.range[1] + WAVE - 1) / WAVE, nrun = (ng + WAVE - 1) / WAVE;
    const int64_t stride = (int64_t)gridDim.x * (DEP_THREADS / WAVE);
    for (int64_t r = blockIdx.x * (int64_t)(DEP_THREADS / WAVE) + threadIdx.x / WAVE; r < nrun; r += stride) {
        const int64_t g = min(r * WAVE + lane, ng - 1);
        for (int c = 0; c < 3; c++) {
            const int l = wave_min_i(wd.boxes[g * 6 + c]), h = wave_max_i(wd.boxes[g * 6 + 3 + c]);
            if (lane == 0) {
                wd.runs[r * 6 + c] = l;
                wd.runs[r * 6 + 3 + c] = h;
            }
        }
    }
}

// conservative: 1 / (sum of the weights), a block per particle
template <class P>
__global__ __launch_bounds__(DEP_THREADS) void k_wide_totals(typename P::Args a, Wide wd) {
    __shared__ double part[DEP_THREADS / WAVE];
    const uint32_t first = wd.range[0], count = wd.range[1];
    for (uint32_t e = blockIdx.x; e < count; e += gridDim.x) {
        typename P::F fp;
        P::foot(a, wd.list[first + e], fp);  // listed, so it has a footprint
        const double p = wave_sum(P::total(a, fp, threadIdx.x, DEP_THREADS));
        if (threadIdx.x % WAVE == 0) part[threadIdx.x / WAVE] = p;
        __syncthreads();
        if (threadIdx.x == 0) {
            double tot = 0.0;
            for (int w = 0; w < DEP_THREADS / WAVE; w++) tot += part[w];
            wd.inv[e] = tot > 0.0 ? 1.0 / tot : 0.0;
        }
        __syncthreads();
    }
}

// a block per particle, every cell added to the grid
template <class P>
__global__ __launch_bounds__(DEP_THREADS) void k_wide_direct(typename P::Args a, Wide wd, int64_t ntile) {
    if (!wide_few<P>(wd, ntile)) return;
    const uint32_t first = wd.range[0], count = wd.range[1];
    for (uint32_t e = blockIdx.x; e < count; e += gridDim.x) {
        typename P::F fp;
        P::foot(a, wd.list[first + e], fp);  // listed, so it has a footprint
        P::spread(a, fp, wd.inv ? wd.inv[e] : 1.0, threadIdx.x, DEP_THREADS);
    }
}

// block b: tile b % ntile, groups b / ntile, + nslice, ... of the wide
// particles (neighbouring groups meet the same tiles, so each of a tile's
// blocks gets its share of them).  The block's four wavefronts go over the
// same groups and take every fourth particle.
template <class P>
__global__ __launch_bounds__(DEP_THREADS) void k_wide_tiles(typename P::Args a, Wide wd, int nt, int64_t ntile,
                                                            int nslice) {
    __shared__ double win[WIN_CELLS];
    if (wide_few<P>(wd, ntile)) return;
    const uint32_t first = wd.range[0], count = wd.range[1];
    const int64_t ng = ((int64_t)count + WAVE - 1) / WAVE;
    // runs of 64 groups of this slice
    const int64_t nrun = (ng + (int64_t)WAVE * nslice - 1) / ((int64_t)WAVE * nslice);
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int64_t b = blockIdx.x; b < ntile * nslice; b += gridDim.x) {
        const int slice = (int)(b / ntile);
        int t0[3];
        P::corner(b % ntile, nt, t0);
        // whether 64 groups, and this lane's of them, meet the tile
        auto run_meets = [&](int64_t r) {
            return r < nrun && (!wd.runs || P::meets(a, wd.runs + r * 6, wd.runs + r * 6 + 3, t0));
        };
        auto group_meets = [&](int64_t g) {
            return g < ng && P::meets(a, wd.boxes + g * 6, wd.boxes + g * 6 + 3, t0);
        };
        bool any = false;
        for (int64_t r0 = wave * WAVE; r0 < nrun && !any; r0 += DEP_THREADS)
            for (uint64_t rs = __ballot(run_meets(r0 + lane)); rs && !any; rs &= rs - 1)
                any = __any(group_meets(((r0 + __builtin_ctzll(rs)) * WAVE + lane) * nslice + slice));
        if (!__syncthreads_or(any)) continue;
        for (int c = threadIdx.x; c < WIN_CELLS; c += DEP_THREADS) win[c] = 0.0;
        __syncthreads();
        for (int64_t r0 = 0; r0 < nrun; r0 += WAVE) {
            for (uint64_t rs = __ballot(run_meets(r0 + lane)); rs; rs &= rs - 1) {
                const int64_t g0 = (r0 + __builtin_ctzll(rs)) * WAVE * nslice + slice;
                const bool near = group_meets(g0 + (int64_t)nslice * lane);
                for (uint64_t gs = __ballot(near); gs; gs &= gs - 1) {
                    const int64_t e = (g0 + (int64_t)nslice * __builtin_ctzll(gs)) * WAVE + lane;
                    typename P::F fp;
                    double inv = 1.0;
                    bool take = e < count && lane % (DEP_THREADS / WAVE) == wave && P::foot(a, wd.list[first + e], fp);
                    if (take) {
                        int lo[3], hi[3];
                        P::box(fp, lo, hi);
                        take = P::meets(a, lo, hi, t0);
                        if (wd.inv) {
                            inv = wd.inv[e];
                            take = take && inv != 0.0;
                        }
                    }
                    for (uint64_t ps = __ballot(take); ps; ps &= ps - 1)
                        P::tile_wave(a, fp, inv, __builtin_ctzll(ps), t0, win);
                }
            }
        }
        __syncthreads();
        for (int c = threadIdx.x; c < WIN_CELLS; c += DEP_THREADS) {
            const double v = win[c];
            if (v != 0.0) P::tile_flush(a, t0, c, v);
        }
        __syncthreads();
    }
}

// the wide particles list[range[0] .. + range[1]) into the map.  At least
// WIDE_BLOCKS blocks, so that a few tiles still fill the chip; a block whose
// groups meet nothing ends after the box tests.
// (Map of 1024^2: 2048, 4096, 8192 blocks 2.61, 2.50, 2.62 ms.)
constexpr int64_t WIDE_BLOCKS = 4096;
template <class P>
void wide_deposit(mhip_ctx *ctx, typename P::Args a, Wide wd, int64_t ntile) {
    hipStream_t s = ctx->stream;
    const int64_t ng = (a.n + WAVE - 1) / WAVE;
    const int nt = (a.res + P::SIDE - 1) / P::SIDE;
    const int nslice = (int)std::min<int64_t>(ng, std::max<int64_t>(1, WIDE_BLOCKS / ntile));
    const bool large = ntile >= WIDE_BLOCKS;
    if (large) wd.cells = (unsigned long long *)(wd.range + 2);
    hipLaunchKernelGGL(k_wide_boxes<P>, dim3((unsigned)std::min<int64_t>(1024, (ng + 3) / 4)), dim3(DEP_THREADS), 0, s,
                       a, wd);
    if (large) {
        wd.runs = wd.boxes + ng * 6;
        hipLaunchKernelGGL(k_wide_runs, dim3((unsigned)std::min<int64_t>(1024, (ng / WAVE + 4) / 4)), dim3(DEP_THREADS),
                           0, s, wd);
    }
    if (wd.inv)
        hipLaunchKernelGGL(k_wide_totals<P>, dim3((unsigned)std::min<int64_t>(4096, a.n)), dim3(DEP_THREADS), 0, s, a,
                           wd);
    if (large)
        hipLaunchKernelGGL(k_wide_direct<P>, dim3((unsigned)std::min<int64_t>(4096, a.n)), dim3(DEP_THREADS), 0, s, a,
                           wd, ntile);
    hipLaunchKernelGGL(k_wide_tiles<P>, dim3((unsigned)std::min<int64_t>(1 << 22, ntile * nslice)), dim3(DEP_THREADS),
                       0, s, a, wd, nt, ntile, nslice);
}

// bits of a sort key in [0, top]
static int key_bits(uint32_t top) { return 64 - __builtin_clzll((unsigned long long)top | 1ull); }

// words the boxes of n particles' groups and runs take
static size_t box_words(int64_t n) { return ((size_t)n / WAVE + 1 + (size_t)n / (WAVE * WAVE) + 1) * 6; }
// scratch for n particles: keys 16 n, values 8 n (room for the boxes), radix
// counts, the wide particles' range.  The totals and boxes take the halves of
// the keys and values that the sort leaves free.
static size_t val_words(int64_t n) { return std::max((size_t)n, box_words(n)); }
static size_t bin_scratch_bytes(int64_t n) {
    return (size_t)n * 16 + val_words(n) * 8 + radix_counts_words(std::max<int64_t>(n, 1)) * 4 + 16 + 64;
}

// the binned path: keys, sort, runs, then the tiles of the wide particles
template <class P>
int bin_deposit(mhip_ctx *ctx, typename P::Args a, uint32_t skip, int64_t ntile, bool conservative, char *sc) {
    const int64_t n = a.n;
    if (n <= 0) return 0;
    uint64_t *k0 = (uint64_t *)sc, *k1 = k0 + n;
    uint32_t *v0 = (uint32_t *)(k1 + n), *v1 = v0 + val_words(n), *range = v1 + val_words(n), *counts = range + 4;
    hipStream_t s = ctx->stream;
    hipLaunchKernelGGL(k_bin_keys<P>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, k0, v0);
    uint64_t *ks;
    uint32_t *vs;
    int rc = radix_sort_pairs(ctx, k0, v0, k1, v1, counts, n, key_bits(2 * skip) + SIZE_BITS, &ks, &vs);
    if (rc) return rc;
    hipLaunchKernelGGL(k_bin_deposit<P>, dim3((unsigned)((n + BIN_CHUNK - 1) / BIN_CHUNK)), dim3(DEP_THREADS), 0, s,
                       a, ks, vs);
    hipLaunchKernelGGL(k_wide_range, dim3(1), dim3(WAVE), 0, s, ks, n, skip, range);
    const Wide wd{vs, range, (int *)(vs == v0 ? v1 : v0), nullptr, conservative ? (double *)(ks == k0 ? k1 : k0) : nullptr,
                  nullptr};
    wide_deposit<P>(ctx, a, wd, ntile);
    return 0;
}

__global__ __launch_bounds__(256) void k_grid_fill(double *__restrict__ g, int64_t n, double v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        g[i] = v;
}

__global__ __launch_bounds__(256) void k_grid_scale(double *__restrict__ g, int64_t n, double s) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        g[i] *= s;
}

__global__ void k_range_zero(uint32_t *range) {
    if (threadIdx.x < 2) range[threadIdx.x] = 0u;
}

// ---------------------------------------------------------------------------
// GridDensity: 3-D conservative deposition.  Grid point g at
// center - size/2 + dx/2 + g dx (dx = size/(res-1)); each particle spreads f
// over the points of its cube footprint with weights kernel3d(r/h) / (their
// sum), and the map is divided by dx^3.  Periodic boxes wrap the indices
// (g mod res) instead of clipping them.  kernel3d is the compact-support
// spline: 0 beyond r = h (the reference leaves it unassigned there).
// ---------------------------------------------------------------------------
constexpr int64_t BIG_CELLS_3D = 512;

struct Dep3Args {
    const void *f, *pos, *h;
    int f_f64, pos_f64, h_f64;
    int64_t n;
    double hmin;        // h used = min(max(h, hmin), 1e100)
    double ox, oy, oz;  // position of grid point 0
    double dx;
    int res, periodic;
    double *grid;  // (res, res, res)
    int nb;  // bricks per axis
};

struct Foot3 {
    double x[3], hinv, f;
    int g0[3], g1[3];
};

MHIP_DEV bool footprint3(const Dep3Args &a, int64_t i, Foot3 &fp) {
    const double o[3] = {a.ox, a.oy, a.oz};
    for (int c = 0; c < 3; c++)
        fp.x[c] = (a.pos_f64 ? ld<double>(a.pos, i * 3 + c) : ld<float>(a.pos, i * 3 + c)) - o[c];
    const double hv = a.h_f64 ? ld<double>(a.h, i) : ld<float>(a.h, i);
    fp.f = a.f_f64 ? ld<double>(a.f, i) : ld<float>(a.f, i);
    const double hs = fmin(fmax(hv, a.hmin), 1e100);
    if (!(hs > 0.0) || !isfinite(fp.x[0]) || !isfinite(fp.x[1]) || !isfinite(fp.x[2]) || !isfinite(fp.f))
        return false;
    fp.hinv = 1.0 / hs;
    for (int c = 0; c < 3; c++) {
        const double lo = (fp.x[c] - hs) / a.dx + 1.0, hi = (fp.x[c] + hs) / a.dx;
        if (a.periodic) {
            // unclipped int() (truncation toward zero); the footprint spans at
            // most 2 h / dx + 1 points, h <= the map's extent in practice
            if (!(fabs(lo) < 1e9 && fabs(hi) < 1e9)) return false;
            fp.g0[c] = (int)lo;
            fp.g1[c] = (int)hi;
        } else {
            fp.g0[c] = lo_index(lo, a.res);
            fp.g1[c] = hi_index(hi, a.res);
        }
        if (fp.g0[c] > fp.g1[c]) return false;
    }
    return true;
}

MHIP_DEV Foot3 lane_foot(const Foot3 &f, int l) {
    Foot3 r;
    for (int c = 0; c < 3; c++) {
        r.x[c] = lane_value(f.x[c], l);
        r.g0[c] = lane_value(f.g0[c], l);
        r.g1[c] = lane_value(f.g1[c], l);
    }
    r.hinv = lane_value(f.hinv, l);
    r.f = lane_value(f.f, l);
    return r;
}

// kernel weight without the kernel's constant, which cancels in the shares
MHIP_DEV double weight3(const Dep3Args &a, const Foot3 &fp, int gx, int gy, int gz) {
    const double x = line_off(fp.x[0], gx, a.dx), y = line_off(fp.x[1], gy, a.dx), z = line_off(fp.x[2], gz, a.dx);
    return spline_r2(x * x + y * y + z * z, fp.hinv);
}

// visit(gx, gy, gz, weight) over the footprint
template <typename F>
MHIP_DEV void each_cell3(const Dep3Args &a, const Foot3 &fp, F visit) {
    for (int gx = fp.g0[0]; gx <= fp.g1[0]; gx++)
        for (int gy = fp.g0[1]; gy <= fp.g1[1]; gy++)
            for (int gz = fp.g0[2]; gz <= fp.g1[2]; gz++) visit(gx, gy, gz, weight3(a, fp, gx, gy, gz));
}

MHIP_DEV int64_t cell3(const Dep3Args &a, int gx, int gy, int gz) {
    if (a.periodic) {
        gx = ((gx % a.res) + a.res) % a.res;
        gy = ((gy % a.res) + a.res) % a.res;
        gz = ((gz % a.res) + a.res) % a.res;
    }
    return ((int64_t)gx * a.res + gy) * a.res + gz;
}

MHIP_DEV double foot3_total(const Dep3Args &a, const Foot3 &fp) {
    double tot = 0.0;
    each_cell3(a, fp, [&](int, int, int, double k) { tot += k; });
    return tot;
}

// first footprint index on axis c, wrapped into the grid when periodic
MHIP_DEV int wrapped_first(const Dep3Args &a, const Foot3 &fp, int c) {
    return a.periodic ? ((fp.g0[c] % a.res) + a.res) % a.res : fp.g0[c];
}

// binned volumes: the brick of the (wrapped) first footprint cell; the
// window holds 16^3 cells from the brick's origin, a keyed footprint spans at
// most 9 cells per axis from inside the brick.  Periodic footprints keep
// their unwrapped extent in the window and wrap when it is added to the map.
struct Vol3 {
    using Args = Dep3Args;
    static MHIP_DEV uint32_t skip(const Dep3Args &a) { return (uint32_t)a.nb * (uint32_t)a.nb * (uint32_t)a.nb; }
    static MHIP_DEV uint32_t key(const Dep3Args &a, int64_t i, uint32_t &ncell) {
        Foot3 fp;
        ncell = 0;
        if (!footprint3(a, i, fp)) return 2 * skip(a);
        const uint32_t nb = (uint32_t)a.nb;
        const uint32_t brick =
            ((uint32_t)(wrapped_first(a, fp, 0) / BRICK3) * nb + (uint32_t)(wrapped_first(a, fp, 1) / BRICK3)) * nb +
            (uint32_t)(wrapped_first(a, fp, 2) / BRICK3);
        int64_t cells = 1;
        bool fits = true;
        for (int c = 0; c < 3; c++) {
            const int64_t sp = (int64_t)fp.g1[c] - fp.g0[c] + 1;
            fits = fits && sp <= WIN3 - BRICK3 + 1;
            cells *= fits ? sp : 1;
        }
        if (!fits || cells > BIG_CELLS_3D) {
            ncell = SIZE_MAX_RANK;
            return skip(a) + brick;
        }
        ncell = (uint32_t)cells;
        return brick;
    }
    static MHIP_DEV void direct(const Dep3Args &a, uint32_t i) {
        Foot3 fp;
        footprint3(a, i, fp);  // keyed, so it has a footprint
        const double tot = foot3_total(a, fp);
        if (!(tot > 0.0)) return;
        const double inv = 1.0 / tot;
        each_cell3(a, fp, [&](int gx, int gy, int gz, double k) {
            if (k != 0.0) atomicAdd(&a.grid[cell3(a, gx, gy, gz)], k * inv * fp.f);
        });
    }
    using F = Foot3;
    static MHIP_DEV bool foot(const Dep3Args &a, uint32_t i, F &fp) { return footprint3(a, i, fp); }
    static MHIP_DEV int cells(const F &fp) {
        return (fp.g1[0] - fp.g0[0] + 1) * (fp.g1[1] - fp.g0[1] + 1) * (fp.g1[2] - fp.g0[2] + 1);
    }
    // a cell's place in a window or tile, up to that of its origin (modulo
    // 2^32: unwrapped indices of a periodic box can be large)
    static MHIP_DEV uint32_t slot(int x, int y, int z) {
        return ((uint32_t)x * WIN3 + (uint32_t)y) * WIN3 + (uint32_t)z;
    }
    // window index of the footprint's first cell on each axis (0..7)
    static MHIP_DEV void place(const Dep3Args &a, const F &fp, uint32_t key, int *s) {
        const uint32_t nb = (uint32_t)a.nb;
        const int b[3] = {(int)(key / (nb * nb)), (int)(key / nb % nb), (int)(key % nb)};
        for (int c = 0; c < 3; c++) s[c] = wrapped_first(a, fp, c) - b[c] * BRICK3;
    }
    static MHIP_DEV void window_wave(const Dep3Args &a, const F &mine, int l, uint32_t key, double *win) {
        const F fp = lane_foot(mine, l);
        int s[3];
        place(a, fp, key, s);
        const uint32_t origin = slot(fp.g0[0] - s[0], fp.g0[1] - s[1], fp.g0[2] - s[2]);
        Walk3 w;
        w.start(threadIdx.x % WAVE, WAVE, fp.g0, fp.g1);
        wave_spread(
            w, cells(fp), true, [&](const Walk3 &c) { return weight3(a, fp, c.x, c.y, c.z); },
            [&](const Walk3 &c, double k) { atomicAdd(&win[slot(c.x, c.y, c.z) - origin], k * fp.f); });
    }
    static MHIP_DEV void window(const Dep3Args &a, const F &fp, uint32_t key, double *win) {
        int s[3];
        place(a, fp, key, s);
        const int wx = fp.g1[0] - fp.g0[0] + 1, wy = fp.g1[1] - fp.g0[1] + 1, wz = fp.g1[2] - fp.g0[2] + 1;
        const int ncell = wx * wy * wz;
        // a starting cell for each lane, as in Map2::window
        const uint32_t lane = threadIdx.x % WAVE, row = lane / (uint32_t)wz;
        const int g[3] = {fp.g0[0] + (int)(row / (uint32_t)wy % (uint32_t)wx), fp.g0[1] + (int)(row % (uint32_t)wy),
                          fp.g0[2] + (int)(lane % (uint32_t)wz)};
        int gx = g[0], gy = g[1], gz = g[2];
        auto next = [&]() {
            if (++gz > fp.g1[2]) {
                gz = fp.g0[2];
                if (++gy > fp.g1[1]) {
                    gy = fp.g0[1];
                    if (++gx > fp.g1[0]) gx = fp.g0[0];
                }
            }
        };
        auto at = [&]() {
            return (gx - fp.g0[0] + s[0]) * (WIN3 * WIN3) + (gy - fp.g0[1] + s[1]) * WIN3 + (gz - fp.g0[2] + s[2]);
        };
        if (ncell <= WCACHE3) {
            // small footprints: the weights stay in registers between the
            // total and the deposit
            double wc[WCACHE3];
            double tot = 0.0;
#pragma unroll
            for (int c = 0; c < WCACHE3; c++) {
                wc[c] = 0.0;
                if (c < ncell) {
                    wc[c] = weight3(a, fp, gx, gy, gz);
                    tot += wc[c];
                    next();
                }
            }
            if (!(tot > 0.0)) return;
            const double inv = 1.0 / tot;
            gx = g[0];
            gy = g[1];
            gz = g[2];
#pragma unroll
            for (int c = 0; c < WCACHE3; c++) {
                if (c < ncell) {
                    if (wc[c] != 0.0) atomicAdd(&win[at()], wc[c] * inv * fp.f);
                    next();
                }
            }
            return;
        }
        const double tot = foot3_total(a, fp);
        if (!(tot > 0.0)) return;
        const double inv = 1.0 / tot;
        for (int c = 0; c < ncell; c++) {
            const double k = weight3(a, fp, gx, gy, gz);
            if (k != 0.0) atomicAdd(&win[at()], k * inv * fp.f);
            next();
        }
    }
    static MHIP_DEV void flush(const Dep3Args &a, uint32_t key, int c, double v) {
        const uint32_t nb = (uint32_t)a.nb;
        const int gx = (int)(key / (nb * nb)) * BRICK3 + c / (WIN3 * WIN3);
        const int gy = (int)(key / nb % nb) * BRICK3 + c / WIN3 % WIN3;
        const int gz = (int)(key % nb) * BRICK3 + c % WIN3;
        if (!a.periodic && (gx >= a.res || gy >= a.res || gz >= a.res)) return;
        atomicAdd(&a.grid[cell3(a, gx, gy, gz)], v);
    }

    // ---- tiles of WIN3^3 cells; a periodic footprint meets a tile once for
    // each m with cells of it shifted by m res inside
    static constexpr int SIDE = WIN3;
    // (ms by cells a tile, direct / tiles: 1024^3 450 7.7 / 14.0, 3600 21.5 / 30.0,
    // 14500 67.5 / 64.2; 512^3 3600 2.7 / 3.1, 29000 16.4 / 12.4)
    static constexpr int TILE_CELLS = 8000;
    static MHIP_DEV void spread(const Dep3Args &a, const F &fp, double inv, int thread, int stride) {
        const double f = fp.f * inv;
        Walk3 w;
        for (w.start(thread, stride, fp.g0, fp.g1); w.inside(); w.next()) {
            const double k = weight3(a, fp, w.x, w.y, w.z);
            if (k != 0.0) atomicAdd(&a.grid[cell3(a, w.x, w.y, w.z)], k * f);
        }
    }
    static MHIP_DEV int floor_div(int x, int d) { return x >= 0 ? x / d : -1 - (-1 - x) / d; }
    static MHIP_DEV void box(const F &fp, int *lo, int *hi) {
        for (int c = 0; c < 3; c++) {
            lo[c] = fp.g0[c];
            hi[c] = fp.g1[c];
        }
    }
    static MHIP_DEV void corner(int64_t tile, int nt, int *t0) {
        t0[0] = (int)(tile / ((int64_t)nt * nt)) * SIDE;
        t0[1] = (int)(tile / nt % nt) * SIDE;
        t0[2] = (int)(tile % nt) * SIDE;
    }
    // first and last shift m of the cells lo..hi that meets the tile's cells on
    // one axis (the tile's cells past the grid are none: the grid's own images
    // are there)
    static MHIP_DEV void shifts(const Dep3Args &a, int lo, int hi, int t0, int &m0, int &m1) {
        const int t1 = min(t0 + SIDE, a.res) - 1;
        m0 = a.periodic ? -floor_div(t1 - lo, a.res) : (lo <= t1 ? 0 : 1);
        m1 = a.periodic ? floor_div(hi - t0, a.res) : (hi >= t0 ? 0 : -1);
    }
    static MHIP_DEV bool meets(const Dep3Args &a, const int *lo, const int *hi, const int *t0) {
        bool all = true;
        for (int c = 0; c < 3; c++) {
            int m0, m1;
            shifts(a, lo[c], hi[c], t0[c], m0, m1);
            all = all && m0 <= m1;
        }
        return all;
    }
    static MHIP_DEV double total(const Dep3Args &a, const F &fp, int thread, int stride) {
        Walk3 w;
        double tot = 0.0;
        for (w.start(thread, stride, fp.g0, fp.g1); w.inside(); w.next()) tot += weight3(a, fp, w.x, w.y, w.z);
        return tot;
    }
    static MHIP_DEV void tile_wave(const Dep3Args &a, const F &mine, double inv, int l, const int *t0, double *win) {
        const F fp = lane_foot(mine, l);
        const double f = fp.f * lane_value(inv, l);
        int m0[3], m1[3];
        for (int c = 0; c < 3; c++) shifts(a, fp.g0[c], fp.g1[c], t0[c], m0[c], m1[c]);
        for (int mx = m0[0]; mx <= m1[0]; mx++)
            for (int my = m0[1]; my <= m1[1]; my++)
                for (int mz = m0[2]; mz <= m1[2]; mz++) {
                    // the tile's cells in the footprint's own indices
                    const int o[3] = {t0[0] + mx * a.res, t0[1] + my * a.res, t0[2] + mz * a.res};
                    int lo[3], hi[3];
                    for (int c = 0; c < 3; c++) {
                        lo[c] = max(fp.g0[c], o[c]);
                        hi[c] = min(fp.g1[c], o[c] + min(SIDE, a.res - t0[c]) - 1);
                    }
                    const uint32_t origin = slot(o[0], o[1], o[2]);
                    Walk3 w;
                    for (w.start(threadIdx.x % WAVE, WAVE, lo, hi); w.inside(); w.next()) {
                        const double k = weight3(a, fp, w.x, w.y, w.z);
                        if (k != 0.0) atomicAdd(&win[slot(w.x, w.y, w.z) - origin], k * f);
                    }
                }
    }
    static MHIP_DEV void tile_flush(const Dep3Args &a, const int *t0, int c, double v) {
        const int gx = t0[0] + c / (SIDE * SIDE), gy = t0[1] + c / SIDE % SIDE, gz = t0[2] + c % SIDE;
        atomicAdd(&a.grid[((int64_t)gx * a.res + gy) * a.res + gz], v);
    }
};

int grid_density(mhip_ctx *ctx, const void *f, int f_f64, const void *pos, int pos_f64, int64_t n, const void *h,
                 int h_f64, double hmin, double cx, double cy, double cz, double size, int res, int periodic,
                 double *grid) {
    if (n < 0) return fail(ctx, -1, "negative particle count");
    if (res < 2 || res > 2048) return fail(ctx, -1, "res must be in [2, 2048]");
    if (!(size > 0.0)) return fail(ctx, -1, "size must be positive");
    if (n > 0xffffffffll) return fail(ctx, -4, "more than 2^32 particles");
    Dep3Args a;
    a.f = f;
    a.pos = pos;
    a.h = h;
    a.f_f64 = f_f64;
    a.pos_f64 = pos_f64;
    a.h_f64 = h_f64;
    a.n = n;
    a.hmin = hmin;
    a.dx = size / (res - 1);
    // x - center + size/2 - dx/2: point g at center - size/2 + dx/2 + g dx
    a.ox = cx - 0.5 * size + 0.5 * a.dx;
    a.oy = cy - 0.5 * size + 0.5 * a.dx;
    a.oz = cz - 0.5 * size + 0.5 * a.dx;
    a.res = res;
    a.periodic = periodic ? 1 : 0;
    a.grid = grid;
    a.nb = (res + BRICK3 - 1) / BRICK3;
    int rc = 0;
    char *sc = (char *)scratch(ctx, bin_scratch_bytes(n), &rc);
    if (!sc) return rc;
    hipStream_t s = ctx->stream;
    const int64_t ncell = (int64_t)res * res * res, nt = (res + WIN3 - 1) / WIN3;
    ProfRegion pr(ctx, "grid_density");
    hipLaunchKernelGGL(k_grid_fill, dim3((unsigned)std::min<int64_t>(4096, (ncell + 255) / 256)), dim3(256), 0, s,
                       grid, ncell, 0.0);
    if ((rc = bin_deposit<Vol3>(ctx, a, (uint32_t)(a.nb * a.nb * a.nb), nt * nt * nt, true, sc))) return rc;
    const double inv = 1.0 / (a.dx * a.dx * a.dx);
    hipLaunchKernelGGL(k_grid_scale, dim3((unsigned)std::min<int64_t>(4096, (ncell + 255) / 256)), dim3(256), 0, s,
                       grid, ncell, inv);
    return check_hip(ctx, hipGetLastError(), "grid density launch");
}

int surface_density(mhip_ctx *ctx, const void *f, int f_f64, const void *pos, int pos_f64, int64_t n, int dim,
                    const void *h, int h_f64, double smooth, double hmin, double cx, double cy, double size, int res,
                    int conservative, double *grid) {
    if (n < 0 || dim < 2 || dim > 3) return fail(ctx, -1, "surface density needs (n, 2) or (n, 3) positions");
    if (res < 2 || res > (1 << 20)) return fail(ctx, -1, "res must be in [2, 2^20]");
    if (!(size > 0.0)) return fail(ctx, -1, "size must be positive");
    if (n > 0xffffffffll) return fail(ctx, -4, "more than 2^32 particles");
    DepArgs a;
    a.f = f;
    a.pos = pos;
    a.h = h;
    a.f_f64 = f_f64;
    a.pos_f64 = pos_f64;
    a.h_f64 = h_f64;
    a.dim = dim;
    a.n = n;
    a.smooth = smooth;
    a.hmin = hmin;  // SurfaceDensity: np.clip(smooth_fac * h, 2 * size / res, 1e100)
    a.ox = cx - 0.5 * size;
    a.oy = cy - 0.5 * size;
    a.dx = size / (res - 1);
    a.res = res;
    a.conservative = conservative ? 1 : 0;
    a.grid = grid;
    a.nb = (res + BRICK2 - 1) / BRICK2;
    int rc = 0;
    char *sc = (char *)scratch(ctx, bin_scratch_bytes(n), &rc);
    if (!sc) return rc;
    // whole-map path: totals, range, list, boxes
    uint32_t *range = (uint32_t *)(sc + (size_t)n * 8);
    a.nbig = range + 1;
    a.big = range + 2;
    hipStream_t s = ctx->stream;
    const int64_t ncell = (int64_t)res * res, nt = (res + WIN2 - 1) / WIN2;
    ProfRegion pr(ctx, "surface_density");
    hipLaunchKernelGGL(k_grid_fill, dim3((unsigned)std::min<int64_t>(1024, (ncell + 255) / 256)), dim3(256), 0, s,
                       grid, ncell, 0.0);
    if (n > 0) {
        int ncu = 0;
        if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess || ncu < 1)
            ncu = 256;
        if (res <= DEP_TILE) {
            // the whole map in LDS: one block per CU, particles interleaved
            // over the blocks, each block adds its map to HBM once
            const size_t lds = (size_t)res * res * sizeof(double);
            if (lds > 65536 && hipFuncSetAttribute((const void *)k_deposit_tiles,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
                return check_hip(ctx, hipGetLastError(), "deposit LDS size");
            const int64_t nchunk = std::max<int64_t>(1, std::min<int64_t>(ncu, (n + 255) / 256));
            hipLaunchKernelGGL(k_range_zero, dim3(1), dim3(WAVE), 0, s, range);
            hipLaunchKernelGGL(k_deposit_tiles, dim3((unsigned)nchunk), dim3(DEP_THREADS), lds, s, a, res, 1,
                               (int)nchunk);
            const Wide wd{a.big, range, (int *)(a.big + n), nullptr, conservative ? (double *)sc : nullptr, nullptr};
            wide_deposit<Map2>(ctx, a, wd, nt * nt);
        } else {
            // binned by 32^2 bricks (per-tile LDS copies of the map would
            // re-read every particle per tile)
            if ((rc = bin_deposit<Map2>(ctx, a, (uint32_t)a.nb * (uint32_t)a.nb, nt * nt, conservative != 0, sc))) return rc;
        }
    }
    if (conservative) {
        const double dx2inv = 1.0 / (a.dx * a.dx);
        hipLaunchKernelGGL(k_grid_scale, dim3((unsigned)std::min<int64_t>(1024, (ncell + 255) / 256)), dim3(256), 0,
                           s, grid, ncell, dx2inv);
    }
    return check_hip(ctx, hipGetLastError(), "surface density launch");
}

}  // namespace mhip
