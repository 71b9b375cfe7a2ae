// Which kernel serves a search, and which of its launches finishes a row and puts
// it on the list of ambiguous rows.  Up to three launches see a row: the
// one-lane-per-query kernel, that kernel again over the wavefronts where a radius
// seed was too small (redo), and the one-wavefront-per-query kernel over the
// wavefronts that either of them deferred.  The list has one place per row, so each row is
// appended by exactly one of them, the one that finishes it.
// Header-only and usable from host code (a CPU unit test compiles it with g++).
#pragma once
#include <stdint.h>

#if !defined(MHIP_HD)
#if defined(__HIPCC__)
#define MHIP_HD __host__ __device__ __forceinline__
#else
#define MHIP_HD inline
#endif
#endif

namespace mhip {

// in a row's status between the launches: a deferring wavefront left the row
// to the one-wavefront-per-query kernel (no bit of the public status).  Rows
// that an earlier launch finished keep their status.
constexpr int32_t ROW_DEFERRED = 1 << 30;

// whether the one-lane kernel is to finish this row, in the first launch or in
// the redo launch (missed: the row's radius seed was too small in the first): a
// wavefront lists such rows if it finishes them, and marks them if it defers
MHIP_HD bool row_is_new(bool redo, bool missed) { return !redo || missed; }

// whether the one-wavefront kernel is to finish this row of a deferred wavefront
MHIP_HD bool row_was_deferred(int32_t st) { return (st & ROW_DEFERRED) != 0; }

// Whether the one-wavefront-per-query kernel takes the whole set.  Where the lines
// lie (ms of the whole search, one lane / one wavefront per query): k = 32
// open 3D float32, 65536 particles 0.200 / 0.135, 10^5 0.212 / 0.212, 3 10^5
// 0.369 / 0.560; 2D 32768 0.078 / 0.069, 65536 0.076 / 0.104; k = 64 3D 3 10^5
// 0.69 / 0.68, 10^6 1.85 / 2.31; periodic float64 k = 32 3 10^5 0.77 / 0.68,
// 10^6 1.90 / 2.28 (wavefronts near the faces come here anyway); k = 100 10^6
// 3.31 / 2.84, clustered 2^22 16.0 / 13.7.  Few queries in a large set lie far
// apart and share no leaves (2^22 clustered, k = 32, 10% at random 2.76 / 1.34;
// 10% that lie together 0.70 / 1.13).
constexpr int64_t KNN_PART = 1 << 20;
MHIP_HD bool knn_wave_serves(int64_t n, int64_t nq, int k, int dim, bool per) {
    // 16 threads a query, below 2^32 in a launch; 32-bit byte offsets
    if (n >= (int64_t)1 << 28 || nq >= (int64_t)1 << 28) return false;
    if (k > 64 || (nq < n / 4 && nq <= KNN_PART)) return true;
    int64_t most = dim == 3 ? 100000 : 45000;
    if (k > 32) most *= 3;
    if (per) most *= 3;
    return n <= most;
}

// A larger part of a large set is shared out by wavefronts (64 queries in sorted
// order): those whose queries span more than KNN_SPREAD particles go to the
// one-wavefront-per-query kernel, those that lie side by side share their leaves
// and go to the one-lane kernel.  (2^24 clustered, k = 32, one lane / one
// wavefront per query / shared out: 20% that lie together 3.5 / 8.5 / 3.7 ms, at
// random 15% 9.8 / 7.2 / 7.2, 20% 7.1 / 9.5 / 9.5; k = 64, 2^22, 24% at random
// 5.3 / 3.5 / 3.5.  With a span of 320, 20% at random fell to both kernels: 9.7.)
constexpr uint32_t KNN_SPREAD = 160;
MHIP_HD bool knn_splits(int64_t n, int64_t nq, int k, int dim, bool per) {
    return n < (int64_t)1 << 28 && !knn_wave_serves(n, nq, k, dim, per) && nq < n / (k > 32 ? 4 : 5);
}

}  // namespace mhip
