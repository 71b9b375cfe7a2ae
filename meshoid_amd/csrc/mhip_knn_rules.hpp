// Which of a search's launches finishes a row and puts it on the list of
// ambiguous rows.  Up to three launches see a row: the one-lane-per-query
// kernel, that kernel again over the wavefronts where a radius seed was too
// small (redo), and the one-wavefront-per-query kernel over the wavefronts that
// either of them deferred.  The list has one place per row, so each row is
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

}  // namespace mhip
