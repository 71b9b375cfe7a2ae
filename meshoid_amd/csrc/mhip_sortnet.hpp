// In-register sorting networks for the kNN's lists: Batcher's odd-even merge
// sort and the merge of a sorted run into a sorted list that keeps its length.  Index arithmetic is compile-time, so the arrays stay in registers.
// Header-only and usable from host code (a CPU unit test compiles it with g++).
// Values must not be NaN (callers map NaN to +inf first).
#pragma once

#if defined(__HIPCC__)
#define MHIP_HD __host__ __device__ __forceinline__
#else
#define MHIP_HD inline
#endif

namespace mhip {

// On the device the minimum and maximum are written out: from the comparison
// the compiler makes a compare and two selects, three instructions for two.
MHIP_HD void cmpx(float &a, float &b) {
#if defined(__HIP_DEVICE_COMPILE__)
    float lo, hi;
    asm("v_min_f32 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f32 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
#else
    const float lo = a < b ? a : b;
    const float hi = a < b ? b : a;
    a = lo;
    b = hi;
#endif
}

// a = the smaller of a and b
MHIP_HD void keep_min(float &a, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_min_f32 %0, %0, %1" : "+v"(a) : "v"(b));
#else
    a = a < b ? a : b;
#endif
}

// Batcher's odd-even merge sort, ascending (K. E. Batcher, "Sorting networks
// and their applications", AFIPS 1968): for N = 32, 191 compare-exchanges.
template <int N>
MHIP_HD void oddeven_sort(float (&v)[N]) {
    static_assert((N & (N - 1)) == 0, "power of two");
#pragma unroll
    for (int p = 1; p < N; p <<= 1) {
#pragma unroll
        for (int k = p; k >= 1; k >>= 1) {
#pragma unroll
            for (int j = k % p; j + k < N; j += 2 * k) {
#pragma unroll
                for (int i = 0; i < k; i++) {
                    if (i + j + k < N && (i + j) / (2 * p) == (i + j + k) / (2 * p)) cmpx(v[i + j], v[i + j + k]);
                }
            }
        }
    }
}

// A[0..K-1] and S[0..NS-1] ascending, NS <= K: afterwards A holds the K
// smallest of A and S, ascending.  With both lists thought of as padded to P,
// the next power of two (A below with -inf, S above with +inf), the P smallest
// of the union are min(A[i], S[P-1-i]), a bitonic sequence that a bitonic
// merge sorts.  Only the top NS slots meet a real entry of S, and a
// compare-exchange whose lower end is padding changes nothing: both are left
// out (K = 33, NS = 16: 16 minima and 81 compare-exchanges).
template <int K, int NS>
MHIP_HD void merge_sorted(float (&A)[K], const float (&S)[NS]) {
    static_assert(NS <= K, "the list must hold the new values");
    constexpr int P = K <= 1 ? 1 : K <= 2 ? 2 : K <= 4 ? 4 : K <= 8 ? 8 : K <= 16 ? 16 : K <= 32 ? 32 : K <= 64 ? 64 : K <= 128 ? 128 : 256;
    static_assert(K <= P, "list too long");
    constexpr int V = P - K;
#pragma unroll
    for (int i = 0; i < NS; i++) keep_min(A[K - NS + i], S[NS - 1 - i]);
#pragma unroll
    for (int w = P / 2; w >= 1; w >>= 1) {
#pragma unroll
        for (int i = V; i < P; i++) {
            if ((i & w) == 0) cmpx(A[i - V], A[i + w - V]);
        }
    }
}

// the N + 1 smallest of A (N + 1 slots) and S
template <int N>
MHIP_HD void merge_into(float (&A)[N + 1], const float (&S)[N]) {
    merge_sorted<N + 1, N>(A, S);
}

}  // namespace mhip
