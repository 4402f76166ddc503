// row_walk.h -- index walks over rows of up to 2^31 - 1 values.  An index is
// an int, and a step from the last values of the longest rows would pass its
// range, so the steps are counted from a segment's start or in 64 bits.  Plain
// C++ (constexpr: host and device): a host build runs under
// UndefinedBehaviorSanitizer in the CPU tests.
#pragma once

#include <cstdint>

namespace myl {

// The passes over whole logit rows (argmax, log-softmax, sampling) run one
// block of 16 waves per row and walk it in segments of kRowSeg values per wave.
constexpr int kRowThreads = 1024;
constexpr int kRowWaves = kRowThreads / 64;
constexpr int kRowSeg = 1024;

// Short rows (argmax, log-softmax) take blocks of kRowShortThreads threads
// instead, which step over them by four values a thread: with more rows than
// CUs, blocks of 16 waves wait for each other (and the log-softmax's counters cost
// more than a second read of the row); with fewer, the 16 waves' loads in
// flight win earlier.  us on MI355X, short / long block, rows x values:
//   argmax       1 x 1000 2.2 / 2.2    1 x 2048 2.3 / 2.2    2000 x 1000 3.3 / 7.7   2000 x 8192 11.2 / 13.9
//   log-softmax  1 x 4096 5.5 / 5.6    1 x 6000 6.4 / 5.8    600 x 8192 8.9 / 12.9   2000 x 1000 7.2 / 25.1
constexpr int kRowFew = 256;  // one row per CU
constexpr int kRowShort = 8192, kRowShortArgmax = 1024, kRowShortLogsoftmax = 4096;
constexpr bool row_short_argmax(int M, int n) { return n <= (M > kRowFew ? kRowShort : kRowShortArgmax); }
constexpr bool row_short_logsoftmax(int M, int n) { return n <= (M > kRowFew ? kRowShort : kRowShortLogsoftmax); }
constexpr int kRowShortThreads = 256;

// quad(i) for each whole four values of a short row that fall to thread tid (i
// their first index), then one(i) for at most one of the last n % 4.
template <class Quad, class One>
constexpr void row_quads(int n, int tid, const Quad& quad, const One& one) {
#pragma unroll 4
    for (int i = 4 * tid; i < (n & ~3); i += 4 * kRowShortThreads) quad(i);
    if (tid < (n & 3)) one((n & ~3) + tid);
}

// f(i) for thread tid's values of the partial last segment [i0, n), spread over
// all of the block's threads: at most one each for a block of kRowThreads, so
// the segment costs one memory latency (one wave alone takes up to 16, which is
// all the time of a row of less than one segment).
template <class F>
constexpr void row_tail(int i0, int n, int tid, int threads, const F& f) {
    for (int k = tid; k < n - i0; k += threads) f(i0 + k);
}

// f(i) for every kRowThreads-th value from tid on.
template <class F>
constexpr void row_strided(int n, int tid, const F& f) {
    for (int64_t i = tid; i < n; i += kRowThreads) f((int)i);
}

// Lane `lane`'s four values of step k0 (a multiple of 256 below the group's
// length) of a group that starts at g0, both multiples of 256: the first index.
constexpr int row_group_index(int g0, int k0, int lane) { return g0 + k0 + 4 * lane; }

}  // namespace myl
