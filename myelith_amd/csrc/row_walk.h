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
