// Sizes and bookkeeping of the host side that need no HIP, so that a plain C++
// compiler builds them and tests reach them without a device.
#pragma once
#include <algorithm>
#include <cstdint>

namespace fbh {

// Blocks of quantile_partials_kernel, each leaving a pair of doubles; the scale's
// value depends on their number, so it is the same at any row count.
constexpr uint32_t QUANTILE_BLOCKS = 256;

// Blocks of the bounds and quantisation passes, whose results reduce_max_kernel and
// grow_prep_kernel go through on one workgroup: a row a thread, and rows in turn
// from 8192 blocks on. With 8192 at any size the four kernels took 40 us a tree of
// 5000 rows, now 16.
inline uint32_t reduction_blocks(uint64_t n_rows) {
    return (uint32_t)std::min<uint64_t>((n_rows + 255) / 256, 8192);
}

// Words (doubles or int64s) of each reduction scratch: a pair a block of the bounds
// and quantisation passes and the pair they reduce to, or, where that is more (up to
// 65,024 rows), the quantile scale's pairs.
inline uint64_t reduction_words(uint32_t n_red_blocks) {
    return std::max<uint64_t>(2ull * n_red_blocks + 2, 2ull * QUANTILE_BLOCKS);
}

// Replaces a kept buffer of `bytes` by one of at least `want` where it is smaller. The
// old one is forgotten before the new one is asked for: when `take` throws, nothing
// points to memory that has been given back, and a later call asks again.
template <class T, class Release, class Take>
void regrow(T *&p, uint64_t &bytes, uint64_t want, Release &&release, Take &&take) {
    if (bytes >= want) return;
    T *old = p;
    p = nullptr;
    bytes = 0;
    release(old);
    p = take(want);
    bytes = want;
}

}  // namespace fbh
