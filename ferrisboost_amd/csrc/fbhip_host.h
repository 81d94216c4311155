// Sizes and bookkeeping of the host side that need no HIP, so that a plain C++
// compiler builds them and tests reach them without a device.
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

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

// ---- The device sketch's summary buffers (fbhip_sketch.hip), in slots of one batch's
// entries. Features are summarised in groups that share the buffers, of
// SKETCH_GROUP_BYTES of batch summaries but no fewer than SKETCH_GROUP_FEATS features:
// a merge of each still gives every CU a workgroup at the counter's last levels. 400k x
// 2000 at 256 bins takes 33 GB in one group, more than is kept for the next job
// (fbhip_keep.hip), and 11 in groups: the whole job, 40 rounds, 239 -> 226 ms, and 221
// with a group's task tables built while the groups before it run.
constexpr uint32_t SKETCH_GROUP_FEATS = 256;
constexpr uint64_t SKETCH_GROUP_BYTES = 2ull << 30;
constexpr uint64_t SKETCH_ENTRY_BYTES = 16;

struct SketchSlots {
    // of the largest group: batch summaries, merged blocks (two slots each), final merges
    uint64_t a = 0, b = 0, t = 0;
    uint64_t all_a = 0, all_t = 0;  // of all features
};

struct SketchPlan {
    struct Group {
        uint32_t j0, j1;
    };
    std::vector<uint64_t> abase, bbase, tbase;  // a feature's first slots, and the ends
    std::vector<Group> groups;
    SketchSlots slots;
};

// For features of m[j] batches of `limit` entries.
inline SketchPlan sketch_plan(const std::vector<uint64_t> &m, uint64_t limit) {
    const uint32_t n = (uint32_t)m.size();
    SketchPlan p;
    p.abase.assign(n + 1, 0);
    p.bbase.assign(n + 1, 0);
    p.tbase.assign(n + 1, 0);
    for (uint32_t j = 0; j < n; j++) {
        p.abase[j + 1] = p.abase[j] + m[j];
        p.bbase[j + 1] = p.bbase[j] + (m[j] + 1) / 2;
        p.tbase[j + 1] = p.tbase[j] + 2ull * __builtin_popcountll(m[j]);
    }
    for (uint32_t j0 = 0, j1; j0 < n; j0 = j1) {
        j1 = j0 + 1;
        while (j1 < n && (j1 - j0 < SKETCH_GROUP_FEATS ||
                          (p.abase[j1 + 1] - p.abase[j0]) * limit * SKETCH_ENTRY_BYTES <=
                              SKETCH_GROUP_BYTES))
            j1++;
        if (n - j1 < SKETCH_GROUP_FEATS / 2) j1 = n;  // no short last group
        p.groups.push_back({j0, j1});
        p.slots.a = std::max(p.slots.a, p.abase[j1] - p.abase[j0]);
        p.slots.b = std::max(p.slots.b, p.bbase[j1] - p.bbase[j0]);
        p.slots.t = std::max(p.slots.t, p.tbase[j1] - p.tbase[j0]);
    }
    p.slots.all_a = p.abase[n];
    p.slots.all_t = p.tbase[n];
    return p;
}

// The most that any n features of at most `m` batches each take.
inline SketchSlots sketch_slots_most(uint64_t m, uint32_t n, uint64_t limit) {
    uint64_t bits = 0;
    while (m >> bits) bits++;
    SketchSlots s;
    s.all_a = m * n;
    s.all_t = 2 * bits * n;
    // a group is full at SKETCH_GROUP_FEATS features or SKETCH_GROUP_BYTES, and the last
    // one takes a short rest in
    s.a = std::min(s.all_a, std::max(SKETCH_GROUP_FEATS * m,
                                     SKETCH_GROUP_BYTES / (limit * SKETCH_ENTRY_BYTES)) +
                                SKETCH_GROUP_FEATS / 2 * m);
    // (k + 1) / 2 and 2 popcount(k) slots for a feature's k > 0 batches
    s.b = std::min((s.a + std::min<uint64_t>(n, s.a)) / 2, (m + 1) / 2 * n);
    s.t = std::min(2 * s.a, s.all_t);
    return s;
}

}  // namespace fbh
