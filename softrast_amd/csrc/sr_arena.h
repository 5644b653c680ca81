// sr_arena.h -- sizes of a frame's entry and pair arenas, host arithmetic.
//
// The count walks record every (record, bin) pair in three arrays -- record,
// part-bin key, slot in the part's list -- each cut into regions with a
// counter of their own (FrameDev). An index into one of the arrays, and a sum
// of bin entries, is a 32-bit word on the device, so an array holds fewer than
// 2^32 pairs; a bin entry is a recorded pair, so a frame whose regions hold all
// of its pairs has fewer than 2^32 entries as well. The arrays together may be
// larger: each is addressed from a base pointer of its own.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace srg {

constexpr uint32_t kPairRegions = 256, kClipPairRegions = 8;
constexpr uint64_t kMaxPairs = 0xFFFFFFF0ull;        // of one array
constexpr uint64_t kMaxEntries = kMaxPairs / 3 * 2;  // the entry arena that has them

// Pairs of an array beside `entries` bin entries: as many for k_setup's
// regions, half as many for k_clip's.
constexpr uint64_t pair_words(uint64_t entries) { return entries + entries / 2; }

struct PairLayout {
    uint32_t regions;     // k_setup's: a power of two, so that it finds its region with a mask
    uint32_t region_cap;  // pairs of one of them
    uint32_t clip_cap;    // pairs of one of k_clip's kClipPairRegions regions, which follow
    uint32_t total;       // words of an array
};

// entries: at most kMaxEntries. workgroups: k_setup's.
constexpr PairLayout pair_layout(uint64_t entries, uint32_t workgroups)
{
    PairLayout P{ 1, 0, 0, 0 };
    while (P.regions < kPairRegions && P.regions * 2 <= workgroups) P.regions *= 2;
    P.region_cap = (uint32_t)(entries / P.regions);
    P.clip_cap = (uint32_t)(entries / 2 / kClipPairRegions);
    P.total = P.regions * P.region_cap + kClipPairRegions * P.clip_cap;
    return P;
}

// Array k (0 record, 1 key, 2 slot) of an arena of 3 * pair_words(entries) words.
inline uint32_t* pair_array(uint32_t* arena, const PairLayout& P, uint32_t k) { return arena + (size_t)P.total * k; }

// Entry arena for a frame that overflowed one of `entries` and asked for
// `need`; 0 if no arena is large enough.
constexpr uint64_t grown_entries(uint64_t entries, uint64_t need)
{
    if (entries >= kMaxEntries || need > kMaxEntries) return 0;
    const uint64_t n = entries * 2 > need ? entries * 2 : need;
    return n < kMaxEntries ? n : kMaxEntries;
}

}  // namespace srg
