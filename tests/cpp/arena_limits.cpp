// Sizes of the entry and pair arenas at their limits (csrc/sr_arena.h): every
// pair of every region has a place of its own inside the arena, a 32-bit index
// reaches all of them, and an arena that grows ends at the limit.
#include <cstdio>

#include "sr_arena.h"

using namespace srg;

static int bad = 0;
#define CHECK(c, ...) ((c) ? (void)0 : (void)(++bad, std::printf("%d: %s: ", __LINE__, #c), std::printf(__VA_ARGS__), std::printf("\n")))

int main()
{
    const uint64_t G = 1ull << 32;
    CHECK(pair_words(kMaxEntries) <= kMaxPairs && pair_words(kMaxEntries + 2) > kMaxPairs, "limit");
    // sizes whose second or third array starts or ends on either side of 2^32 words, and the ends of the range
    const uint64_t entries[] = { 1, 2, 15, 16, 17, 4096, 954437176, 954437177, 1431655765, 1431655766, G / 2 + 1,
                                 kMaxEntries - 1, kMaxEntries };
    const uint32_t workgroups[] = { 0, 1, 2, 3, 255, 256, 257, 0xFFFFFFFFu };
    for (uint64_t e : entries)
        for (uint32_t w : workgroups) {
            const PairLayout P = pair_layout(e, w);
            const uint64_t clip_first = (uint64_t)P.regions * P.region_cap;
            const uint64_t end = clip_first + (uint64_t)kClipPairRegions * P.clip_cap;
            CHECK((P.regions & (P.regions - 1)) == 0 && P.regions <= kPairRegions && P.regions <= (w ? w : 1), "%llu %u",
                  (unsigned long long)e, w);
            CHECK(P.regions * 2 > w || P.regions == kPairRegions, "%llu %u", (unsigned long long)e, w);
            CHECK(end < G && end == P.total && end <= pair_words(e), "%llu %u: %llu", (unsigned long long)e, w,
                  (unsigned long long)end);
            // a wave's reservation that passes a region's end does not wrap: at most 64 triangles x 2^22 bins
            CHECK(P.region_cap + (64ull << 22) < G && P.clip_cap + (64ull << 22) < G, "%llu %u", (unsigned long long)e, w);
            uint32_t* const arena = reinterpret_cast<uint32_t*>(uintptr_t(1) << 40);  // an address only
            for (uint32_t k = 0; k < 3; ++k) {
                const uint64_t first = (uint64_t)(pair_array(arena, P, k) - arena);
                CHECK(first == (uint64_t)P.total * k && first + P.total <= 3 * pair_words(e), "%llu %u array %u",
                      (unsigned long long)e, w, k);
            }
        }
    CHECK(grown_entries(1, 0) == 2 && grown_entries(1000, 5000) == 5000 && grown_entries(1000, 1500) == 2000, "growth");
    CHECK(grown_entries(kMaxEntries / 2 + 1, 7) == kMaxEntries && grown_entries(7, kMaxEntries) == kMaxEntries, "to the limit");
    CHECK(grown_entries(kMaxEntries, 7) == 0 && grown_entries(7, kMaxEntries + 1) == 0, "past the limit");
    std::printf("failed: %d\n", bad);
    return bad ? 1 : 0;
}
