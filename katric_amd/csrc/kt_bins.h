// Which work-queue bucket of the intersection a tail goes to: plain arithmetic,
// shared by the binning kernels and the host test of its ranges.
#pragma once

#include <stdint.h>

namespace kt {

// Work-queue buckets: three classes of eight.  Class PACK holds the tails that
// a wave takes several at a time, SOLO the other wave tails, TEAM the
// workgroup tails; the eight are size steps (by degree) or the contiguous
// eighths of the walk entries, one per XCD, each in vertex order (by vertex).
// Then the tails beyond any LDS table (binary search, k_tc_huge) and those
// above the workgroup bin whose table still fits a workgroup's whole LDS
// (k_tc_big), and, in a list of their own, the parts of tails whose walk is
// too long for one team (split_rule): entries (part << 32 | tail), taken by
// workgroup teams and by waves before everything else.
constexpr int CLASS_STEPS = 8;
constexpr int CLASS_PACK = 0, CLASS_SOLO = CLASS_STEPS, CLASS_TEAM = 2 * CLASS_STEPS;
constexpr int BUCKET_HUGE = 24;
constexpr int BUCKET_BIG = 25;
constexpr int NLIST = 26;  // buckets whose tails share the u32 list
constexpr int BUCKET_TEAM_PARTS = 26;
constexpr int BUCKET_WAVE_PARTS = 27;
// Parts of the workgroup tails that k_tc_hub takes (every such tail, whole or
// split).
constexpr int BUCKET_HUB_PARTS = 28;
constexpr int NBUCKET = 29;
// Tails of class PACK: at most 64 ids in S(x) and 64 walk entries.
constexpr uint32_t PACK_MAX = 64;

constexpr uint32_t ceil_log2(uint64_t x) { return x <= 1 ? 0 : 64 - (uint32_t)__builtin_clzll(x - 1); }

struct BinRule {
    uint32_t wave_max_deg, group_max_deg, bsearch_min_deg;
    uint32_t wave_split, team_split, hub_split;  // walk entries per part
    bool min_side;
};

// bucket: one of the buckets from BUCKET_HUGE on, or a class, of which step is
// the size step; parts: entries in the part list.
struct TailBin {
    int bucket, step;
    uint32_t parts;
};

// A tail with s ids in S and r walk entries (neither empty); hub(): k_tc_hub
// may take it (asked for workgroup tails only).
template <class Hub>
constexpr TailBin tail_bin(uint64_t s, uint64_t r, const BinRule& k, Hub hub) {
    if (s > k.bsearch_min_deg) return {BUCKET_HUGE, 0, 1};
    if (s > k.group_max_deg) return {BUCKET_BIG, 0, 1};
    int b = (int)ceil_log2(s);  // size step, 0..11
    // a min-side walk covers the whole input row: a long row goes to a
    // bigger bucket (a workgroup team beyond 512 entries), whatever |S(x)|
    if (k.min_side) {
        const int row = (int)ceil_log2(r) - 2, top = (int)ceil_log2(k.group_max_deg);
        const int up = row < top ? row : top;
        b = b > up ? b : up;
    }
    const bool wave = b <= (int)ceil_log2(k.wave_max_deg);
    if (!wave && hub()) return {BUCKET_HUB_PARTS, 0, (uint32_t)((r + k.hub_split - 1) / k.hub_split)};
    const uint32_t split = wave ? k.wave_split : k.team_split;
    if (r > split) return {wave ? BUCKET_WAVE_PARTS : BUCKET_TEAM_PARTS, 0, (uint32_t)((r + split - 1) / split)};
    const int cls = !wave ? CLASS_TEAM : s <= PACK_MAX && r <= PACK_MAX ? CLASS_PACK : CLASS_SOLO;
    // steps of the class: sets of up to 1, 2, 4 .. 64 ids (PACK); 2 .. 256
    // (SOLO: a message with one known ghost, which has step 0 by its size, and
    // more entries than a pack holds goes with the twos); 16 .. 2048 (TEAM)
    const int lo = cls == CLASS_TEAM ? 4 : cls == CLASS_SOLO ? 1 : 0;
    const int step = b < lo ? 0 : b - lo >= CLASS_STEPS ? CLASS_STEPS - 1 : b - lo;
    return {cls, step, 1};
}

}  // namespace kt
