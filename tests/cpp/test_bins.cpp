// Every tail's bucket lies in the class whose kernel phase can take it.
#include <cstdio>
#include <vector>

#include "../../katric_amd/csrc/kt_bins.h"

using namespace kt;

int main() {
    std::vector<uint64_t> sizes, rows;
    for (uint64_t s = 1; s <= 300; ++s) sizes.push_back(s);
    for (uint64_t p = 512; p <= 16384; p *= 2)
        for (uint64_t s : {p - 1, p, p + 1}) sizes.push_back(s);
    for (uint64_t r = 1; r <= 300; ++r) rows.push_back(r);
    for (uint64_t p = 512; p <= (1ull << 33); p *= 2)
        for (uint64_t r : {p - 1, p, p + 1}) rows.push_back(r);
    const uint32_t none = 0xffffffffu;
    unsigned long long cases = 0;
    for (uint32_t wave_max : {1u, 2u, 32u, 64u, 128u, 256u})
        for (uint32_t group_max : {1u, 64u, 700u, 2048u})
            for (uint32_t wave_split : {16u, 32u, 64u, 128u, 256u, 512u, none})
                for (uint32_t team_split : {128u, 4096u, none})
                    for (bool min_side : {false, true})
                        for (bool hub : {false, true}) {
                            const BinRule k{wave_max, group_max, 8192, wave_split, team_split, team_split, min_side};
                            for (uint64_t s : sizes)
                                for (uint64_t r : rows) {
                                    if (wave_split == none && r > none) continue;  // entries are counted in 32 bits
                                    const TailBin t = tail_bin(s, r, k, [&] { return hub; });
                                    const int b = t.bucket + t.step;
                                    bool ok = b >= 0 && b < NBUCKET;
                                    ok = ok && (t.bucket < BUCKET_HUGE || t.step == 0);
                                    if (b < CLASS_SOLO)
                                        ok = ok && s <= PACK_MAX && r <= PACK_MAX && t.parts == 1;
                                    else if (b < CLASS_TEAM)
                                        ok = ok && s <= 256 && t.parts == 1 && (s > PACK_MAX || r > PACK_MAX);
                                    else if (b < BUCKET_HUGE)
                                        ok = ok && s <= 2048 && t.parts == 1;
                                    else if (b == BUCKET_HUGE)
                                        ok = ok && s > 8192;
                                    else if (b == BUCKET_BIG)
                                        ok = ok && s > group_max && s <= 8192;
                                    else if (b == BUCKET_WAVE_PARTS)
                                        ok = ok && s <= 256 && (uint64_t)t.parts * wave_split >= r;
                                    else
                                        ok = ok && s <= 2048 && (uint64_t)t.parts * team_split >= r;
                                    ++cases;
                                    if (!ok) {
                                        std::printf("s=%llu r=%llu wave_max=%u group_max=%u wave_split=%u team_split=%u "
                                                    "min_side=%d hub=%d: bucket %d + %d, %u parts\n",
                                                    (unsigned long long)s, (unsigned long long)r, wave_max, group_max,
                                                    wave_split, team_split, min_side, hub, t.bucket, t.step, t.parts);
                                        return 1;
                                    }
                                }
                        }
    std::printf("ALL OK (%llu cases)\n", cases);
    return 0;
}
