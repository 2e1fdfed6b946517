// Which host ranges the server's gather kernel may read in place: allocations
// [100, 200), [300, 400) and, next to it, [400, 500) of a made-up address space.
#include <cstdio>

#include "../../katric_amd/csrc/kt_pinned.h"

using namespace kt;

static PinnedAt query(const void* p) {
    static const uint64_t from[] = {100, 300, 400};
    const uint64_t x = reinterpret_cast<uint64_t>(p);
    for (uint64_t b : from)
        if (x >= b && x < b + 100)
            return {reinterpret_cast<const char*>(x + 1000), reinterpret_cast<const char*>(b), 100};
    return {nullptr, nullptr, 0};
}

int main() {
    struct {
        uint64_t p, bytes;
        bool in_place;
    } cases[] = {
        {100, 100, true}, {150, 50, true},  {199, 1, true},    {100, 1, true},   {300, 100, true},
        {100, 0, false},  {100, 101, false}, {99, 10, false},  {200, 10, false}, {0, 1, false},
        {150, 200, false},  // both ends page-locked, the middle not
        {350, 100, false},  // two allocations next to each other
        {199, ~0ull, false},
    };
    for (const auto& c : cases) {
        const void* got = pinned_view(reinterpret_cast<const void*>(c.p), c.bytes, query);
        if (got != (c.in_place ? reinterpret_cast<const void*>(c.p + 1000) : nullptr)) {
            std::printf("[%llu, + %llu): %p\n", (unsigned long long)c.p, (unsigned long long)c.bytes, got);
            return 1;
        }
    }
    std::printf("ALL OK\n");
    return 0;
}
