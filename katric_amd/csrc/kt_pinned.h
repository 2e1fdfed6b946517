// Whether a host range can be read by the device where it is.
#pragma once

#include <stdint.h>

namespace kt {

// What the runtime knows about a host address: the page-locked allocation
// [base, base + size) that holds it, and the device's address of it (null: the
// address is in no such allocation).
struct PinnedAt {
    const char* device;
    const char* base;
    uint64_t size;
};

// The device's address of p[0, bytes), or null.  The whole range has to be in
// the allocation of its first byte: with both ends page-locked the middle need
// not be (two pieces of one array registered separately), and a kernel that
// reads it there faults.
template <class Query>
const void* pinned_view(const void* p, uint64_t bytes, Query query) {
    if (!bytes) return nullptr;
    const PinnedAt a = query(p);
    if (!a.device || a.base > static_cast<const char*>(p)) return nullptr;
    const uint64_t at = (uint64_t)(static_cast<const char*>(p) - a.base);
    return at <= a.size && bytes <= a.size - at ? a.device : nullptr;
}

}  // namespace kt
