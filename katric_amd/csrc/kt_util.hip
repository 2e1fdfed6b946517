// Fill kernels: used in place of hipMemsetAsync so that every pipeline of
// the library stays capturable in a HIP graph.
#include "kt_device.h"
#include "kt_internal.h"

namespace kt {

__global__ void k_fill_u64(uint64_t* __restrict__ p, uint64_t count, uint64_t value) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

__global__ void __launch_bounds__(256) k_clear(ClearList c) {
    const uint64_t n = c.n[blockIdx.y];
    uint64_t* p = c.p[blockIdx.y];
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) p[i] = 0;
}

void clear(const ClearList& c, hipStream_t st) {
    if (c.count == 0) return;
    uint64_t most = 0;
    for (uint32_t i = 0; i < c.count; ++i) most = c.n[i] > most ? c.n[i] : most;
    const uint64_t g = (most + 1023) / 1024;
    k_clear<<<dim3((unsigned)(g > 4096 ? 4096 : g), c.count), 256, 0, st>>>(c);
}

static unsigned fill_grid(uint64_t count) {
    uint64_t g = (count + 255) / 256;
    if (g > 8192) g = 8192;
    if (g == 0) g = 1;
    return (unsigned)g;
}

void fill_u64(uint64_t* p, uint64_t count, uint64_t value, hipStream_t st) {
    if (count == 0) return;
    k_fill_u64<<<fill_grid(count), 256, 0, st>>>(p, count, value);
}

}  // namespace kt
