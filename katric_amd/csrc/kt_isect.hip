// Batched intersection of caller-given sorted id lists (kt_intersect).
//
// Replaces cetric::intersection (counters/intersection.h:40-79) for callers
// that intersect lists of their own, as tests/intersection_test.cpp:35-173
// does: the common ids of every pair are counted and, optionally, written in
// ascending order -- the order merge_intersection (:81-96) emits them in.
//
// The a ids of all pairs are one array, cut into tiles of 2048; a block takes
// a tile, resolves its ids' pairs in LDS and looks every id up by binary
// search in its pair's b list in global memory (consecutive ids of a sorted
// list share most of the search path, so it stays in the L1).  The work is
// spread over all ids whatever the pairs' lengths are: with a wave per pair,
// 300 pairs of 16 to 60000 ids left most of the chip idle and the longest pair
// took 1.2 ms.  The hits stay as a bit per id; their scan over the tiles gives
// every match its place, pair after pair in list order.  Both lists are
// checked to be strictly increasing (the reference's debug precondition,
// intersection.h:50-54): the check reads every id once.  Measured on device
// arrays, a whole call: 300 pairs of 2 to 60000 ids 93 us (1730 with a wave per
// pair), 64 pairs of 2 to 200 ids 63 us (98).
#include <algorithm>

#include "../../include/katric.h"
#include "kt_ctx.h"
#include "kt_device.h"

namespace kt {

constexpr int IS_THREADS = 256;
constexpr int IS_ITEMS = 8;  // ids of a thread
constexpr uint64_t IS_TILE = IS_THREADS * IS_ITEMS;
constexpr uint64_t SMALL_IDS = 1ull << 16;  // of both arrays: one id per thread
#define KT_ERR_ISECT_ORDER 0x1u  // a list is not strictly increasing
#define KT_ERR_ISECT_OFFSETS 0x2u

// Index of the first entry >= w in l[0, n).
__device__ __forceinline__ uint64_t lower_bound_u32(const uint32_t* __restrict__ l, uint64_t n, uint32_t w) {
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
        const uint64_t mid = (lo + hi) >> 1;
        if (l[mid] < w)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// Per pair: offsets checked (ascending, inside [0, na) / [0, nb), the id
// arrays' lengths), its count cleared, and the pairs that hold the first and
// last id of every tile of `tile` ids noted for tile_rows; the hits of every
// IS_TILE ids cleared.  Tiles that malformed offsets
// leave out keep what the workspace held: tile_rows clamps it.
__global__ void __launch_bounds__(IS_THREADS)
    k_isect_rows(uint32_t P, const uint64_t* __restrict__ aoff, uint64_t na, const uint64_t* __restrict__ boff,
                 uint64_t nb, uint64_t tile, uint64_t* __restrict__ counts, uint64_t* __restrict__ tile_cnt,
                 uint32_t* __restrict__ abnd, uint32_t* __restrict__ bbnd, uint32_t* __restrict__ err) {
    uint32_t flags = 0;
    const uint64_t stride = (uint64_t)gridDim.x * IS_THREADS;
    for (uint64_t t = (uint64_t)blockIdx.x * IS_THREADS + threadIdx.x; t * IS_TILE < na; t += stride) tile_cnt[t] = 0;
    for (uint64_t p = (uint64_t)blockIdx.x * IS_THREADS + threadIdx.x; p < P; p += stride) {
        counts[p] = 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint64_t* off = k ? boff : aoff;
            const uint64_t n = k ? nb : na, b = off[p], e = off[p + 1];
            uint32_t* bnd = k ? bbnd : abnd;
            if (e < b || e > n) {
                flags = KT_ERR_ISECT_OFFSETS;
                continue;
            }
            note_tiles((uint32_t)p, b, e, n, tile, bnd);
        }
    }
    or_flags(err, flags);
}

// Blocks [0, atiles): a tile of a ids -- order check, lookup in b, hit bits,
// the pairs' counts and those of every IS_TILE ids.  The others: a tile of b
// ids, order check.  Tiles hold ITEMS ids per thread: IS_ITEMS, or one for few
// ids, where the chip has room for a wave per 64 of them (64 pairs of up to 200
// ids: 13.4 us with eight, 6.3 with one; a pair of 48,000 and 58,000 ids, whose
// tiles all add to one count: 40 us more with one).
// A pair whose bounds are bad finds nothing (k_isect_rows flags it).
template <int ITEMS>
__global__ void __launch_bounds__(IS_THREADS)
    k_isect_tiles(uint32_t P, const uint64_t* __restrict__ aoff, const uint32_t* __restrict__ a, uint64_t na,
                  const uint64_t* __restrict__ boff, const uint32_t* __restrict__ b, uint64_t nb, uint32_t atiles,
                  const uint32_t* __restrict__ abnd, const uint32_t* __restrict__ bbnd, uint64_t* __restrict__ bits,
                  uint64_t* __restrict__ counts, uint64_t* __restrict__ tile_cnt, uint32_t* __restrict__ err) {
    constexpr int TILE = IS_THREADS * ITEMS;
    __shared__ uint32_t marks[TILE];
    __shared__ uint32_t rowcnt[TILE];
    __shared__ uint32_t wmax[IS_THREADS / KT_WAVE];
    __shared__ uint32_t wcnt[IS_THREADS / KT_WAVE];
    __shared__ uint32_t bnd[2];
    const unsigned tid = threadIdx.x, lane = lane_id();
    const bool second = blockIdx.x >= atiles;
    const uint64_t* off = second ? boff : aoff;
    const uint32_t* ids = second ? b : a;
    const uint64_t n = second ? nb : na;
    const uint32_t tile = second ? blockIdx.x - atiles : blockIdx.x;
    const uint64_t tile0 = (uint64_t)tile * TILE, tend = min(tile0 + TILE, n);
    for (int i = tid; i < TILE; i += IS_THREADS) rowcnt[i] = 0;
    uint32_t lo, hi;
    tile_rows<IS_THREADS, ITEMS>(off, P, tile0, tend, marks, bnd, wmax, lo, hi, second ? bbnd : abnd);
    const bool lds_rows = hi - lo < (uint32_t)TILE;
    uint32_t id[ITEMS], nx[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint64_t i = tile0 + k * IS_THREADS + tid;
        id[k] = i < tend ? ids[i] : 0u;
        // the id after a wave's last one
        nx[k] = (lane == KT_WAVE - 1 && i + 1 < n) ? ids[i + 1] : 0u;
    }
    // the lookups of a thread's ids go step by step together, so that their loads
    // are in flight together: one after the other, the eight chains of loads were
    // the time of a call with few short pairs
    bool hits[ITEMS] = {};
    if (!second && nb) {
        uint64_t at[ITEMS];
        uint32_t len[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const unsigned s = k * IS_THREADS + tid;
            const bool in = tile0 + s < tend;
            const uint32_t p = lo + (in ? marks[s] : 0u);
            const uint64_t b0 = boff[p], b1 = boff[p + 1];
            const bool good = in && b0 <= b1 && b1 <= nb;
            at[k] = good ? b0 : 0;
            // (a list of more ids than there are is not ascending)
            len[k] = good ? (uint32_t)min(b1 - b0, (uint64_t)0xffffffffu) : 0u;
        }
        uint32_t most = 1;
        while (most) {
            uint32_t w[ITEMS];
            most = 0;
#pragma unroll
            for (int k = 0; k < ITEMS; ++k) w[k] = b[len[k] ? at[k] + (len[k] >> 1) : 0];
#pragma unroll
            for (int k = 0; k < ITEMS; ++k) {
                const uint32_t half = len[k] >> 1;
                const bool up = len[k] && w[k] < id[k];
                hits[k] = hits[k] || (len[k] && w[k] == id[k]);
                at[k] += up ? half + 1 : 0u;
                len[k] = up ? len[k] - half - 1 : half;
                most |= len[k];
            }
        }
    }
    uint32_t flags = 0, cnt = 0;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const unsigned s = k * IS_THREADS + tid;
        const uint64_t i = tile0 + s;
        const bool in = i < tend;
        const uint32_t r = in ? marks[s] : 0xffffffffu, p = lo + r;
        const uint32_t down = __shfl_down(id[k], 1, KT_WAVE), r_down = __shfl_down(r, 1, KT_WAVE);
        const uint32_t next = lane == KT_WAVE - 1 ? nx[k] : down;
        const bool same = in && (lane == KT_WAVE - 1 ? i + 1 < n && i + 1 < off[p + 1] : r_down == r);
        if (same && id[k] >= next) flags = KT_ERR_ISECT_ORDER;
        if (second) continue;
        const bool hit = hits[k];
        const uint64_t m = __ballot(hit);
        cnt += (uint32_t)__popcll(m);
        if (lane == 0 && tile0 + s < tend) bits[(tile0 + s) / 64] = m;
        // hits per pair: one add from the last lane of every run of equal pairs
        const bool end = in && (lane == KT_WAVE - 1 || r_down != r);
        const uint64_t ends = __ballot(end);
        if (end) {
            const uint64_t below = ends & lanemask_lt();
            const uint64_t upto = lane == KT_WAVE - 1 ? ~0ull : (2ull << lane) - 1;
            const uint64_t run = upto & (below ? ~((2ull << (63 - __clzll((long long)below))) - 1) : ~0ull);
            const uint32_t c = (uint32_t)__popcll(m & run);
            if (c) {
                if (lds_rows)
                    atomicAdd(&rowcnt[r], c);
                else
                    atomic_add_u64(&counts[p], c);
            }
        }
    }
    or_flags(err, flags);
    if (second) return;
    if (lane == 0) wcnt[tid / KT_WAVE] = cnt;
    __syncthreads();
    if (lds_rows)
        for (uint32_t r = tid; r <= hi - lo; r += IS_THREADS)
            if (rowcnt[r]) atomic_add_u64(&counts[lo + r], rowcnt[r]);
    if (tid == 0) {
        uint64_t t = 0;
        for (int w = 0; w < IS_THREADS / KT_WAVE; ++w) t += wcnt[w];
        if (t) atomic_add_u64(&tile_cnt[tile0 / IS_TILE], t);
    }
}

// A wave per pair, for more pairs than a tile's 32-bit pair numbers reach: the
// shorter list is looked up in the longer.
// WRITE = false: counts[p] = |A_p cap B_p| and order / offset validation.
// WRITE = true: pair p's common ids, ascending, from out + out_off[p] on.
// A pair whose bounds are not ascending or leave [0, na) / [0, nb) (na, nb:
// the id arrays' lengths, the offsets' last entries) is flagged and skipped,
// so no read leaves the id arrays whatever the offsets hold.
template <bool WRITE>
__global__ void __launch_bounds__(IS_THREADS)
    k_isect(uint64_t P, const uint64_t* __restrict__ aoff, const uint32_t* __restrict__ a, uint64_t na,
            const uint64_t* __restrict__ boff, const uint32_t* __restrict__ b, uint64_t nb,
            uint64_t* __restrict__ counts, const uint64_t* __restrict__ out_off, uint32_t* __restrict__ out,
            uint32_t* __restrict__ err) {
    const uint32_t lane = lane_id();
    const uint64_t nw = (uint64_t)gridDim.x * (IS_THREADS / KT_WAVE);
    uint32_t flags = 0;
    for (uint64_t p = (uint64_t)blockIdx.x * (IS_THREADS / KT_WAVE) + threadIdx.x / KT_WAVE; p < P; p += nw) {
        const uint64_t a0 = aoff[p], a1 = aoff[p + 1], b0 = boff[p], b1 = boff[p + 1];
        if (a1 < a0 || b1 < b0 || a1 > na || b1 > nb) {
            flags |= KT_ERR_ISECT_OFFSETS;
            if (!WRITE && lane == 0) counts[p] = 0;
            continue;
        }
        const bool a_short = a1 - a0 <= b1 - b0;
        const uint32_t* s = a_short ? a + a0 : b + b0;
        const uint32_t* l = a_short ? b + b0 : a + a0;
        const uint64_t ns = a_short ? a1 - a0 : b1 - b0;
        const uint64_t nl = a_short ? b1 - b0 : a1 - a0;
        if (!WRITE) {
            for (uint64_t i = lane; i + 1 < nl; i += KT_WAVE)
                if (l[i] >= l[i + 1]) flags |= KT_ERR_ISECT_ORDER;
        }
        uint64_t hits = 0;
        uint64_t dst = WRITE ? out_off[p] : 0;
        for (uint64_t j = 0; j < ns; j += KT_WAVE) {
            const uint64_t i = j + lane;
            bool hit = false;
            uint32_t w = 0;
            if (i < ns) {
                w = s[i];
                if (!WRITE && i + 1 < ns && w >= s[i + 1]) flags |= KT_ERR_ISECT_ORDER;
                const uint64_t k = lower_bound_u32(l, nl, w);
                hit = k < nl && l[k] == w;
            }
            const uint64_t m = __ballot(hit);
            if (WRITE && hit) out[dst + __popcll(m & lanemask_lt())] = w;
            dst += (uint64_t)__popcll(m);
            hits += (uint64_t)__popcll(m);
        }
        if (!WRITE && lane == 0) counts[p] = hits;
    }
    or_flags(err, flags);
}

}  // namespace kt

using namespace kt;

extern "C" int kt_intersect(kt_ctx* c, uint64_t num_pairs, const uint64_t* a_offsets, const uint32_t* a_ids,
                            const uint64_t* b_offsets, const uint32_t* b_ids, uint32_t flags, uint64_t* counts,
                            uint32_t* matches, uint64_t capacity, uint64_t* total_out) {
    if (!c) return KT_EINVAL;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = c->begin_call(true);
    if (rc) return rc;
    if (!a_offsets || !b_offsets || !counts || !total_out) return c->fail(KT_EINVAL, "null argument");
    *total_out = 0;
    if (num_pairs == 0) return KT_OK;
    if (num_pairs >= (1ull << 40)) return c->fail(KT_EINVAL, "too many pairs");
    const bool host_in = !(flags & KT_DEVICE_INPUT);
    const bool dev_out = (flags & KT_DEVICE_OUTPUT) != 0;
    hipStream_t st = c->stream;
    // list lengths of the two id arrays
    uint64_t na = 0, nb = 0;
    if (host_in) {
        if (a_offsets[0] != 0 || b_offsets[0] != 0) return c->fail(KT_EINVAL, "offsets[0] != 0");
        na = a_offsets[num_pairs];
        nb = b_offsets[num_pairs];
    } else {
        uint64_t v[4];
        const uint64_t* src[4] = {a_offsets, a_offsets + num_pairs, b_offsets, b_offsets + num_pairs};
        rc = c->read_words(src, 4, v, "D2H offsets");
        if (rc) return rc;
        if (v[0] != 0 || v[2] != 0) return c->fail(KT_EINVAL, "offsets[0] != 0");
        na = v[1];
        nb = v[3];
    }
    if ((na && !a_ids) || (nb && !b_ids)) return c->fail(KT_EINVAL, "null id array");
    const uint64_t P = num_pairs;
    Carver cv{nullptr, 0};
    // (sums: of the hits of every IS_TILE ids of a, or of the pairs' counts)
    const uint64_t sums = (na + IS_TILE - 1) / IS_TILE;
    const bool small_tiles = na + nb <= SMALL_IDS;
    const uint64_t tile = small_tiles ? IS_THREADS : IS_TILE;
    const uint64_t at = (na + tile - 1) / tile, bt = (nb + tile - 1) / tile;
    const bool tiles = P < 0xffffffffull && at + bt <= 0x7fffffffull;
    const uint64_t scan_len = tiles ? sums : P;
    uint64_t *small, *aoff, *boff, *cnt, *bits, *tcnt, *toff, *stmp;
    uint32_t *a, *b, *abnd, *bbnd;
    auto layout = [&](Carver& k) {
        small = static_cast<uint64_t*>(k.take(64 * 8));
        aoff = host_in ? static_cast<uint64_t*>(k.take((P + 1) * 8)) : nullptr;
        boff = host_in ? static_cast<uint64_t*>(k.take((P + 1) * 8)) : nullptr;
        a = host_in ? static_cast<uint32_t*>(k.take(std::max<uint64_t>(na, 1) * 4)) : nullptr;
        b = host_in ? static_cast<uint32_t*>(k.take(std::max<uint64_t>(nb, 1) * 4)) : nullptr;
        cnt = static_cast<uint64_t*>(k.take(P * 8));
        bits = static_cast<uint64_t*>(k.take((na / 64 + 1) * 8));
        tcnt = tiles ? static_cast<uint64_t*>(k.take((sums + 1) * 8)) : cnt;
        toff = static_cast<uint64_t*>(k.take((scan_len + 1) * 8));
        stmp = static_cast<uint64_t*>(k.take(scan_tmp_words(scan_len + 1) * 8));
        abnd = static_cast<uint32_t*>(k.take((2 * at + 1) * 4));
        bbnd = static_cast<uint32_t*>(k.take((2 * bt + 1) * 4));
    };
    layout(cv);
    rc = c->reserve(cv.used);
    if (rc) return rc;
    cv = Carver{c->arena, 0};
    layout(cv);
    (void)hipEventRecord(c->ev[EV_START], st);
    if (host_in) {
        rc = c->hip_check(hipMemcpyAsync(aoff, a_offsets, (P + 1) * 8, hipMemcpyHostToDevice, st), "H2D");
        if (!rc) rc = c->hip_check(hipMemcpyAsync(boff, b_offsets, (P + 1) * 8, hipMemcpyHostToDevice, st), "H2D");
        if (!rc && na) rc = c->hip_check(hipMemcpyAsync(a, a_ids, na * 4, hipMemcpyHostToDevice, st), "H2D");
        if (!rc && nb) rc = c->hip_check(hipMemcpyAsync(b, b_ids, nb * 4, hipMemcpyHostToDevice, st), "H2D");
        if (rc) return rc;
    } else {
        aoff = const_cast<uint64_t*>(a_offsets);
        boff = const_cast<uint64_t*>(b_offsets);
        a = const_cast<uint32_t*>(a_ids);
        b = const_cast<uint32_t*>(b_ids);
    }
    (void)hipEventRecord(c->ev[EV_H2D], st);
    uint32_t* err = reinterpret_cast<uint32_t*>(small);
    fill_u64(small, 64, 0, st);
    const unsigned grid = (unsigned)std::min<uint64_t>((P + IS_THREADS - 1) / IS_THREADS, (uint64_t)c->num_cus * 16);
    if (tiles) {
        k_isect_rows<<<grid, IS_THREADS, 0, st>>>((uint32_t)P, aoff, na, boff, nb, tile, cnt, tcnt, abnd, bbnd, err);
        if (at + bt)
            (small_tiles ? k_isect_tiles<1> : k_isect_tiles<IS_ITEMS>)<<<(unsigned)(at + bt), IS_THREADS, 0, st>>>(
                (uint32_t)P, aoff, a, na, boff, b, nb, (uint32_t)at, abnd, bbnd, bits, cnt, tcnt, err);
    } else {
        k_isect<false><<<grid, IS_THREADS, 0, st>>>(P, aoff, a, na, boff, b, nb, cnt, nullptr, nullptr, err);
    }
    const uint64_t* end[2] = {small, toff + scan_len};
    if (tiles && sums <= 1) {  // nothing to scan
        toff = small + 1;      // zero
        end[1] = sums ? tcnt : toff;
    } else {
        scan_u64(tcnt, toff, scan_len, stmp, st);
    }
    uint64_t got[2];
    rc = c->read_words(end, 2, got, "intersect count");
    if (rc) return rc;
    const uint32_t fl = (uint32_t)got[0];
    const uint64_t total = got[1];
    if (fl & KT_ERR_ISECT_OFFSETS) return c->fail(KT_EINVAL, "pair offsets not ascending");
    if (fl & KT_ERR_ISECT_ORDER) return c->fail(KT_EINVAL, "a list is not strictly increasing");
    *total_out = total;
    c->stats.local_triangles = 0;
    c->stats.wedge_checks = 0;
    c->stats.intersection_size_local = na + nb;  // ids of both lists, as the reference counts per intersection
    rc = c->hip_check(hipMemcpyAsync(counts, cnt, P * 8, dev_out ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, st),
                      "copy counts");
    if (rc) return rc;
    if (matches && total > capacity) {
        rc = c->hip_check(hipStreamSynchronize(st), "intersect");
        if (rc) return rc;
        return c->fail(KT_ERANGE, "%llu matches do not fit a buffer of %llu", (unsigned long long)total,
                       (unsigned long long)capacity);
    }
    if (matches && total) {
        uint32_t* dm = matches;
        if (!dev_out) {
            rc = c->reserve_aux(1, total * 4);
            if (rc) return rc;
            dm = static_cast<uint32_t*>(c->aux[1]);
        }
        if (tiles)
            emit_bits_launch(na, a, bits, toff, dm, nullptr, st);
        else
            k_isect<true><<<grid, IS_THREADS, 0, st>>>(P, aoff, a, na, boff, b, nb, nullptr, toff, dm, err);
        if (!dev_out) {
            rc = c->hip_check(hipMemcpyAsync(matches, dm, total * 4, hipMemcpyDeviceToHost, st), "D2H matches");
            if (rc) return rc;
        }
    }
    (void)hipEventRecord(c->ev[EV_END], st);
    rc = c->hip_check(hipStreamSynchronize(st), "intersect");
    if (rc) return rc;
    c->timing.h2d_ms = c->elapsed(EV_START, EV_H2D);
    c->timing.count_ms = c->elapsed(EV_H2D, EV_END);
    c->timing.total_ms = c->elapsed(EV_START, EV_END);
    return KT_OK;
}
