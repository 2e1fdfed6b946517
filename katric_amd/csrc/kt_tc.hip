// Per-edge set intersection on the oriented CSR -- the hot loop of the local
// phase.  Replaces CetricEdgeIterator::run_local_* (counters/
// cetric_edge_iterator.h:229-388, 888-1066) and cetric::intersection /
// merge_intersection (counters/intersection.h:40-96) with a degree-binned
// hash-probe design for CDNA (wave64, LDS):
//
//   * a "team" -- one wave, or all eight waves of a 512-thread workgroup for
//     heavier tails -- takes a tail x and builds a bucketed hash of
//     S(x) = N+(x) in LDS (load <= 1/8 where the table allows, <= 1/2
//     at the bins' largest sets): few buckets are full, so a probe rarely
//     has to continue into the next bucket; tails of at most 64 ids and 64
//     walk entries share a wave, several at a time (pack_process);
//   * a wave takes up to 64 walk entries of R(x) at once and streams their T
//     lists as one sequence of 16-byte blocks, a block per lane and step
//     (walk_lists), the next step's blocks loaded while the current ones are
//     probed;
//   * every hit w is one emitted Triangle{x, u, w}; per-vertex counts are
//     privatised -- per-slot LDS counters for w, a count per list for u, a
//     team sum for x -- and flushed with one global atomic per non-zero counter;
//   * tails are bucketed by ceil(log2 |S(x)|), largest first; walks longer than
//     a team's share are split into parts (split_rule); the workgroups' shares
//     are fixed in advance (Shares), with queues only where they pay;
//   * tails above the workgroup bin go to 16-wave teams whose table fills a
//     workgroup's LDS (16384 slots, |S| <= 8192); only larger S(x) are probed
//     by binary search in the sorted S(x) in global memory.
//
// Counts are exact integers; the hash only changes where a set member is
// stored, never which members match.  T lists are read in aligned 16-byte
// blocks and may be touched up to 3 ids past their end: every heads array
// handed to this kernel carries 4 ids of padding.
#include <algorithm>

#include "kt_bins.h"
#include "kt_device.h"
#include "kt_internal.h"

namespace kt {

constexpr int TC_THREADS = 512;
constexpr int TC_WAVES = TC_THREADS / KT_WAVE;           // 8
constexpr uint32_t GROUP_SLOTS = 4096;                   // shared table of the 8-wave team
constexpr uint32_t WAVE_SLOTS = GROUP_SLOTS / TC_WAVES;  // private table of a 1-wave team (512)
constexpr uint32_t MIN_LOGS = 6;
// k_tc_big: one 1024-thread workgroup per CU with a 16384-slot table (128 KB
// of LDS for keys and counters), for |S| <= 8192
constexpr int BIG_THREADS = 1024;
constexpr int BIG_WAVES = BIG_THREADS / KT_WAVE;
constexpr uint32_t BIG_SLOTS = 16384;
constexpr int NXCD = 8;  // MI355X: workgroup i runs on XCD i % 8
static_assert(NXCD == CLASS_STEPS, "a class' buckets are size steps or XCDs");
static_assert(PACK_MAX == KT_WAVE, "a tail of class PACK fits a wave by itself");

// work-queue header (u32 words at the start of the workspace); every counter
// that waves update concurrently sits on its own 128-byte line so that the
// queues of different buckets land on different L2 channels:
//   [0, 29)               tails (parts) per bucket (written by binning, then read-only)
//   Q_PULL + 32 * b       pull cursor of bucket b
//   Q_FILL + 32 * b       fill cursor of bucket b (binning pass 2)
enum : int { Q_CNT = 0, Q_PULL = 32, Q_FILL = 32 * (NBUCKET + 1), Q_STRIDE = 32, Q_WORDS = 32 * (2 * NBUCKET + 2) };
// stats words after the queue header (the reference's work counters, and
// the T-list ids the probes stream)
enum : int { ST_WEDGE = 0, ST_ISZ = 1, ST_SKIP = 2, ST_STREAM = 3, ST_WORDS = 4 };
// After the stats, every workgroup's sums (ST_* and the triangles), added up by
// k_tc_finish: an atomic add per wave on the same few words held the last
// workgroups of a launch up by 250 us.  Rows: binning, k_tc_huge, k_tc_big,
// k_tc_hub, k_tc_main, of 1, 1, 1, 2 and 3 workgroups per CU.
enum : int { SUM_TOTAL = ST_WORDS, SUM_WORDS = 5 };
enum : int { ROW_BIN = 0, ROW_HUGE = 1, ROW_BIG = 2, ROW_HUB = 3, ROW_MAIN = 5, ROWS = 8 };
static uint64_t head_words(int num_cus) {
    return Q_WORDS / 2 + ST_WORDS + (uint64_t)ROWS * num_cus * SUM_WORDS;
}

template <bool PLAIN>
struct View {
    TcView v;
    __device__ __forceinline__ void s_range(uint32_t x, uint64_t& b, uint64_t& e) const {
        if (PLAIN || v.s_beg == nullptr) {
            b = v.s_off[x];
            e = v.s_off[x + 1];
        } else {
            b = v.s_beg[x];
            e = v.s_end[x];
        }
    }
    // Min-side walk (plain views with in_off set): tail x walks its whole
    // input row N(x) instead of N+(x).  The entry of an out-neighbour u
    // streams T(u) here when |T(u)| <= |S(x)| (or when T(u)'s owner has no
    // LDS table), the entry of an in-neighbour y streams T(y) here when
    // |T(y)| < |S(x)| and S(x) is in an LDS table: every oriented edge is
    // intersected exactly once, from the side whose streamed list is shorter.
    __device__ __forceinline__ bool min_side() const { return PLAIN && v.in_off != nullptr; }
    __device__ __forceinline__ void r_range(uint32_t x, uint64_t& b, uint64_t& e) const {
        if (min_side()) {
            b = v.in_off[x];
            e = v.in_off[x + 1];
        } else if (PLAIN || v.r_beg == nullptr) {
            s_range(x, b, e);
        } else {
            b = v.r_beg[x];
            e = v.r_end[x];
        }
    }
    __device__ __forceinline__ uint32_t r_head(uint64_t i) const {
        return (PLAIN || v.rheads == nullptr) ? v.sheads[i] : v.rheads[i];
    }
    __device__ __forceinline__ void t_range(uint32_t u, uint64_t& b, uint64_t& e) const {
        if (PLAIN) {
            b = v.s_off[u];
            e = v.s_off[u + 1];
        } else {
            b = v.t_beg[u];
            e = v.t_end ? v.t_end[u] : v.t_beg[u + 1];
        }
    }
    __device__ __forceinline__ const uint32_t* t_heads() const { return PLAIN ? v.sheads : v.theads; }
    // Entry i of the walk, in two dependent steps so that the first can be
    // issued a chunk ahead: entry_head loads the neighbour u (and, for a
    // min-side walk, the keep-bitmask word of the slot); entry_bounds then
    // gives the bounds of T(u) (empty when T(u) is not streamed by this tail,
    // whose |S(x)| is ns) and what the entry adds to the reference's work
    // counters (st_len to wedge_checks; st_cnt: one receiver for
    // intersection_size).
    __device__ __forceinline__ void entry_head(uint64_t i, uint32_t& u, uint32_t& kw) const {
        if (min_side()) {
            u = v.in_heads[i];
            kw = reinterpret_cast<const uint32_t*>(v.in_keep)[i >> 5];
        } else {
            u = r_head(i);
            kw = 0;
        }
    }
    __device__ __forceinline__ void entry_bounds(uint64_t i, uint32_t u, uint32_t kw, uint64_t ns, uint64_t& b,
                                                 uint64_t& e, uint64_t& st_len, bool& st_cnt) const {
        t_range(u, b, e);
        if (min_side()) {
            const bool fwd = (kw >> (i & 31)) & 1u;
            const uint64_t dr = e - b;
            st_len = fwd ? dr : 0;
            st_cnt = fwd;
            const bool here = fwd ? (dr <= ns || dr > v.in_hash_max) : (dr < ns && ns <= v.in_hash_max);
            if (!here) e = b;
            return;
        }
        st_len = e - b;
        st_cnt = !(stat_skip_empty() && e == b);
    }
    __device__ __forceinline__ void walk_entry(uint64_t i, uint64_t ns, uint32_t& u, uint64_t& b, uint64_t& e,
                                               uint64_t& st_len, bool& st_cnt) const {
        uint32_t kw;
        entry_head(i, u, kw);
        entry_bounds(i, u, kw, ns, b, e, st_len, st_cnt);
    }
    __device__ __forceinline__ uint32_t tail_pv(uint32_t x) const {
        return (PLAIN || v.tail_id == nullptr) ? x : v.tail_id[x];
    }
    // length tail x charges to intersection_size per receiver (ns = |S(x)|)
    __device__ __forceinline__ uint64_t stat_len(uint32_t x, uint64_t ns) const {
        return (!PLAIN && v.stat_off) ? v.stat_off[x + 1] - v.stat_off[x] : ns;
    }
    // the input failed its checks (read after the kernels that check it)
    __device__ __forceinline__ bool gated() const { return v.gate && (*v.gate & v.gate_bits); }
    __device__ __forceinline__ bool stat_skip_empty() const { return !PLAIN && v.stat_skip_empty; }
};

__device__ __forceinline__ uint32_t uniform(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
    uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
    uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// ---------------------------------------------------------------------------
// hubs: the (at most HUB_MAX) vertices of the highest degrees, numbered 0.. in
// no particular order.  A hub's out-neighbours have at least its degree, so
// they are hubs too: S(x) of a hub fits a table indexed by hub number, in
// which a lookup is one 2-byte LDS read (k_tc_hub).
// ---------------------------------------------------------------------------
constexpr uint32_t HUB_MAX = 32000;            // 2-byte entries: 64,000 bytes of LDS, two workgroups per CU
constexpr uint32_t HUB_NONE = 2 * HUB_MAX;     // hub-list entry of any other id: its table entry stays empty
constexpr uint32_t DEG_BINS = 1024;
constexpr int HUB_BLOCKS = 256, HUB_HIST_THREADS = 256, HUB_NUMBER_THREADS = 256;

// Monotone degree bin: exact below 64, then 32 steps per power of two.
__device__ __forceinline__ uint32_t deg_bin(uint32_t d) {
    if (d < 64) return d;
    const uint32_t e = 31u - (uint32_t)__clz(d);
    return 32 * (e - 4) + ((d >> (e - 5)) & 31);  // at most 32 * 27 + 31
}

// Hub workspace: degree histogram (vertices, then their degrees' sum, per
// bin), then the lowest hub bin, the histogram's
// finished blocks, the hubs numbered so far; the bits and number bases of 32
// vertices each; the hub lists (2-byte entries, one per oriented slot).
struct HubWs {
    uint32_t* hist;
    uint64_t* sum;
    uint32_t* min_bin;
    uint32_t* done;
    uint32_t* count;
    uint2* rs;
    uint16_t* lists;
};
enum : uint64_t { HUB_HEAD_WORDS = DEG_BINS / 2 + DEG_BINS + 2 };

static uint64_t hub_ws_words(uint32_t X, uint64_t slots) {
    // lists are read 16 bytes at a time from any entry on
    return slots ? HUB_HEAD_WORDS + ((uint64_t)X + 31) / 32 + (slots + 8 + 3) / 4 : 0;
}

static HubWs hub_ws(uint64_t* ws, uint32_t X) {
    HubWs h;
    h.hist = reinterpret_cast<uint32_t*>(ws);
    h.sum = ws + DEG_BINS / 2;
    h.min_bin = reinterpret_cast<uint32_t*>(h.sum + DEG_BINS);
    h.done = h.min_bin + 1;
    h.count = h.min_bin + 2;
    h.rs = reinterpret_cast<uint2*>(ws + HUB_HEAD_WORDS);
    h.lists = reinterpret_cast<uint16_t*>(h.rs + ((uint64_t)X + 31) / 32);
    return h;
}

// Degree histogram; the last block picks the lowest bin such that no more
// than HUB_MAX vertices are in it or above -- or none, where the hubs' rows
// hold less than a quarter of the `entries`: numbering them and writing the
// lists (0.5 ms for 106 M oriented slots of 768 mixed graphs, where hubs hold a
// sixth) then costs more than k_tc_hub gains.  The combined tails of a shard
// (rows: their lists' offsets) have the whole graph's degrees, which say nothing
// about the rank's entries: of these, the lists of the hubs that k_tc_hub would
// take (longer than wave_max) have to hold a sixth.  R-MAT, count phase without
// and with hubs: scale 22 / 2 (0.24 of the entries) 14.4 and 12.9 ms, / 4 (0.18)
// 10.5 and 10.3, / 8 (0.13) 6.88 and 6.91, / 16 (0.12) 4.41 and 4.48, scale 26 / 16
// 105.1 and 106.4.
__global__ void __launch_bounds__(HUB_HIST_THREADS) k_hub_hist(uint32_t X, const uint32_t* __restrict__ deg,
                                                               const uint64_t* __restrict__ rows, uint32_t wave_max,
                                                               uint64_t entries, HubWs h) {
    __shared__ uint32_t bins[DEG_BINS];
    __shared__ unsigned long long sums[DEG_BINS];
    __shared__ uint32_t wcnt[HUB_HIST_THREADS / KT_WAVE];
    __shared__ unsigned long long wsum[HUB_HIST_THREADS / KT_WAVE];
    __shared__ uint32_t last, pick;
    for (uint32_t i = threadIdx.x; i < DEG_BINS; i += HUB_HIST_THREADS) bins[i] = 0, sums[i] = 0;
    __syncthreads();
    // degrees below 8 are left out: a hub has more neighbours than that where hubs matter
    for (uint64_t x = (uint64_t)blockIdx.x * HUB_HIST_THREADS + threadIdx.x; x < X;
         x += (uint64_t)gridDim.x * HUB_HIST_THREADS) {
        const uint32_t d = deg[x];
        if (d >= 8) {
            atomicAdd(&bins[deg_bin(d)], 1u);
            const uint64_t len = rows ? rows[x + 1] - rows[x] : d;
            if (!rows || len > wave_max) atomicAdd(&sums[deg_bin(d)], (unsigned long long)len);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < DEG_BINS; i += HUB_HIST_THREADS)
        if (bins[i]) {
            atomicAdd(&h.hist[i], bins[i]);
            atomic_add_u64(&h.sum[i], sums[i]);
        }
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) {
        last = atomicAdd(h.done, 1u) == gridDim.x - 1;
        pick = 8;
    }
    __syncthreads();
    if (!last) return;
    // thread t takes the bins 4t .. 4t + 3 counted from the top
    constexpr uint32_t PER = DEG_BINS / HUB_HIST_THREADS;
    uint32_t c[PER], cnt = 0;
    for (uint32_t i = 0; i < PER; ++i) {
        c[i] = __hip_atomic_load(&h.hist[DEG_BINS - 1 - (threadIdx.x * PER + i)], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
        cnt += c[i];
    }
    uint32_t run = wave_incl_sum(cnt);
    if (lane_id() == KT_WAVE - 1) wcnt[threadIdx.x / KT_WAVE] = run;
    __syncthreads();
    for (uint32_t w = 0; w < threadIdx.x / KT_WAVE; ++w) run += wcnt[w];
    run -= cnt;
    for (uint32_t i = 0; i < PER; ++i) {
        // the first bin from the top that no longer fits: hubs start above it
        if (run <= HUB_MAX && run + c[i] > HUB_MAX) pick = DEG_BINS - (threadIdx.x * PER + i);
        run += c[i];
    }
    __syncthreads();
    uint64_t sum = 0;
    for (uint32_t i = threadIdx.x; i < DEG_BINS; i += HUB_HIST_THREADS)
        if (i >= pick) sum += __hip_atomic_load(&h.sum[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sum = wave_sum(sum);
    if (lane_id() == 0) wsum[threadIdx.x / KT_WAVE] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        sum = 0;
        for (int w = 0; w < HUB_HIST_THREADS / KT_WAVE; ++w) sum += wsum[w];
        *h.min_bin = (rows ? 6 * sum >= rows[X] : 4 * sum >= entries) ? pick : DEG_BINS;
    }
}

// Numbers the hubs: block b takes a contiguous run of 64-vertex words, counts
// its hubs, reserves their numbers with one atomic and writes the words.
__global__ void __launch_bounds__(HUB_NUMBER_THREADS) k_hub_number(uint32_t X, const uint32_t* __restrict__ deg, HubWs h,
                                                                 const uint32_t* __restrict__ q) {
    if (q[BUCKET_HUB_PARTS] == 0) return;
    constexpr uint32_t NW = HUB_NUMBER_THREADS / KT_WAVE;
    __shared__ uint32_t wcnt[NW];
    __shared__ uint32_t base;
    const uint32_t wave = threadIdx.x / KT_WAVE, lane = lane_id();
    const uint32_t min_bin = *h.min_bin;
    // every wave takes a contiguous run of words
    const uint64_t words = ((uint64_t)X + 63) / 64, waves = (uint64_t)gridDim.x * NW;
    const uint64_t per = (words + waves - 1) / waves, w0 = min(words, ((uint64_t)blockIdx.x * NW + wave) * per),
                   w1 = min(words, w0 + per);
    auto hub_bits = [&](uint64_t w) {
        const uint64_t x = 64 * w + lane;
        return __ballot(x < X && deg_bin(deg[x]) >= min_bin);
    };
    uint32_t c = 0;
    for (uint64_t w = w0; w < w1; ++w) c += (uint32_t)__popcll(hub_bits(w));
    if (lane == 0) wcnt[wave] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (uint32_t i = 0; i < NW; ++i) t += wcnt[i];
        base = t ? atomicAdd(h.count, t) : 0;
    }
    __syncthreads();
    uint32_t at = base;
    for (uint32_t i = 0; i < wave; ++i) at += wcnt[i];
    for (uint64_t w = w0; w < w1; ++w) {
        const uint64_t m = hub_bits(w);
        const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
        if (lane == 0) h.rs[2 * w] = uint2{lo, at};
        if (lane == 1 && 64 * w + 32 < X) h.rs[2 * w + 1] = uint2{hi, at + (uint32_t)__popc(lo)};
        at += (uint32_t)__popcll(m);
    }
}

// The hub list entry of every oriented slot: twice the hub's number (its
// table entry's byte offset), HUB_NONE for other ids.  Bound by the 8-byte
// gathers from the X / 4 byte table (L2) and HBM (4 bytes read, 2 written).
__global__ void __launch_bounds__(256) k_hub_lists(uint32_t X, const uint64_t* __restrict__ off,
                                                   const uint32_t* __restrict__ heads, HubWs h,
                                                   const uint32_t* __restrict__ q) {
    if (q[BUCKET_HUB_PARTS] == 0) return;
    const uint64_t m = off[X], stride = (uint64_t)gridDim.x * 256;
    constexpr int U = 4;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < m; i += U * stride) {
        uint32_t id[U];
        uint2 e[U];
#pragma unroll
        for (int k = 0; k < U; ++k) id[k] = heads[min(i + k * stride, m - 1)];
#pragma unroll
        for (int k = 0; k < U; ++k) e[k] = h.rs[id[k] >> 5];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const uint32_t bit = 1u << (id[k] & 31);
            const uint32_t v = (e[k].x & bit) ? 2 * (e[k].y + (uint32_t)__popc(e[k].x & (bit - 1))) : HUB_NONE;
            if (i + k * stride < m) h.lists[i + k * stride] = (uint16_t)v;
        }
    }
}

// ---------------------------------------------------------------------------
// binning: bucket tails by ceil(log2 |S(x)|), two passes (count, fill)
// ---------------------------------------------------------------------------
template <bool PLAIN>
__device__ __forceinline__ int tail_bucket(const View<PLAIN>& V, const TcParams& prm,
                                           const uint32_t* __restrict__ hub_min, uint32_t x, uint64_t& s, uint64_t& r,
                                           uint32_t& parts) {
    uint64_t sb, se, rb, re;
    parts = 1;
    V.s_range(x, sb, se);
    V.r_range(x, rb, re);
    s = se - sb;
    r = re - rb;
    if (s == 0 || r == 0 || ((PLAIN || prm.pseudo2core) && s < 2)) return -1;
    const BinRule rule{prm.wave_max_deg, prm.group_max_deg, prm.bsearch_min_deg, prm.wave_split,
                       prm.team_split,   prm.hub_split,     V.min_side()};
    const TailBin t = tail_bin(s, r, rule, [&]() { return hub_min && deg_bin(V.v.deg[x]) >= *hub_min; });
    parts = t.parts;
    if (t.bucket >= BUCKET_HUGE) return t.bucket;
    // by vertex: the XCD whose eighth of the walk entries the tail starts in
    // (an eighth of the vertices is a poor share where degrees drift with the
    // id, as in a batch: 768 mixed graphs 8.6 ms, 8.2 with this).  The entries
    // say little about the work where the lists that they stream differ with the
    // id: of a CeTriC shard's combined tails, owned first and then ghosts, one
    // eighth had twice the mean (R-MAT scale 26, rank 0 of 16: local phase 70.8 ms,
    // 49.2 in stripes of 128 to 8192; scale 20 / 16 0.48 and 0.35)
    if (prm.order == TC_BY_VERTEX) {
        if (!PLAIN) return t.bucket + (int)(((uint64_t)x * NXCD) / V.v.X);
        if (V.v.stripe) return t.bucket + (int)(x / V.v.stripe % NXCD);
        const uint64_t all = V.min_side() ? V.v.in_off[V.v.X] : V.v.s_off[V.v.X];
        return t.bucket + min(NXCD - 1, (int)((float)rb * ((float)NXCD / (float)all)));
    }
    return t.bucket + t.step;
}

// Bucket regions in one list, the highest bucket first, so that by degree the
// workgroup tails and the wave tails are each one run, largest first (the part
// buckets: in the part list, in order).
__device__ __forceinline__ uint32_t bucket_base(const uint32_t* q, int b, int cnt = Q_CNT) {
    uint32_t s = 0;
    if (b < NLIST)
        for (int i = b + 1; i < NLIST; ++i) s += q[cnt + i];
    else
        for (int i = NLIST; i < b; ++i) s += q[cnt + i];
    return s;
}

// Grid-stride over tails; per-block bucket counts in LDS, one global atomic
// per bucket per block.  ONE: one block, which knows every tail's place from its
// own counts, so it writes the list too (a call on a small graph is a chain of
// launches of 3 to 15 us each: n = 1531 115 -> 111 us with this one in place of
// two).
constexpr int BIN_THREADS = 1024;
constexpr uint32_t BIN_ONE = 4;  // tails per thread of that block
template <bool PLAIN, bool ONE>
__global__ void __launch_bounds__(BIN_THREADS) k_tc_bin_count(View<PLAIN> V, TcParams prm, uint32_t* __restrict__ q,
                                                      const uint32_t* __restrict__ hub_min,
                                                      uint64_t* __restrict__ sums, uint32_t* __restrict__ list,
                                                      uint64_t* __restrict__ plist) {
    __shared__ uint32_t cnt[NBUCKET];
    constexpr int NW = BIN_THREADS / KT_WAVE;
    __shared__ uint64_t red[3][NW];
    if (V.gated()) return;
    if (threadIdx.x < NBUCKET) cnt[threadIdx.x] = 0;
    __syncthreads();
    uint64_t wedge = 0, isz = 0, skipped = 0;
    auto tally = [&](uint32_t x, int& b, uint32_t& parts, uint32_t& rank) {
        uint64_t s, r;
        b = tail_bucket(V, prm, hub_min, x, s, r, parts);
        rank = b >= 0 ? atomicAdd(&cnt[b], parts) : 0;
        // pseudo2core: tails with fewer than two out-neighbours are skipped
        // and counted (cetric_edge_iterator.h:239-242)
        if (prm.pseudo2core && s < 2) ++skipped;
        // a plain tail with |N+(x)| == 1 emits nothing but still counts one
        // intersection in the reference's counters (cetric_edge_iterator.h:279-281)
        if (PLAIN && s == 1 && !prm.pseudo2core) {
            uint64_t sb, se, tb, te;
            V.s_range(x, sb, se);
            V.t_range(V.v.sheads[sb], tb, te);
            wedge += te - tb;
            isz += 1 + (te - tb);
        }
        // a message with receivers but no ghost entry finds no triangle and
        // is not binned; its receivers still count (cetric_edge_iterator.h:1850-1856)
        if (!PLAIN && s == 0 && r != 0) {
            uint64_t rb, re;
            V.r_range(x, rb, re);
            const uint64_t len = V.stat_len(x, 0);
            for (uint64_t i = rb; i < re; ++i) {
                uint64_t tb, te, sl;
                uint32_t u;
                bool sc;
                V.walk_entry(i, 0, u, tb, te, sl, sc);
                if (!sc) continue;
                wedge += sl;
                isz += len + sl;
            }
        }
    };
    int tb[BIN_ONE];
    uint32_t tparts[BIN_ONE], trank[BIN_ONE];
    if constexpr (ONE) {
#pragma unroll
        for (uint32_t k = 0; k < BIN_ONE; ++k) {
            const uint32_t x = k * BIN_THREADS + threadIdx.x;
            tb[k] = -1;
            if (x < V.v.X) tally(x, tb[k], tparts[k], trank[k]);
        }
    } else {
        for (uint32_t x = blockIdx.x * BIN_THREADS + threadIdx.x; x < V.v.X; x += gridDim.x * BIN_THREADS)
            tally(x, tb[0], tparts[0], trank[0]);
    }
    wedge = wave_sum(wedge);
    isz = wave_sum(isz);
    skipped = wave_sum(skipped);
    if (lane_id() == 0) {
        red[0][threadIdx.x / KT_WAVE] = wedge;
        red[1][threadIdx.x / KT_WAVE] = isz;
        red[2][threadIdx.x / KT_WAVE] = skipped;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t a = 0, c = 0, d = 0;
        for (int w = 0; w < NW; ++w) {
            a += red[0][w];
            c += red[1][w];
            d += red[2][w];
        }
        uint64_t* row = sums + (uint64_t)blockIdx.x * SUM_WORDS;
        row[ST_WEDGE] = a;
        row[ST_ISZ] = c;
        row[ST_SKIP] = d;
    }
    if constexpr (!ONE) {
        if (threadIdx.x < NBUCKET && cnt[threadIdx.x]) atomicAdd(&q[Q_CNT + threadIdx.x], cnt[threadIdx.x]);
    } else {
        __shared__ uint32_t pos[NBUCKET];
        if (threadIdx.x < NBUCKET) {
            q[Q_CNT + threadIdx.x] = cnt[threadIdx.x];
            pos[threadIdx.x] = bucket_base(cnt, (int)threadIdx.x, 0);
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < BIN_ONE; ++k) {
            if (tb[k] < 0) continue;
            const uint32_t x = k * BIN_THREADS + threadIdx.x, at = pos[tb[k]] + trank[k];
            if (tb[k] < NLIST) {
                list[at] = x;
            } else {
                for (uint32_t j = 0; j < tparts[k]; ++j) plist[at + j] = ((uint64_t)j << 32) | x;
            }
        }
    }
}

// Each block owns a contiguous range of tails: it counts its tails per
// bucket, reserves one range per bucket with a single global atomic, then
// writes its tails into the reserved ranges.
template <bool PLAIN>
__global__ void __launch_bounds__(BIN_THREADS) k_tc_bin_fill(View<PLAIN> V, TcParams prm, uint32_t* __restrict__ q,
                                                     const uint32_t* __restrict__ hub_min,
                                                     uint32_t* __restrict__ list, uint64_t* __restrict__ plist) {
    __shared__ uint32_t cnt[NBUCKET];
    __shared__ uint32_t pos[NBUCKET];
    if (V.gated()) return;
    const uint32_t X = V.v.X;
    const uint32_t per = (X + gridDim.x - 1) / gridDim.x;
    const uint32_t x0 = min(X, blockIdx.x * per), x1 = min(X, x0 + per);
    if (threadIdx.x < NBUCKET) cnt[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t x = x0 + threadIdx.x; x < x1; x += blockDim.x) {
        uint64_t s, r;
        uint32_t parts;
        int b = tail_bucket(V, prm, hub_min, x, s, r, parts);
        if (b >= 0) atomicAdd(&cnt[b], parts);
    }
    __syncthreads();
    if (threadIdx.x < NBUCKET) {
        const uint32_t c = cnt[threadIdx.x];
        pos[threadIdx.x] = c ? bucket_base(q, threadIdx.x) + atomicAdd(&q[Q_FILL + Q_STRIDE * threadIdx.x], c) : 0;
    }
    __syncthreads();
    for (uint32_t x = x0 + threadIdx.x; x < x1; x += blockDim.x) {
        uint64_t s, r;
        uint32_t parts;
        int b = tail_bucket(V, prm, hub_min, x, s, r, parts);
        if (b < 0) continue;
        const uint32_t at = atomicAdd(&pos[b], parts);
        if (b < NLIST) {
            list[at] = x;
        } else {
            for (uint32_t k = 0; k < parts; ++k) plist[at + k] = ((uint64_t)k << 32) | x;
        }
    }
}

// ---------------------------------------------------------------------------
// the team worker
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t readlane32(uint32_t x, int j) { return __builtin_amdgcn_readlane(x, j); }
__device__ __forceinline__ uint64_t readlane64(uint64_t x, int j) {
    uint32_t lo = __builtin_amdgcn_readlane((uint32_t)x, j);
    uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), j);
    return ((uint64_t)hi << 32) | lo;
}

// Per-wave scratch of the list walk: the boundary bits of a window of blocks,
// where each list's blocks are, and the lists' hit counts.
struct PackLds {
    uint32_t bits[KT_WAVE];
    uint4 rec[KT_WAVE];
    uint32_t ucnt[KT_WAVE];
};

// Bounds of a tail's S and R ranges and its counter length.
struct TailBounds {
    uint64_t sb, rb;
    uint32_t ns, nr;  // lists hold distinct 32-bit ids
    uint32_t nstat;
};

// The tails a wave has grabbed (in LDS: in registers they stay live through
// the walk, and at 80 registers a wave that put 61 of them in scratch memory).
template <uint32_t N>
struct GrabLds {
    static constexpr uint32_t MAX = N;
    uint64_t sb[N], rb[N];
    uint32_t x[N], ns[N], nr[N], nstat[N];
    __device__ __forceinline__ TailBounds bounds(uint32_t j) const { return {sb[j], rb[j], ns[j], nr[j], nstat[j]}; }
    __device__ __forceinline__ void put(uint32_t j, uint32_t tail, const TailBounds& b) {
        sb[j] = b.sb;
        rb[j] = b.rb;
        x[j] = tail;
        ns[j] = b.ns;
        nr[j] = b.nr;
        nstat[j] = b.nstat;
    }
};

// 42 of the CU's 128 LDS granules of 1280 bytes at most: three workgroups fit
// (a listing keeps its neighbours' ids beside it).
template <bool LIST>
struct Lds {
    uint32_t keys[GROUP_SLOTS];
    uint32_t cnt[GROUP_SLOTS];
    PackLds pk[TC_WAVES];
    GrabLds<LIST ? 20 : 28> grab[TC_WAVES];
    uint32_t ovf[GROUP_SLOTS / 128];  // a bit per bucket (the team's table, or 4 words per wave table)
    uint64_t red[TC_WAVES];
    unsigned long long list_ctr[TC_WAVES];  // listing: triangles of the current tail written so far
    uint32_t next_u;
    uint32_t bcast;
    uint32_t full;  // the team table has a full bucket
    uint32_t qcnt[NBUCKET], qbase[NBUCKET];  // the queue's buckets
    uint32_t qctr[NBUCKET];                  // wave grabs handed out of this workgroup's shares
};

// Team control words of k_tc_big (its table is dynamic LDS).
struct LdsBig {
    PackLds pk[BIG_WAVES];
    uint32_t ovf[BIG_SLOTS / 128];  // a bit per bucket of the dynamic-LDS table
    uint64_t red[BIG_WAVES];
    unsigned long long list_ctr[BIG_WAVES];
    uint32_t next_u;
    uint32_t bcast;
    uint32_t full;
};

template <int NW>
__device__ __forceinline__ void team_sync() {
    if (NW > 1)
        __syncthreads();
    else
        wave_sync();
}

// Bucketed hash set in LDS: 4-slot buckets (16 bytes, read with one
// ds_read_b128), filled left to right; a key lives in its home bucket
// hash(w) or, when that was full at insertion, in a later bucket (linear
// probing over buckets).  A lookup therefore ends at the first bucket that
// holds w or has an empty last slot.  A table is empty (keys KT_EMPTY, counters
// and bucket bits zero) whenever no tail uses it: the thread that inserted an
// id empties its slot again, so no pass over all slots is needed.
// Home bucket of id w as a byte offset into the table: w xor w rotated right
// by 12, masked with boff_mask = (buckets - 1) << 4 -- two full-rate
// instructions (one v_bitop3 after the rotation) that give the LDS address
// offset directly (a multiplicative hash costs a quarter-rate multiply).  The
// rotation folds the high bits onto the low ones, so ids that share their low
// bits still spread; on vertex ids it fills buckets like a multiplicative hash.
__device__ __forceinline__ uint32_t bucket_off(uint32_t w, uint32_t boff_mask) {
    return (w ^ __builtin_amdgcn_alignbit(w, w, 12)) & boff_mask;
}

__device__ __forceinline__ uint32_t* at_byte(uint32_t* base, uint32_t off) {
    return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(base) + off);
}
__device__ __forceinline__ const uint4* bucket_at(const uint32_t* keys, uint32_t off) {
    return reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(keys) + off);
}

// Inserts w into the table at byte offset toff and returns the byte offset of
// its slot; `moved` is set when w went past its home bucket (which then gets
// its bit in `ovf`, one bit per bucket).  A lookup continues past its home
// bucket only when that bucket is full and has the bit; in a table where no
// insertion went past its home bucket, every lookup ends there.
__device__ __forceinline__ uint32_t table_insert(uint32_t* keys, uint32_t* ovf, uint32_t toff, uint32_t boff_mask,
                                                 uint32_t w, bool& moved) {
    const uint32_t home = bucket_off(w, boff_mask);
    uint32_t b = home;
    bool first = true;
    while (true) {
        uint32_t* bk = at_byte(keys, toff + b);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint32_t old = atomicCAS(&bk[s], KT_EMPTY, w);
            if (old == KT_EMPTY || old == w) return toff + b + 4 * s;
        }
        if (first) atomicOr(&ovf[(toff + home) >> 9], 1u << (((toff + home) >> 4) & 31));
        b = (b + 16) & boff_mask;
        first = false;
        moved = true;
    }
}

// Probes this lane's four ids (id e valid iff e < lim) and returns its number
// of hits.  Each hit bumps the w-counter of its slot and calls
// on_hit(e).  The four slot compares of a probe stay lane masks; hits are
// counted per lane (one add), so the scalar unit only sees the branch masks.
// Two buckets are read at a time: four held 16 registers, and what the walk
// then kept in scratch memory cost more than the second read's latency (768
// mixed graphs: 9.9 ms with four, 8.9 with two).
// Lookups continue past a full home bucket only in a table where some key
// went past its home bucket (moved, wave-uniform), and only from a bucket
// with its `ovf` bit.
template <class OnHit>
__device__ __forceinline__ uint32_t probe_ids(const uint32_t* keys, uint32_t* cnt, const uint32_t* ovf, uint32_t toff,
                                              uint32_t boff_mask, bool moved, const uint32_t (&w)[4], int lim,
                                              OnHit on_hit) {
    uint32_t bo[4], last[4];
    uint32_t nh = 0;
    bool hit[4];
#pragma unroll
    for (int h = 0; h < 4; h += 2) {
        uint4 kk[2];
#pragma unroll
        for (int e = h; e < h + 2; ++e) {
            bo[e] = bucket_off(w[e], boff_mask);
            kk[e - h] = *bucket_at(keys, toff + bo[e]);
        }
#pragma unroll
        for (int e = h; e < h + 2; ++e) {
            const uint4 k = kk[e - h];
            const bool m0 = k.x == w[e], m1 = k.y == w[e], m2 = k.z == w[e], m3 = k.w == w[e];
            hit[e] = e < lim && (m0 || m1 || m2 || m3);
            nh += hit[e] ? 1u : 0u;
            if (hit[e]) {
                atomicAdd(at_byte(cnt, toff + bo[e]) + (m0 ? 0u : m1 ? 1u : m2 ? 2u : 3u), 1u);
                on_hit(e);
            }
            last[e] = k.w;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!moved) return nh;
    // a full home bucket without w: w may sit in a later bucket
    bool need[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) need[e] = e < lim && !hit[e] && last[e] != KT_EMPTY;
    // one branch for the four ids, skipped as a whole when no lane needs it
    if (need[0] || need[1] || need[2] || need[3]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (!need[e]) continue;
            // nothing went past w's home bucket: w is not in the table
            const uint32_t home = toff + bo[e];
            if (!((ovf[home >> 9] >> ((home >> 4) & 31)) & 1u)) continue;
            uint32_t b = bo[e];
            while (true) {
                b = (b + 16) & boff_mask;
                const uint4 k = *bucket_at(keys, toff + b);
                const bool n0 = k.x == w[e], n1 = k.y == w[e], n2 = k.z == w[e], n3 = k.w == w[e];
                if (n0 || n1 || n2 || n3) {
                    atomicAdd(at_byte(cnt, toff + b) + (n0 ? 0u : n1 ? 1u : n2 ? 2u : 3u), 1u);
                    on_hit(e);
                    ++nh;
                    break;
                }
                if (k.w == KT_EMPTY) break;
            }
        }
    }
    return nh;
}

struct NoHitAction {
    __device__ __forceinline__ void operator()(int) const {}
};

// 16 bytes at 4-byte alignment (T lists start anywhere); one global_load_dwordx4.
struct __attribute__((packed, aligned(4))) Ids4 {
    uint32_t x, y, z, w;
};
__device__ __forceinline__ Ids4 load_ids4(const uint32_t* p) { return *reinterpret_cast<const Ids4*>(p); }

// Binary-search probe of the sorted S(x) in global memory (huge tails).
__device__ __forceinline__ uint32_t probe_bsearch(const uint32_t* __restrict__ s, uint32_t ns, uint64_t* pv,
                                                  uint32_t w) {
    uint32_t lo = 0, hi = ns;
    while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if (s[mid] < w)
            lo = mid + 1;
        else
            hi = mid;
    }
    if (lo < ns && s[lo] == w) {
        if (pv) atomic_add_u64(&pv[w], 1);
        return 1;
    }
    return 0;
}

// Triangle listing: the calling lanes (exactly those that hit) write their
// triangles (x, u, w) of the current tail x from the tail's first output
// position on, after a team-wide running count kept in LDS.
// Writes stay inside the tail's own range [base, end) of the output even if
// this pass found more triangles than the counting pass recorded.
struct Emitter {
    uint32_t* tri;
    uint64_t base, end;
    unsigned long long* ctr;
    uint32_t x;
    __device__ __forceinline__ void operator()(uint32_t u, uint32_t w) const {
        const uint64_t m = __builtin_amdgcn_ballot_w64(true);
        const uint32_t leader = (uint32_t)__ffsll((unsigned long long)m) - 1;
        unsigned long long first = 0;
        if (lane_id() == leader) first = atomicAdd(ctr, (unsigned long long)__popcll(m));
        first = __shfl(first, (int)leader, 64);
        const uint64_t pos = base + first + (uint64_t)__popcll(m & lanemask_lt());
        if (pos < end) {
            uint32_t* t = tri + 3 * pos;
            t[0] = x;
            t[1] = u;
            t[2] = w;
        }
    }
};

// Work counters: the reference's wedge_checks and intersection_size (wedge and
// what the receivers add beside their lists), and the T-list ids this design
// streams through probes.  Kept per lane in 32 bits (a register each through
// the walk); sums that could leave them go to the workgroup's row at once.
struct WorkStats {
    uint32_t wedge_lane = 0, recv_lane = 0, stream_lane = 0;
    uint64_t* row;
    __device__ __forceinline__ explicit WorkStats(uint64_t* sums) : row(sums + (uint64_t)blockIdx.x * SUM_WORDS) {}
    __device__ __forceinline__ void flush(uint64_t wedge, uint64_t recv, uint64_t stream) {
        wedge = wave_sum(wedge);
        recv = wave_sum(recv);
        stream = wave_sum(stream);
        if (lane_id() == 0) {
            atomic_add_u64(&row[ST_WEDGE], wedge);
            atomic_add_u64(&row[ST_ISZ], wedge + recv);
            atomic_add_u64(&row[ST_STREAM], stream);
        }
    }
    __device__ __forceinline__ void add(uint64_t wedge, uint32_t recv, uint64_t stream) {
        const uint32_t high = (uint32_t)(wedge >> 32) | (uint32_t)(stream >> 32);
        const uint32_t low = (uint32_t)wedge | recv | (uint32_t)stream | wedge_lane | recv_lane | stream_lane;
        if (__builtin_amdgcn_ballot_w64((high | low >> 31) != 0)) {
            flush(wedge + wedge_lane, (uint64_t)recv + recv_lane, stream + stream_lane);
            wedge_lane = recv_lane = stream_lane = 0;
            return;
        }
        wedge_lane += (uint32_t)wedge;
        recv_lane += recv;
        stream_lane += (uint32_t)stream;
    }
};

// The workgroup's sums to its row (every wave calls it; `red` holds 4 words
// per wave).
template <int NW>
__device__ __forceinline__ void flush_sums(uint64_t total, const WorkStats& wk, uint64_t* red) {
    const uint64_t streamed = wave_sum((uint64_t)wk.stream_lane), wedge = wave_sum((uint64_t)wk.wedge_lane),
                   recv = wave_sum((uint64_t)wk.recv_lane);
    const unsigned wave = threadIdx.x / KT_WAVE;
    __syncthreads();
    if (lane_id() == 0) {
        red[4 * wave] = total;
        red[4 * wave + 1] = wedge;
        red[4 * wave + 2] = wedge + recv;
        red[4 * wave + 3] = streamed;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        uint64_t t = 0;
        for (int i = 0; i < NW; ++i) t += red[4 * i + threadIdx.x];
        const int at[4] = {SUM_TOTAL, ST_WEDGE, ST_ISZ, ST_STREAM};
        atomic_add_u64(&wk.row[at[threadIdx.x]], t);
    }
}

// Per-vertex counts: adds on one word from all XCDs take 50-100 ns each, one
// after the other, and every tail next to a hub adds to the hub's count: R-MAT
// n = 300,007 (4 M pairs) spent 200 of 870 us waiting for them.  So the
// workgroups of each XCD add to a copy of their own, and the copies are summed
// at the end (128 bytes per vertex of traffic).
__device__ __forceinline__ void own_copy(TcOut& out) { out.per_vertex += (blockIdx.x % NXCD) * out.pv_stride; }

// What the walk probes: a hash table in LDS, or (huge tails) the sorted S(x).
struct ProbeCtx {
    Emitter em;  // listing launches only
    uint32_t* keys;
    uint32_t* cnt;
    uint32_t* ovf;      // one bit per bucket: some key went past it
    uint32_t boff;      // (buckets - 1) << 4: bucket byte-offset mask
    bool full;          // some key went past its home bucket (wave-uniform)
    const uint32_t* s;  // sorted S(x) (binary-search probes)
    uint32_t ns;
    uint64_t* pv;
};

// Inclusive prefix sum over the wave (row shifts and row broadcasts, as wave_total_dpp).
__device__ __forceinline__ uint32_t wave_scan_dpp(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

__device__ __forceinline__ uint32_t rank_below(uint64_t mask, uint32_t base) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, base));
}
__device__ __forceinline__ uint32_t from_lane(uint32_t x, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4 * l), (int)x);
}
__device__ __forceinline__ uint64_t from_lane64(uint64_t x, uint32_t l) {
    return ((uint64_t)from_lane((uint32_t)(x >> 32), l) << 32) | from_lane((uint32_t)x, l);
}

// Ids of one list walked per round (its rest follows in further rounds), so
// that a chunk's ids are counted in 32 bits.
constexpr uint32_t ROUND_IDS = 1u << 18;
constexpr uint32_t WINDOW = 2048;  // blocks whose boundary bits fit one word per lane

// Streams the T lists of up to 64 walk entries through the probe: lane j's
// list is T[tb, tb + rem) (empty: rem == 0), its neighbour uj, its table the
// one at byte offset ttab >> 16 with bucket mask ttab & 0xffff (TAILS, the
// entries of several tails, each with its own table; else P.boff).  The lists
// are cut into blocks of four ids (16 bytes) and the blocks of all lists
// numbered through; a step takes 64 consecutive blocks, one per lane,
// whichever lists they belong to.  A lane finds its list from the bits that
// mark each list's last block: their number below the lane (two mbcnt) is the
// list's rank, under which its start and end lie in LDS.  So a step is full
// whatever the lists' lengths are -- a wave that walked one list at a time
// left most of its lanes idle on the short lists that most edges have (60 ids
// on average at R-MAT n = 300,007, 4 M pairs) -- and costs one list's worth
// of address work.  The next step's blocks are loaded before the current ones
// are probed.  Hits are counted per lane; a wave scan gives every list's
// share, which the lanes at the lists' ends add to the list's count in LDS.
// Returns the hits on lane j's list; `total` receives all of them.
template <bool HASH, bool TAILS, bool LIST>
__device__ __forceinline__ uint32_t walk_lists(const uint32_t* __restrict__ T, uint64_t tb, uint64_t rem, uint32_t uj,
                                               uint32_t ttab, const ProbeCtx& P, PackLds& pk, uint32_t* uid,
                                               uint64_t& total) {
    const uint32_t lane = lane_id();
    uint32_t mine = 0;
    total = 0;
    while (true) {
        const uint32_t len = (uint32_t)min<uint64_t>(rem, ROUND_IDS);
        const uint64_t nem = __builtin_amdgcn_ballot_w64(len != 0);
        if (nem == 0) break;
        const uint32_t nb = (len + 3) >> 2;
        const uint32_t incl = wave_scan_dpp(nb);
        const uint32_t first = incl - nb;  // the list's first block
        const uint32_t blocks = readlane32(incl, KT_WAVE - 1);
        const uint32_t rank = rank_below(nem, 0);
        const bool bounded = len != 0 && rank != 0;  // a list whose first block ends another's
        pk.ucnt[lane] = 0;
        if (len) {
            const uint64_t t0 = tb - 4ull * first;  // modulo 2^64: + 4 * block is inside the list
            pk.rec[rank] = uint4{(uint32_t)t0, (uint32_t)(t0 >> 32), len + 4 * first, ttab};
            if (LIST) uid[rank] = uj;
        }
        for (uint32_t w0 = 0; w0 < blocks; w0 += WINDOW) {
            pk.bits[lane] = 0;
            wave_sync();
            const uint32_t at = first - 1 - w0;
            if (bounded && at < WINDOW) atomicOr(&pk.bits[at >> 5], 1u << (at & 31));
            wave_sync();
            const uint32_t bits = pk.bits[lane];
            uint32_t base = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(bounded && first <= w0));
            wave_sync();
            const uint32_t steps = min((blocks - w0 + KT_WAVE - 1) / KT_WAVE, WINDOW / KT_WAVE);
            // step s: this lane's block, its list's rank and table, its ids'
            // number (<= 0 past the end)
            uint64_t ends = 0;
            uint32_t rk = 0, tt = 0;
            int lim = 0;
            Ids4 q;
            // (s == steps, loaded but not probed: every lane takes the step's
            // first block, which is in list `base`, or the last block there is;
            // without a branch, as the loop waits longest for its own issue)
            const uint32_t last = min(w0 + steps * KT_WAVE, blocks - 1);
            auto load = [&](uint32_t s) {
                const uint64_t on = s == steps ? 0 : ~0ull;
                const uint32_t l0 = 2 * s % KT_WAVE;
                ends = ((uint64_t)readlane32(bits, (int)l0) | ((uint64_t)readlane32(bits, (int)l0 + 1) << 32)) & on;
                rk = rank_below(ends, base);
                base += (uint32_t)__popcll(ends);
                const uint4 r = pk.rec[rk];
                const uint32_t p = w0 + s * KT_WAVE + lane;
                lim = (int)r.z - (int)(4 * p);  // past the last block: its list's, and not above zero
                tt = r.w;
                q = load_ids4(T + ((((uint64_t)r.y << 32) | r.x) + 4ull * min(p, last)));
            };
            load(0);
            for (uint32_t s = 0; s < steps; ++s) {
                const uint32_t w[4] = {q.x, q.y, q.z, q.w};
                const uint64_t c_ends = ends;
                const uint32_t c_rk = rk;
                const uint32_t c_off = TAILS ? tt >> 16 : 0u, c_mask = TAILS ? tt & 0xffffu : P.boff;
                const int c_lim = lim;
                load(s + 1);
                uint32_t nh = 0;
                if (HASH) {
                    if constexpr (LIST) {
                        const uint32_t u = uid[c_rk];
                        nh = probe_ids(P.keys, P.cnt, P.ovf, c_off, c_mask, P.full, w, c_lim,
                                       [&](int e) { P.em(u, w[e]); });
                    } else {
                        nh = probe_ids(P.keys, P.cnt, P.ovf, c_off, c_mask, P.full, w, c_lim, NoHitAction{});
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (e >= c_lim) continue;
                        const uint32_t h = probe_bsearch(P.s, P.ns, P.pv, w[e]);
                        nh += h;
                        if (LIST && h) P.em(uid[c_rk], w[e]);
                    }
                }
                if (__builtin_amdgcn_ballot_w64(nh != 0)) {
                    const uint32_t sum = wave_scan_dpp(nh);
                    total += readlane32(sum, KT_WAVE - 1);
                    const bool end = (c_ends >> lane) & 1;
                    if (end || lane == KT_WAVE - 1) atomicAdd(&pk.ucnt[c_rk], sum);
                    if (end && lane != KT_WAVE - 1) atomicSub(&pk.ucnt[c_rk + 1], sum);
                }
            }
            wave_sync();
        }
        if (len) mine += pk.ucnt[rank];
        wave_sync();
        tb += len;
        rem -= len;
    }
    return mine;
}

template <bool PLAIN>
__device__ __forceinline__ TailBounds tail_bounds(const View<PLAIN>& V, uint32_t x) {
    TailBounds t;
    uint64_t e;
    V.s_range(x, t.sb, e);
    t.ns = (uint32_t)(e - t.sb);
    V.r_range(x, t.rb, e);
    t.nr = (uint32_t)(e - t.rb);
    t.nstat = (uint32_t)V.stat_len(x, t.ns);
    return t;
}

// Bounds of part `part` (of `split` walk entries) of tail x.
template <bool PLAIN>
__device__ __forceinline__ TailBounds part_bounds(const View<PLAIN>& V, uint32_t x, uint32_t part, uint32_t split) {
    TailBounds t = tail_bounds(V, x);
    t.rb += (uint64_t)part * split;
    t.nr = min(split, t.nr - part * split);
    return t;
}

// Process tail x, whose bounds are tb, with a team of NW waves (NW == 1:
// this wave alone); KS: the most ids of S(x) per thread.
template <int NW, int KS, bool HASH, bool PLAIN, bool LIST, class LdsT>
__device__ __forceinline__ void team_process(const View<PLAIN>& V, uint32_t x, const TailBounds& tb, LdsT& L,
                                             uint32_t* keys, uint32_t* cnt, uint32_t* ovf, uint32_t cap_slots,
                                             uint32_t shift, uint32_t chunk, const TcOut& out,
                                             uint64_t& my_total, WorkStats& wk, uint32_t* uid) {
    const unsigned lane = lane_id();
    const unsigned wave = threadIdx.x / KT_WAVE;
    const unsigned twave = NW > 1 ? wave : 0;
    const unsigned tid = twave * KT_WAVE + lane;

    const uint64_t sb = uniform64(tb.sb), rb = uniform64(tb.rb);
    const uint32_t ns = uniform(tb.ns), nr = uniform(tb.nr), nstat = uniform(tb.nstat);
    // every wave of the team gets at least two grabs where the walk allows
    if (NW > 1) chunk = min(chunk, max(1u, (nr + 2 * NW - 1) / (2 * NW)));
    // The first chunk's neighbours are loaded before the tail's table is
    // built (inserting S(x) hides the round trip); every later chunk's
    // neighbours are loaded while the chunk before it is scanned (the bounds
    // of their T lists depend on them).
    uint32_t k = twave * chunk;
    uint32_t u_nx = 0, kw_nx = 0;
    if (k < nr && lane < min(chunk, nr - k)) V.entry_head(rb + k + lane, u_nx, kw_nx);

    ProbeCtx P;
    P.keys = keys;
    P.cnt = cnt;
    P.ovf = ovf;
    P.boff = 0;
    P.full = false;
    P.s = V.v.sheads + sb;
    P.ns = ns;
    P.pv = out.per_vertex;
    uint32_t slot[(KS + 1) / 2] = {};  // where this thread's ids of S(x) are (byte offsets, two per word)
    if (HASH) {
        uint32_t logS = max(ceil_log2((uint64_t)ns << shift), MIN_LOGS);  // load <= 2^-shift unless capped
        logS = min(logS, 31u - (uint32_t)__clz(cap_slots));               // bins guarantee cap_slots >= 2 * ns
        P.boff = ((1u << logS >> 2) - 1) << 4;
        bool full = false;
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const uint32_t i = tid + j * NW * KT_WAVE;
            if (i < ns) slot[j / 2] |= table_insert(keys, ovf, 0, P.boff, P.s[i], full) << (16 * (j & 1));
        }
        if (NW > 1) {
            if (full) L.full = 1;
        } else {
            P.full = __builtin_amdgcn_ballot_w64(full) != 0;
        }
    }
    if (NW > 1 && tid == 0) L.next_u = NW * chunk;
    if (LIST) {
        P.em = Emitter{out.tri, out.tail_off[x], out.tail_off[x + 1], &L.list_ctr[NW > 1 ? 0 : wave], x};
        if (tid == 0) *P.em.ctr = 0;
    }
    team_sync<NW>();
    if (HASH && NW > 1) P.full = uniform(L.full) != 0;

    uint64_t hsum = 0;  // wave-uniform
    while (k < nr) {
        const uint32_t c = min(chunk, nr - k);
        const uint32_t u = u_nx, kw = kw_nx;
        uint32_t nk;
        if (NW > 1) {
            uint32_t g = 0;
            if (lane == 0) g = atomicAdd(&L.next_u, chunk);
            nk = uniform(g);
        } else {
            nk = k + chunk;
        }
        if (nk < nr && lane < min(chunk, nr - nk)) V.entry_head(rb + nk + lane, u_nx, kw_nx);
        uint64_t b = 0, e = 0, stl = 0;
        bool stc = false;
        if (lane < c) V.entry_bounds(rb + k + lane, u, kw, ns, b, e, stl, stc);
        const uint64_t len = e > b ? e - b : 0;
        wk.add(stl, stc ? nstat : 0u, len);
        uint64_t hits;
        const uint32_t h = walk_lists<HASH, false, LIST>(V.t_heads(), b, len, u, 0, P, L.pk[wave], uid, hits);
        if (h && P.pv) atomic_add_u64(&P.pv[u], h);
        hsum += hits;
        k = nk;
    }

    // team reduction of the tail's hits
    if (NW > 1) {
        if (lane == 0) L.red[wave] = hsum;
        __syncthreads();
        hsum = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) hsum += L.red[i];
    }
    if (HASH) {
        if (NW == 1) wave_sync();
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            if (tid + j * NW * KT_WAVE >= ns) break;
            const uint32_t o = (slot[j / 2] >> (16 * (j & 1))) & 0xffffu;
            const uint32_t c = *at_byte(cnt, o);
            if (c) {
                if (P.pv) atomic_add_u64(&P.pv[*at_byte(keys, o)], c);
                *at_byte(cnt, o) = 0;
            }
            *at_byte(keys, o) = KT_EMPTY;
        }
        if (P.full)
            for (uint32_t i = tid; i < (P.boff >> 9) + 1; i += NW * KT_WAVE) ovf[i] = 0;
        if (NW > 1 && tid == 0) L.full = 0;  // read by every wave before the walk
    }
    if (tid == 0 && out.tail_count) out.tail_count[x] = hsum;
    if (tid == 0 && hsum) {
        if (P.pv) atomic_add_u64(&P.pv[V.tail_pv(x)], hsum);
        my_total += hsum;
    }
    team_sync<NW>();  // table reuse by the next tail
}

// Tails that a wave takes several at a time, so that the entries and set
// members of a few such tails fill one wave.  (One by one, each tail of R-MAT
// or G(n, m) -- 16 to 36 entries on average -- cost the wave a chain of six
// dependent round trips with most of its lanes idle: 12-19 us.)
__device__ __forceinline__ uint32_t pack_slots(uint32_t ns) {  // load 1/8 to 1/4
    return 1u << max(ceil_log2(4ull * ns), 4u);
}

// Tails [j0, j0 + n) of a grab; lane j's walk entries, set members and table
// slots start er, es and et after the pack's first.
template <bool PLAIN, class GrabT>
__device__ __forceinline__ void pack_process(const View<PLAIN>& V, const GrabT& gb, uint32_t er, uint32_t es,
                                             uint32_t et, uint32_t j0, uint32_t n, uint32_t nR, uint32_t nS,
                                             PackLds& pk, uint32_t* keys, uint32_t* cnt, uint32_t* ovf,
                                             const TcOut& out, uint64_t& my_total, WorkStats& wk) {
    const uint32_t lane = lane_id();
    // which tail a lane's entry / set member belongs to, from the bits at the
    // tails' last ones
    pk.bits[lane] = 0;
    wave_sync();
    if (lane > j0 && lane < j0 + n) {
        atomicOr(&pk.bits[(er - 1) >> 5], 1u << ((er - 1) & 31));
        atomicOr(&pk.bits[2 + ((es - 1) >> 5)], 1u << ((es - 1) & 31));
    }
    wave_sync();
    const uint32_t word = pk.bits[lane];
    wave_sync();
    const uint64_t mr = (uint64_t)readlane32(word, 0) | ((uint64_t)readlane32(word, 1) << 32);
    const uint64_t ms = (uint64_t)readlane32(word, 2) | ((uint64_t)readlane32(word, 3) << 32);
    // (at most the grab's last tail: lanes past the pack's entries read it)
    const uint32_t tr = j0 + rank_below(mr, 0), ts = j0 + rank_below(ms, 0);
    const uint32_t tab = (4 * et << 16) | (((pack_slots(gb.ns[min(lane, GrabT::MAX - 1)]) >> 2) - 1) << 4);
    // set members and walk entries
    const uint64_t si = gb.sb[ts] + (lane - from_lane(es, ts));
    const uint64_t ri = gb.rb[tr] + (lane - from_lane(er, tr));
    const uint32_t stab = from_lane(tab, ts), rtab = from_lane(tab, tr);
    uint32_t id = 0, u = 0, kw = 0;
    if (lane < nS) id = V.v.sheads[si];
    if (lane < nR) V.entry_head(ri, u, kw);
    uint32_t slot = 0;
    bool moved = false;
    if (lane < nS) slot = table_insert(keys, ovf, stab >> 16, stab & 0xffffu, id, moved);
    ProbeCtx P;
    P.keys = keys;
    P.cnt = cnt;
    P.ovf = ovf;
    P.boff = 0;
    P.full = __builtin_amdgcn_ballot_w64(moved) != 0;
    P.pv = out.per_vertex;
    uint64_t b = 0, e = 0, stl = 0;
    bool stc = false;
    if (lane < nR) V.entry_bounds(ri, u, kw, gb.ns[tr], b, e, stl, stc);
    const uint64_t len = e > b ? e - b : 0;
    wk.add(stl, stc ? (PLAIN ? gb.ns[tr] : gb.nstat[tr]) : 0u, len);
    uint64_t hits;
    const uint32_t h = walk_lists<true, true, false>(V.t_heads(), b, len, u, rtab, P, pk, nullptr, hits);
    if (hits) {
        my_total += hits;
        if (P.pv) {
            if (h) atomic_add_u64(&P.pv[u], h);
            const uint32_t sum = wave_scan_dpp(h), j = min(lane, GrabT::MAX - 1);
            const uint32_t last = from_lane(sum, er + gb.nr[j] - 1), before = from_lane(sum, er - 1);
            const uint32_t th = last - (lane > j0 ? before : 0u);
            if (lane >= j0 && lane < j0 + n && th) atomic_add_u64(&P.pv[V.tail_pv(gb.x[j])], th);
        }
    }
    if (lane < nS) {
        const uint32_t c = *at_byte(cnt, slot);
        if (c) {
            if (P.pv) atomic_add_u64(&P.pv[*at_byte(keys, slot)], c);
            *at_byte(cnt, slot) = 0;
        }
        *at_byte(keys, slot) = KT_EMPTY;
    }
    if (P.full && lane < WAVE_SLOTS / 128) ovf[lane] = 0;
    wave_sync();
}

// A run of the tail list.
struct Segment {
    uint32_t base, cnt;
};

// The segment of a class (a bucket of parts: that bucket): by vertex the
// bucket of XCD sx, by degree all eight, largest first.
template <class LdsT>
__device__ __forceinline__ Segment class_segment(const LdsT& L, int cls, bool parts, bool by_vertex, uint32_t sx) {
    if (parts) return {L.qbase[cls], L.qcnt[cls]};
    if (by_vertex) return {L.qbase[cls + sx], L.qcnt[cls + sx]};
    return {L.qbase[cls + NXCD - 1], L.qbase[cls] + L.qcnt[cls] - L.qbase[cls + NXCD - 1]};
}

// How a segment is shared out without a queue access: an atomic on one word
// that many XCDs update costs 50-100 ns, one after the other (with every tail
// taken from a queue, R-MAT n = 300,007 with 4 M pairs spent 1.2 of its
// 1.4 ms on them), so the first items go to the workgroups in turn.  `whole`:
// the segment is shared by the grid, starting at workgroup rot, else by the
// workgroups of XCD sx.
struct Shares {
    uint32_t first, blocks;
    bool mine;
    __device__ __forceinline__ Shares(uint32_t cnt, bool whole, uint32_t sx, uint32_t rot) {
        whole = whole || cnt < 4 * gridDim.x;  // too few for the XCD's own caches to matter
        if (whole) {
            blocks = gridDim.x;
            first = (blockIdx.x + blocks - rot % blocks) % blocks;
            mine = true;
        } else {
            blocks = (gridDim.x + NXCD - 1 - sx) / NXCD;
            first = blockIdx.x / NXCD;
            mine = blockIdx.x % NXCD == sx;
        }
    }
};

// 80 VGPRs and 51.6 KB of LDS: three workgroups per CU, 6 waves per SIMD.  Bound
// by the chain of dependent loads that every pack or chunk of 64 entries starts
// with, and by VALU (72 % busy at R-MAT scale 22, where it takes 2.7 ms; 768
// mixed graphs 6.0 ms).  On a large shard's long lists VALU and latency, which its
// 24 waves a CU hide less of than 32 would (R-MAT scale 26, rank 0 of 16: local
// phase 47 ms, contracted phase 56).
template <bool PLAIN, bool LIST>
__global__ void __launch_bounds__(TC_THREADS) __attribute__((amdgpu_waves_per_eu(6, 6))) k_tc_main(View<PLAIN> V, TcOut out, TcParams prm,
                                                         uint32_t* __restrict__ q,
                                                         const uint32_t* __restrict__ list,
                                                         const uint64_t* __restrict__ plist,
                                                         uint64_t* __restrict__ sums) {
    own_copy(out);
    __shared__ Lds<LIST> L;
    __shared__ uint32_t uids[LIST ? TC_THREADS : 1];  // a listing's neighbours, per wave
    const unsigned wave = threadIdx.x / KT_WAVE;
    const unsigned lane = lane_id();
    uint32_t* uid = uids + (LIST ? wave * KT_WAVE : 0);
    uint64_t my_total = 0;
    WorkStats wk(sums);

    // Every bucket's count and place in the list, read once.
    if (wave == 0) {
        const uint32_t c = lane < (unsigned)NBUCKET ? q[Q_CNT + lane] : 0u;
        if (lane < (unsigned)NBUCKET) {
            L.qcnt[lane] = c;
            L.qctr[lane] = 0;
        }
        uint32_t base = 0;
        for (int i = 0; i < NBUCKET; ++i) {
            const uint32_t ci = readlane32(c, i);
            const bool same = (i < NLIST) == (lane < (unsigned)NLIST);
            base += (same && (i < NLIST ? i > (int)lane : i < (int)lane)) ? ci : 0u;
        }
        if (lane < (unsigned)NBUCKET) L.qbase[lane] = base;
    }
    for (uint32_t i = threadIdx.x; i < GROUP_SLOTS; i += TC_THREADS) {
        L.keys[i] = KT_EMPTY;
        L.cnt[i] = 0;
    }
    if (threadIdx.x < GROUP_SLOTS / 128) L.ovf[threadIdx.x] = 0;
    if (threadIdx.x == 0) L.full = 0;
    __syncthreads();
    const bool by_vertex = prm.order == TC_BY_VERTEX;
    const uint32_t xcd = blockIdx.x % NXCD;
    // Shares of a segment start where those of the one before ended (by
    // vertex, where the order of the segments differs per XCD: an eighth of the
    // grid further per XCD), so that every workgroup gets as many.
    const uint32_t team_parts = L.qcnt[BUCKET_TEAM_PARTS], wave_parts = L.qcnt[BUCKET_WAVE_PARTS];
    // team phase: the parts of long walks, then, by degree, the workgroup
    // tails from the largest down (one segment); by vertex, this XCD's
    // workgroup tails first, then the other XCDs'
    for (uint32_t k = 0; k <= (by_vertex ? NXCD : 1u); ++k) {
        const bool parts = k == 0;
        const uint32_t sx = (xcd + k - 1) % NXCD;  // by vertex: the segment's XCD
        const Segment sg = class_segment(L, parts ? BUCKET_TEAM_PARTS : CLASS_TEAM, parts, by_vertex, sx);
        if (sg.cnt == 0) continue;
        const Shares sh(sg.cnt, parts || !by_vertex, sx, parts ? 0 : by_vertex ? sx * (gridDim.x / NXCD) : team_parts);
        uint32_t* pull = &q[Q_PULL + Q_STRIDE * (parts ? BUCKET_TEAM_PARTS : CLASS_TEAM + (by_vertex ? (int)sx : 0))];
        const uint32_t fixed = !by_vertex || sg.cnt <= 4 * sh.blocks ? sg.cnt : sg.cnt - sg.cnt / 4;
        uint32_t i = sh.mine ? sh.first : fixed;
        while (true) {
            if (i >= fixed) {
                if (fixed == sg.cnt) break;
                if (threadIdx.x == 0)
                    L.bcast = (__hip_atomic_load(pull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= sg.cnt - fixed)
                                  ? sg.cnt
                                  : fixed + atomicAdd(pull, 1u);
                __syncthreads();
                i = L.bcast;
                __syncthreads();
                if (i >= sg.cnt) break;
            }
            const uint64_t xp = parts ? plist[sg.base + i] : list[sg.base + i];
            const uint32_t x = (uint32_t)xp;
            const TailBounds tb =
                parts ? part_bounds(V, x, (uint32_t)(xp >> 32), prm.team_split) : tail_bounds(V, x);
            team_process<TC_WAVES, GROUP_SLOTS / 2 / TC_THREADS, true, PLAIN, LIST>(V, x, tb, L, L.keys, L.cnt, L.ovf, GROUP_SLOTS,
                                                          prm.table_shift, prm.team_chunk, out, my_total, wk, uid);
            i = i < fixed ? i + sh.blocks : fixed;
        }
    }
    // wave phase: independent waves with private tables: the parts, the SOLO
    // tails (a few per grab: they are the long ones, and a grab that holds
    // several ends late), then the PACK tails.  Grabs are the workgroup's share,
    // handed out by an LDS counter: with the last quarter of a segment taken from
    // a queue, its word's atomics at 41 ns each were the time (G(n, m) n =
    // 900,000, 3.6 M pairs 842 us by degree, 243 without; R-MAT scale 22 14.4 and
    // 12.2 ms).  By vertex a queue per XCD also lets an XCD that is done help the
    // others, which counts in long segments only: 8192 mixed graphs (290 grabs a
    // wave) 82 ms with and 93 without, 768 of them (31 and 34 grabs) 8.2 and 9.0,
    // G(n, m) n = 900,000 (8 grabs) 372 and 245 us.
    {
        uint32_t* keys = L.keys + wave * WAVE_SLOTS;
        uint32_t* tcnt = L.cnt + wave * WAVE_SLOTS;
        uint32_t* wovf = L.ovf + wave * (WAVE_SLOTS / 128);
        const uint32_t segs = by_vertex ? NXCD : 1u;
        for (uint32_t k = 0; k <= 2 * segs; ++k) {
            const bool parts = k == 0, pack = k > segs;
            const uint32_t sx = (xcd + k - 1) % NXCD;
            const int cls = parts ? BUCKET_WAVE_PARTS : pack ? CLASS_PACK : CLASS_SOLO;
            const Segment sg = class_segment(L, cls, parts, by_vertex, sx);
            if (sg.cnt == 0) continue;
            const Shares sh(sg.cnt, parts || !by_vertex, sx,
                            parts ? 0 : by_vertex ? sx * (gridDim.x / NXCD) : wave_parts);
            const bool packs = !LIST && pack && !out.tail_count;
            // SOLO tails: two while a wave gets at least four grabs, from 32 grabs a
            // wave on up to eight (one round trip for the bounds of all: R-MAT
            // scale 26, rank 0 of 16, DiTriC's distributed phase 64.6 -> 64.0 ms
            // with 4, 8 or 16; no change at scale 22 and for batches)
            const uint32_t most = pack ? min(max(prm.wave_grab, 1u), L.grab[0].MAX) : 2u;
            const uint32_t per_wave = sg.cnt / (TC_WAVES * sh.blocks);
            const uint32_t grab = max(max(1u, min(most, per_wave / 4)), pack ? 0u : min(8u, per_wave / 32));
            const uint32_t grabs = (sg.cnt + grab - 1) / grab;
            const uint32_t fixed = !by_vertex || grabs <= (pack ? 24 : 16) * TC_WAVES * sh.blocks ? grabs : grabs - grabs / 4;
            const int qi = parts ? cls : cls + (by_vertex ? (int)sx : 0);
            uint32_t* pull = &q[Q_PULL + Q_STRIDE * qi];
            bool own = sh.mine;
            while (true) {
                uint32_t g = 0;
                if (own) {
                    if (lane == 0) g = sh.first + atomicAdd(&L.qctr[qi], 1u) * sh.blocks;
                    g = uniform(g);
                    own = g < fixed;
                }
                if (!own) {
                    if (fixed == grabs) break;
                    if (lane == 0)
                        g = (__hip_atomic_load(pull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= grabs - fixed)
                                ? grabs
                                : fixed + atomicAdd(pull, 1u);
                    g = uniform(g);
                    if (g >= grabs) break;
                }
                // the grabbed tails and their bounds, loaded by one lane each
                // before the first is processed: one round trip for the batch
                // instead of two per tail
                const uint32_t i = g * grab;
                const uint32_t ng = min(sg.cnt, i + grab) - i;
                auto& gb = L.grab[wave];
                uint32_t nr = 0, ns = 0;
                if (lane < ng) {
                    const uint64_t xp = parts ? plist[sg.base + i + lane] : list[sg.base + i + lane];
                    const TailBounds bl = parts ? part_bounds(V, (uint32_t)xp, (uint32_t)(xp >> 32), prm.wave_split)
                                                : tail_bounds(V, (uint32_t)xp);
                    gb.put(lane, (uint32_t)xp, bl);
                    nr = bl.nr;
                    ns = bl.ns;
                }
                wave_sync();
                uint32_t j = 0;
                if (packs) {
                    // Consecutive small tails are taken together while their
                    // entries, set members and tables fit the wave.  (Every tail
                    // of the class fits by itself; the sums are of capped sizes
                    // and the loop ends at one that does not, so that no bin
                    // rule could make it spin.)
                    const uint32_t rs = wave_scan_dpp(min(nr, 2 * PACK_MAX) << 16 | min(ns, 2 * PACK_MAX)),
                                   st = wave_scan_dpp(lane < ng ? pack_slots(ns) : 0u);
                    while (j < ng) {
                        const uint32_t brs = j ? readlane32(rs, j - 1) : 0u, bt = j ? readlane32(st, j - 1) : 0u;
                        const uint32_t in = rs - brs;  // (both halves ascend: no borrow from lane j on)
                        const bool fits = lane < ng && (in >> 16) <= KT_WAVE && (in & 0xffffu) <= KT_WAVE &&
                                          st - bt <= WAVE_SLOTS;
                        const uint64_t run = __builtin_amdgcn_ballot_w64(fits) >> j;
                        const uint32_t n = (uint32_t)__builtin_ctzll(~run);
                        if (n == 0) break;
                        const uint32_t last = readlane32(in, j + n - 1), k = min(lane, gb.MAX - 1);
                        pack_process(V, gb, (in >> 16) - gb.nr[k], (in & 0xffffu) - gb.ns[k],
                                     st - pack_slots(gb.ns[k]) - bt, j, n, last >> 16, last & 0xffffu, L.pk[wave], keys,
                                     tcnt, wovf, out, my_total, wk);
                        j += n;
                    }
                }
                for (; j < ng; ++j)
                    team_process<1, WAVE_SLOTS / 2 / KT_WAVE, true, PLAIN, LIST>(
                        V, uniform(gb.x[j]), gb.bounds(j), L, keys, tcnt, wovf, WAVE_SLOTS, prm.table_shift, KT_WAVE,
                        out, my_total, wk, uid);
                wave_sync();  // the records are written again
            }
        }
    }
    flush_sums<TC_WAVES>(my_total, wk, reinterpret_cast<uint64_t*>(L.keys));
}

// Tails whose S(x) exceeds the LDS table: 8-wave teams, binary-search probes
// of the sorted S(x) in global memory.
template <bool PLAIN, bool LIST>
__global__ void __launch_bounds__(TC_THREADS) k_tc_huge(View<PLAIN> V, TcOut out, TcParams prm,
                                                         uint32_t* __restrict__ q,
                                                         const uint32_t* __restrict__ list,
                                                         uint64_t* __restrict__ sums) {
    own_copy(out);
    __shared__ Lds<LIST> L;
    __shared__ uint32_t uids[LIST ? TC_THREADS : 1];
    uint32_t* uid = uids + (LIST ? threadIdx.x / KT_WAVE * KT_WAVE : 0);
    uint64_t my_total = 0;
    WorkStats wk(sums);
    const uint32_t cnt = q[Q_CNT + BUCKET_HUGE];
    if (cnt == 0) return;
    const uint32_t base = bucket_base(q, BUCKET_HUGE);
    uint32_t* pull = &q[Q_PULL + Q_STRIDE * BUCKET_HUGE];
    while (true) {
        if (threadIdx.x == 0)
            L.bcast = (__hip_atomic_load(pull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= cnt)
                          ? cnt
                          : atomicAdd(pull, 1u);
        __syncthreads();
        const uint32_t i = L.bcast;
        __syncthreads();
        if (i >= cnt) break;
        const uint32_t x = list[base + i];
        team_process<TC_WAVES, 1, false, PLAIN, LIST>(V, x, tail_bounds(V, x), L, nullptr, nullptr, nullptr, 0, 0,
                                                            prm.team_chunk, out, my_total, wk, uid);
    }
    flush_sums<TC_WAVES>(my_total, wk, reinterpret_cast<uint64_t*>(L.keys));
}

// Tails above the workgroup bin whose hash table fits one workgroup's LDS
// (|S| <= 8192): a 16-wave team per tail with a 16384-slot table in dynamic
// LDS, one workgroup per CU.
template <bool PLAIN, bool LIST>
__global__ void __launch_bounds__(BIG_THREADS) k_tc_big(View<PLAIN> V, TcOut out, TcParams prm,
                                                        uint32_t* __restrict__ q, const uint32_t* __restrict__ list,
                                                        uint64_t* __restrict__ sums) {
    own_copy(out);
    __shared__ LdsBig L;
    __shared__ uint32_t uids[LIST ? BIG_THREADS : 1];
    uint32_t* uid = uids + (LIST ? threadIdx.x / KT_WAVE * KT_WAVE : 0);
    extern __shared__ uint32_t big_table[];  // keys[BIG_SLOTS], then cnt[BIG_SLOTS]
    if (q[Q_CNT + BUCKET_BIG] == 0) return;
    for (uint32_t i = threadIdx.x; i < BIG_SLOTS; i += BIG_THREADS) {
        big_table[i] = KT_EMPTY;
        big_table[BIG_SLOTS + i] = 0;
    }
    if (threadIdx.x < BIG_SLOTS / 128) L.ovf[threadIdx.x] = 0;
    if (threadIdx.x == 0) L.full = 0;
    uint64_t my_total = 0;
    WorkStats wk(sums);
    const uint32_t cnt = q[Q_CNT + BUCKET_BIG];
    const uint32_t base = bucket_base(q, BUCKET_BIG);
    uint32_t* pull = &q[Q_PULL + Q_STRIDE * BUCKET_BIG];
    while (true) {
        if (threadIdx.x == 0)
            L.bcast = (__hip_atomic_load(pull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= cnt)
                          ? cnt
                          : atomicAdd(pull, 1u);
        __syncthreads();
        const uint32_t i = L.bcast;
        __syncthreads();
        if (i >= cnt) break;
        const uint32_t x = list[base + i];
        team_process<BIG_WAVES, BIG_SLOTS / 2 / BIG_THREADS, true, PLAIN, LIST>(V, x, tail_bounds(V, x), L, big_table,
                                                            big_table + BIG_SLOTS, L.ovf, BIG_SLOTS, prm.table_shift,
                                                            prm.team_chunk, out, my_total, wk, uid);
    }
    flush_sums<BIG_WAVES>(my_total, wk, reinterpret_cast<uint64_t*>(big_table));
}

// ---------------------------------------------------------------------------
// hub tails
// ---------------------------------------------------------------------------
constexpr int HUB_THREADS = 768;
constexpr int HUB_WAVES = HUB_THREADS / KT_WAVE;
struct HubPack {
    uint2 rec[KT_WAVE];
    union {
        uint32_t bits[KT_WAVE];  // while a window is set up
        uint32_t ucnt[KT_WAVE];  // while it is walked
    };
};
constexpr uint64_t REC_BIAS = 1ull << 25;     // keeps a list's start less its blocks' ids above zero
constexpr uint32_t REC_END = (1u << 25) - 1;  // low bits of rec.y: the list's end; above them the start's high bits

constexpr uint32_t HUB_CNT = GROUP_SLOTS / 2 + 4;  // counters: 1 .. |S(x)|, |S(x)| <= 2048
constexpr uint32_t HUB_LDS = (2 * HUB_MAX + 16) + 4 * HUB_CNT + HUB_WAVES * sizeof(HubPack);
static_assert(2 * (HUB_LDS + 256) <= 160 * 1024, "two workgroups per CU");

// Eight hub-list entries at 2-byte alignment; one global_load_dwordx4.
struct __attribute__((packed, aligned(2))) Hubs8 {
    uint32_t x, y, z, w;
};

typedef __attribute__((address_space(3))) uint32_t LdsWord;
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// walk_lists over hub lists, eight entries (16 bytes) per block and lane:
// tab (byte offsets from the list entries) holds the LDS address of a set
// member's counter, zero for all others, so a lookup is one 2-byte LDS read
// and one compare, against five compares and an address of two instructions
// in a hash bucket.
__device__ __forceinline__ uint32_t walk_hub_lists(const uint16_t* __restrict__ lists, uint64_t tb, uint64_t rem,
                                                   const char* tab, HubPack& pk, uint64_t& total) {
    const uint32_t lane = lane_id();
    const uint16_t* __restrict__ T = lists - REC_BIAS;
    uint32_t mine = 0;
    total = 0;
    while (true) {
        const uint32_t len = (uint32_t)min<uint64_t>(rem, ROUND_IDS);
        const uint64_t nem = __builtin_amdgcn_ballot_w64(len != 0);
        if (nem == 0) break;
        const uint32_t nb = (len + 7) >> 3;
        const uint32_t incl = wave_scan_dpp(nb);
        const uint32_t first = incl - nb;
        const uint32_t blocks = readlane32(incl, KT_WAVE - 1);
        const uint32_t rank = rank_below(nem, 0);
        const bool bounded = len != 0 && rank != 0;
        if (len) {
            const uint64_t t0 = tb + REC_BIAS - 8ull * first;
            pk.rec[rank] = uint2{(uint32_t)t0, (len + 8 * first) | ((uint32_t)(t0 >> 32) << 25)};
        }
        for (uint32_t w0 = 0; w0 < blocks; w0 += WINDOW) {
            pk.bits[lane] = 0;
            wave_sync();
            const uint32_t at = first - 1 - w0;
            if (bounded && at < WINDOW) atomicOr(&pk.bits[at >> 5], 1u << (at & 31));
            wave_sync();
            const uint32_t bits = pk.bits[lane];
            uint32_t base = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(bounded && first <= w0));
            wave_sync();
            pk.ucnt[lane] = 0;
            wave_sync();
            const uint32_t steps = min((blocks - w0 + KT_WAVE - 1) / KT_WAVE, WINDOW / KT_WAVE);
            uint64_t ends = 0;
            uint32_t rk = 0;
            int lim = 0;
            Hubs8 q;
            // (s == steps, loaded but not probed: every lane takes the step's
            // first block, which is in list `base`, or the last block there is)
            auto load = [&](uint32_t s) {
                const bool over = s == steps;
                const int l0 = over ? 0 : (int)(2 * s);
                ends = over ? 0 : (uint64_t)readlane32(bits, l0) | ((uint64_t)readlane32(bits, l0 + 1) << 32);
                rk = rank_below(ends, base);
                base += (uint32_t)__popcll(ends);
                const uint2 r = pk.rec[rk];
                const uint32_t p = w0 + s * KT_WAVE + (over ? 0 : lane);
                lim = p < blocks ? (int)(r.y & REC_END) - (int)(8 * p) : 0;
                q = *reinterpret_cast<const Hubs8*>(
                    T + ((((uint64_t)(r.y >> 25) << 32) | r.x) + 8ull * min(p, blocks - 1)));
            };
            load(0);
            for (uint32_t s = 0; s < steps; ++s) {
                const uint32_t d[4] = {q.x, q.y, q.z, q.w};
                const uint64_t c_ends = ends;
                const uint32_t c_rk = rk;
                const int c_lim = lim;
                load(s + 1);
                uint32_t t[8];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    t[2 * k] = *reinterpret_cast<const uint16_t*>(tab + (d[k] & 0xffffu));
                    t[2 * k + 1] = *reinterpret_cast<const uint16_t*>(tab + (d[k] >> 16));
                }
                uint32_t nh = 0;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const bool hit = k < c_lim && t[k] != 0;
                    nh += hit ? 1u : 0u;
                    if (hit)
                        __hip_atomic_fetch_add(reinterpret_cast<LdsWord*>((uintptr_t)t[k]), 1u, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                if (__builtin_amdgcn_ballot_w64(nh != 0)) {
                    const uint32_t sum = wave_scan_dpp(nh);
                    total += readlane32(sum, KT_WAVE - 1);
                    const bool end = (c_ends >> lane) & 1;
                    if (end || lane == KT_WAVE - 1) atomicAdd(&pk.ucnt[c_rk], sum);
                    if (end && lane != KT_WAVE - 1) atomicSub(&pk.ucnt[c_rk + 1], sum);
                }
            }
            wave_sync();
            if (len) mine += pk.ucnt[rank];
            wave_sync();
        }
        tb += len;
        rem -= len;
    }
    return mine;
}

// Workgroup tails that are hubs, part by part: 12-wave teams, two workgroups
// per CU, each with a table of one entry per hub in dynamic LDS.  The table is
// empty between parts (the thread that set an entry clears it).  Bound by LDS
// reads (56 % busy, half of it bank conflicts) and VALU (64 %) of 24 waves a CU:
// R-MAT scale 22 4.8 to 5.0 ms (8 waves a workgroup 5.3, 16 with room for 29,696
// hubs 4.9 and 0.4 more in k_tc_main).  The last quarter of the parts comes from
// a queue: without one 9.2 ms in place of 8.4 for the whole count phase.
__global__ void __launch_bounds__(HUB_THREADS) __attribute__((amdgpu_waves_per_eu(6, 6)))
    k_tc_hub(View<true> V, TcOut out, TcParams prm, uint32_t* __restrict__ q, const uint64_t* __restrict__ plist,
             const uint16_t* __restrict__ lists, uint64_t* __restrict__ sums) {
    own_copy(out);
    extern __shared__ uint32_t hub_lds[];
    __shared__ uint64_t red[HUB_WAVES];
    __shared__ uint32_t next_u, bcast;
    const uint32_t parts = q[Q_CNT + BUCKET_HUB_PARTS];
    if (parts == 0) return;
    const uint32_t base = bucket_base(q, BUCKET_HUB_PARTS);
    uint32_t* pull = &q[Q_PULL + Q_STRIDE * BUCKET_HUB_PARTS];
    // counters first: their LDS addresses fit two bytes, and a table entry is one
    char* cnt = reinterpret_cast<char*>(hub_lds);
    char* tab = cnt + 4 * HUB_CNT;
    const uint32_t cnt0 = lds_address(cnt);
    const uint32_t tid = threadIdx.x, wave = tid / KT_WAVE, lane = lane_id();
    HubPack& pk = reinterpret_cast<HubPack*>(tab + 2 * HUB_MAX + 16)[wave];
    for (uint32_t i = tid; i < (2 * HUB_MAX + 16) / 4 + HUB_CNT; i += HUB_THREADS) hub_lds[i] = 0;
    __syncthreads();
    uint64_t my_total = 0;
    WorkStats wk(sums);
    const uint32_t fixed = parts <= 4 * gridDim.x ? parts : parts - parts / 4;
    uint32_t i = blockIdx.x;
    // the tail and bounds of the fixed share's next part, loaded a part ahead
    uint64_t xp_nx = i < parts ? plist[base + i] : 0;
    TailBounds tb_nx = part_bounds(V, (uint32_t)xp_nx, (uint32_t)(xp_nx >> 32), prm.hub_split);
    while (true) {
        if (i >= fixed) {
            if (fixed == parts) break;
            if (tid == 0)
                bcast = (__hip_atomic_load(pull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= parts - fixed)
                            ? parts
                            : fixed + atomicAdd(pull, 1u);
            __syncthreads();
            i = bcast;
            __syncthreads();
            if (i >= parts) break;
            xp_nx = plist[base + i];
            tb_nx = part_bounds(V, (uint32_t)xp_nx, (uint32_t)(xp_nx >> 32), prm.hub_split);
        }
        const uint32_t x = uniform((uint32_t)xp_nx);
        const TailBounds tb = tb_nx;
        const uint64_t sb = uniform64(tb.sb), rb = uniform64(tb.rb);
        const uint32_t ns = uniform(tb.ns), nr = uniform(tb.nr);
        const uint32_t chunk = min((uint32_t)KT_WAVE, max(1u, (nr + 2 * HUB_WAVES - 1) / (2 * HUB_WAVES)));
        uint32_t k = wave * chunk;
        uint32_t u_nx = 0, kw_nx = 0;
        if (k < nr && lane < min(chunk, nr - k)) V.entry_head(rb + k + lane, u_nx, kw_nx);
        for (uint32_t j = tid; j < ns; j += HUB_THREADS)
            *reinterpret_cast<uint16_t*>(tab + lists[sb + j]) = (uint16_t)(cnt0 + 4 * (j + 1));
        if (tid == 0) next_u = HUB_WAVES * chunk;
        const uint32_t i_nx = i + gridDim.x;
        if (i_nx < fixed) xp_nx = plist[base + i_nx];
        __syncthreads();
        uint64_t hsum = 0;
        while (k < nr) {
            const uint32_t c = min(chunk, nr - k), u = u_nx, kw = kw_nx;
            uint32_t nk = 0;
            if (lane == 0) nk = atomicAdd(&next_u, chunk);
            nk = uniform(nk);
            if (nk < nr && lane < min(chunk, nr - nk)) V.entry_head(rb + nk + lane, u_nx, kw_nx);
            uint64_t b = 0, e = 0, stl = 0;
            bool stc = false;
            if (lane < c) V.entry_bounds(rb + k + lane, u, kw, ns, b, e, stl, stc);
            const uint64_t len = e > b ? e - b : 0;
            wk.add(stl, stc ? ns : 0u, len);
            uint64_t hits;
            const uint32_t h = walk_hub_lists(lists, b, len, tab, pk, hits);
            if (h && out.per_vertex) atomic_add_u64(&out.per_vertex[u], h);
            hsum += hits;
            k = nk;
        }
        if (lane == 0) red[wave] = hsum;
        if (i_nx < fixed) tb_nx = part_bounds(V, (uint32_t)xp_nx, (uint32_t)(xp_nx >> 32), prm.hub_split);
        __syncthreads();
        for (uint32_t j = tid; j < ns; j += HUB_THREADS) {
            uint32_t* p = reinterpret_cast<uint32_t*>(cnt + 4 * (j + 1));
            const uint32_t c = *p;
            if (c) {
                if (out.per_vertex) atomic_add_u64(&out.per_vertex[V.v.sheads[sb + j]], c);
                *p = 0;
            }
            *reinterpret_cast<uint16_t*>(tab + lists[sb + j]) = 0;
        }
        if (tid == 0) {
            hsum = 0;
            for (int w = 0; w < HUB_WAVES; ++w) hsum += red[w];
            if (hsum) {
                if (out.per_vertex) atomic_add_u64(&out.per_vertex[x], hsum);
                my_total += hsum;
            }
        }
        __syncthreads();
        i = i < fixed ? i_nx : fixed;
    }
    flush_sums<HUB_WAVES>(my_total, wk, reinterpret_cast<uint64_t*>(hub_lds));
}

// Adds up the per-XCD copies of the n per-vertex counts (n == 0: none) and,
// in the first block, the workgroups' sums.
// With `host` (page-locked words) the results go there too: gate word, kept
// slots, total, work counters; then the per-vertex counts are assigned, and
// left alone when the gate is closed.
__global__ void __launch_bounds__(256) k_tc_finish(uint64_t n, const uint64_t* __restrict__ copies,
                                                   uint64_t* __restrict__ pv, uint32_t rows,
                                                   const uint64_t* __restrict__ sums, uint64_t* __restrict__ stats,
                                                   uint64_t* __restrict__ total, uint64_t* __restrict__ host,
                                                   const uint32_t* __restrict__ gate, uint32_t gate_bits,
                                                   const uint64_t* __restrict__ kept) {
    if (!host || !(*gate & gate_bits))
        for (uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (uint64_t)gridDim.x * 256) {
            uint64_t s = 0;
#pragma unroll
            for (int c = 0; c < NXCD; ++c) s += copies[c * n + v];
            if (host)
                pv[v] = s;
            else if (s)
                pv[v] += s;
        }
    if (blockIdx.x != 0) return;
    __shared__ uint64_t red[256 / KT_WAVE][SUM_WORDS];
    uint64_t t[SUM_WORDS] = {};
    for (uint32_t r = threadIdx.x; r < rows; r += 256)
#pragma unroll
        for (int k = 0; k < SUM_WORDS; ++k) t[k] += sums[(uint64_t)r * SUM_WORDS + k];
#pragma unroll
    for (int k = 0; k < SUM_WORDS; ++k) {
        const uint64_t w = wave_sum(t[k]);
        if (lane_id() == 0) red[threadIdx.x / KT_WAVE][k] = w;
    }
    __syncthreads();
    if (threadIdx.x < SUM_WORDS) {
        const uint64_t x = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
        if (threadIdx.x == SUM_TOTAL)
            *total += x;
        else
            stats[threadIdx.x] = x;
        if (host) {
            host[threadIdx.x == SUM_TOTAL ? 2 : 3 + threadIdx.x] = x;
            if (threadIdx.x == 0) {
                host[0] = *gate;
                host[1] = *kept;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Walk entries per part: tails with longer walks are split, so that a few
// long rows (an R-MAT hub's row has a large share of all entries) do not
// leave the rest of the chip waiting for the team that drew them.
struct Split {
    uint32_t wave, team, hub;
};

static Split split_rule(uint64_t entries, int num_cus) {
    const uint64_t teams = (uint64_t)num_cus * 3, waves = teams * TC_WAVES;
    auto size = [](uint64_t want, uint64_t lo, uint64_t hi) {
        uint64_t p = lo;
        while (p < want && p < hi) p <<= 1;
        return (uint32_t)p;
    };
    return {size(entries / (2 * waves), 16, 1024), size(entries / (4 * teams), 128, 4096),
            size(entries / (16 * (uint64_t)num_cus), 256, 4096)};
}

// A walk of r > split entries becomes ceil(r / split) <= 2 r / split parts.
// A hub tail is at least one part.
static uint64_t max_parts(uint64_t entries, const Split& s, bool hubs) {
    if (!entries) return 0;
    return 2 * entries / s.team + (s.wave < 1024 ? 2 * entries / s.wave : 0) +
           (hubs ? HUB_MAX + 2 * entries / s.hub : 0);
}

static uint64_t parts_of(const TcRoom& r, int num_cus) {
    return max_parts(r.entries, split_rule(r.entries, num_cus), r.hub_slots != 0);
}

// queue header, stats and sums; one u32 list of X; the part list, the
// hubs, the copies of the per-vertex counts
uint64_t tc_ws_words(uint32_t X, const TcRoom& room, int num_cus) {
    return head_words(num_cus) + (uint64_t(X) + 1) / 2 + 1 + parts_of(room, num_cus) +
           hub_ws_words(X, room.hub_slots) + NXCD * room.pv_n;
}

void tc_clear(uint64_t* ws, uint32_t X, const TcRoom& room, int num_cus, ClearList& c) {
    c.add(ws, head_words(num_cus));
    uint64_t* p = ws + head_words(num_cus) + (uint64_t(X) + 1) / 2 + 1 + parts_of(room, num_cus);
    if (room.hub_slots) c.add(p, HUB_HEAD_WORDS);
    c.add(p + hub_ws_words(X, room.hub_slots), NXCD * room.pv_n);
}

TcRoom tc_room(uint64_t entries, uint64_t slots, uint64_t pv_n) {
    TcRoom r;
    r.entries = entries;
    // below, the launches for the hubs cost what they gain (R-MAT n = 65,521 with
    // 1.8 M entries: 206 us without, 213 us with)
    if (entries >= (1ull << 22)) r.hub_slots = slots;
    // (beyond, clearing and adding up 128 bytes per vertex costs more than the
    // copies save: G(n, m) n = 5 M, 15 M pairs 1.51 ms without, 1.62 with; R-MAT
    // scale 23 with 4 and 16 pairs per vertex 4.15 and 4.44, 22.6 and 23.0)
    if (pv_n <= (1ull << 22)) r.pv_n = pv_n;
    return r;
}

uint64_t* tc_stats_ptr(uint64_t* ws) { return ws + Q_WORDS / 2; }

template <bool PLAIN>
static hipError_t launch_impl(const TcView& view, const TcOut& user_out, const TcParams& prm, uint64_t* ws, int num_cus,
                              hipStream_t st, hipEvent_t ev_begin, hipEvent_t ev_end) {
    (void)hipGetLastError();  // a status left by an earlier call is not this launch's
    View<PLAIN> V;
    V.v = view;
    TcOut out = user_out;
    // min-side walks move triangles between tails: listing launches (and
    // their per-tail counting pass) keep every triangle at its first vertex
    if (out.tri || out.tail_count) V.v.in_off = nullptr;
    uint32_t* q = reinterpret_cast<uint32_t*>(ws);
    uint64_t* stats = ws + Q_WORDS / 2;
    uint64_t* sums = stats + ST_WORDS;
    auto row = [&](int r) { return sums + (uint64_t)r * num_cus * SUM_WORDS; };
    uint32_t* list = reinterpret_cast<uint32_t*>(ws + head_words(num_cus));
    uint64_t* plist = ws + head_words(num_cus) + (uint64_t(view.X) + 1) / 2 + 1;
    if (!view.cleared) {
        TcRoom r = view.room;
        if (!user_out.per_vertex) r.pv_n = 0;
        ClearList cl;
        tc_clear(ws, view.X, r, num_cus, cl);
        clear(cl, st);
    }
    TcParams p = prm;
    if (p.wave_max_deg > WAVE_SLOTS / 2) p.wave_max_deg = WAVE_SLOTS / 2;
    if (p.group_max_deg > GROUP_SLOTS / 2) p.group_max_deg = GROUP_SLOTS / 2;
    if (p.bsearch_min_deg > BIG_SLOTS / 2) p.bsearch_min_deg = BIG_SLOTS / 2;
    // bucket edges are powers of two: round the wave threshold up to one
    uint32_t wm = 1;
    while (wm < p.wave_max_deg) wm <<= 1;
    p.wave_max_deg = wm;
    // |S| up to this is probed in an LDS table (k_tc_main or k_tc_big)
    V.v.in_hash_max = p.bsearch_min_deg;
    // parts: the workspace holds the part list of view.entries entries; a
    // listing writes whole tails
    p.wave_split = p.team_split = p.hub_split = 0xffffffffu;
    HubWs hub{};
    uint64_t* room = plist + parts_of(view.room, num_cus);
    if (view.room.entries && !out.tri && !out.tail_count) {
        const Split sp = split_rule(view.room.entries, num_cus);
        p.team_split = sp.team;
        if (sp.wave < 1024) p.wave_split = sp.wave;
        if (PLAIN && view.room.hub_slots && view.deg && view.X) {
            p.hub_split = sp.hub;
            hub = hub_ws(room, view.X);
            // few blocks: each adds up to a thousand bins to the global ones
            k_hub_hist<<<std::clamp<unsigned>(view.X / (32 * HUB_HIST_THREADS), 1, HUB_BLOCKS), HUB_HIST_THREADS, 0,
                         st>>>(view.X, view.deg, view.sym_slots ? nullptr : view.s_off, p.wave_max_deg, view.room.entries,
                               hub);
        }
    }
    room += hub_ws_words(view.X, view.room.hub_slots);
    uint64_t* const pv = user_out.per_vertex;
    if (pv && view.room.pv_n) {
        out.per_vertex = room;
        out.pv_stride = view.room.pv_n;
    }
    // a min-side walk covers in- and out-neighbours and streams from only
    // some of them: four times the entries per team grab
    if (V.v.in_off) p.team_chunk = std::min<uint32_t>(4 * std::max<uint32_t>(p.team_chunk, 1), KT_WAVE);
    if (view.X > 0) {
        const unsigned g = std::min<unsigned>((view.X + BIN_THREADS - 1) / BIN_THREADS, (unsigned)num_cus);
        if (view.X <= BIN_ONE * BIN_THREADS) {
            k_tc_bin_count<PLAIN, true><<<1, BIN_THREADS, 0, st>>>(V, p, q, hub.min_bin, row(ROW_BIN), list, plist);
        } else {
            k_tc_bin_count<PLAIN, false><<<g, BIN_THREADS, 0, st>>>(V, p, q, hub.min_bin, row(ROW_BIN), list, plist);
            k_tc_bin_fill<PLAIN><<<g, BIN_THREADS, 0, st>>>(V, p, q, hub.min_bin, list, plist);
        }
    }
    // no more workgroups than fit at once (three per CU): shares are fixed per
    // workgroup, and one that starts late would hold its share back
    const unsigned grid = (unsigned)num_cus * std::clamp<unsigned>(p.grid_per_cu, 1, 3);
    auto finish = [&]() {
        const uint64_t n = out.pv_stride;
        k_tc_finish<<<(unsigned)std::clamp<uint64_t>((n + 255) / 256, 1, 4096), 256, 0, st>>>(
            n, out.per_vertex, pv, (uint32_t)(ROWS * num_cus), sums, stats, out.totals, view.host_out, view.gate,
            view.gate_bits, view.kept);
    };
    constexpr uint32_t big_lds = 2 * BIG_SLOTS * sizeof(uint32_t);
    if constexpr (PLAIN) {
        if (out.tri) {  // listing: streamed walks only
            k_tc_huge<PLAIN, true><<<(unsigned)num_cus, TC_THREADS, 0, st>>>(V, out, p, q, list, row(ROW_HUGE));
            static const hipError_t big_list_ok =
                hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tc_big<PLAIN, true>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)big_lds);
            if (big_list_ok != hipSuccess) return big_list_ok;
            k_tc_big<PLAIN, true><<<(unsigned)num_cus, BIG_THREADS, big_lds, st>>>(V, out, p, q, list, row(ROW_BIG));
            if (ev_begin) (void)hipEventRecord(ev_begin, st);
            k_tc_main<PLAIN, true><<<grid, TC_THREADS, 0, st>>>(V, out, p, q, list, plist, row(ROW_MAIN));
            finish();
            if (ev_end) (void)hipEventRecord(ev_end, st);
            return hipGetLastError();
        }
    }
    // huge and big tails are rare: one workgroup per CU; they exit at once
    // when there are none, and are not launched where none can be
    auto longer = [&](uint64_t s) {
        return (view.sym_slots == 0 || view.sym_slots > s * s) && (view.longest == 0 || view.longest > s);
    };
    if (longer(p.bsearch_min_deg))
        k_tc_huge<PLAIN, false><<<(unsigned)num_cus, TC_THREADS, 0, st>>>(V, out, p, q, list, row(ROW_HUGE));
    if (longer(p.group_max_deg)) {
        static const hipError_t big_ok =
            hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tc_big<PLAIN, false>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)big_lds);
        if (big_ok != hipSuccess) return big_ok;
        k_tc_big<PLAIN, false><<<(unsigned)num_cus, BIG_THREADS, big_lds, st>>>(V, out, p, q, list, row(ROW_BIG));
    }
    if (ev_begin) (void)hipEventRecord(ev_begin, st);
    if constexpr (PLAIN) {
        if (hub.lists) {
            static const hipError_t hub_ok = hipFuncSetAttribute(
                reinterpret_cast<const void*>(&k_tc_hub), hipFuncAttributeMaxDynamicSharedMemorySize, (int)HUB_LDS);
            if (hub_ok != hipSuccess) return hub_ok;
            k_hub_number<<<HUB_BLOCKS, HUB_NUMBER_THREADS, 0, st>>>(view.X, view.deg, hub, q);
            k_hub_lists<<<(unsigned)std::min<uint64_t>((view.room.hub_slots + 1023) / 1024, (uint64_t)num_cus * 16), 256, 0,
                          st>>>(view.X, view.s_off, view.sheads, hub, q);
            k_tc_hub<<<2 * (unsigned)num_cus, HUB_THREADS, HUB_LDS, st>>>(V, out, p, q, plist, hub.lists, row(ROW_HUB));
        }
    }
    k_tc_main<PLAIN, false><<<grid, TC_THREADS, 0, st>>>(V, out, p, q, list, plist, row(ROW_MAIN));
    finish();
    if (ev_end) (void)hipEventRecord(ev_end, st);
    return hipGetLastError();  // a launch that did not start (e.g. LDS beyond the device's limit)
}

hipError_t tc_launch(const TcView& view, const TcOut& out, const TcParams& prm, uint64_t* ws, int num_cus,
                     hipStream_t st, hipEvent_t ev_begin, hipEvent_t ev_end) {
    const bool plain = view.s_beg == nullptr && view.r_beg == nullptr && view.rheads == nullptr &&
                       view.t_beg == nullptr && view.theads == nullptr && view.tail_id == nullptr;
    return plain ? launch_impl<true>(view, out, prm, ws, num_cus, st, ev_begin, ev_end)
                 : launch_impl<false>(view, out, prm, ws, num_cus, st, ev_begin, ev_end);
}

}  // namespace kt
