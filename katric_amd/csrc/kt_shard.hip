// One rank's shard of CeTriC ("cetric-x") / DiTriC ("patric") on one GPU.
//
// Vertex space: a combined index c over the rank's owned vertices
// [0, n_local) (c = id - from) followed by its ghosts [n_local, n_local +
// n_ghost) in ascending id order.  Sorting any list by c therefore equals the
// reference's node_ordering::id_outward(rank) (owned first, then by id,
// distributed_graph.h:102-112), and the ghost part of a list is its suffix.
//
// Preprocessing (lists placed by rank and sorted one by one):
//   every owned slot (v, u) with c = map(u) contributes
//     (v, c)  if (deg v, v) < (deg u, u)           -- N+(v), global degrees
//     (c, v)  if not, c is a ghost and cetric-x     -- ghost_adj(c)
//   (remove_in_edges_and_expand_ghosts, distributed_graph.h:1057-1169, with
//   node_ordering::degree on exchanged ghost degrees, :113-146), and the sorted
//   lists form a CSR L over the combined space.
// Local phase (same intersection kernel as the plain path):
//   cetric-x: every tail x (owned or ghost), S = R = L(x), T(u) = L(u)
//             (run_local_sequential_with_ghosts, cetric_edge_iterator.h:300-388);
//   patric:   owned tails, S = L(v), R = owned part of L(v), T(u) = L(u)
//             (run_local_sequential with ghost heads skipped, :229-298).
// Contracted / distributed phase: message i = [a, list]; its entries split
// into owned receivers R and ghosts G (entries unknown to this rank can match
// nothing).  cetric-x: S = G, T(u) = N+cut(u) = ghost suffix of L(u)
// (contraction, distributed_graph.h:679-764, then intersect_from_message,
// cetric_edge_iterator.h:1797-1889); patric: S = R ++ G, T(u) = L(u).  Every
// hit w emits Triangle{a, u, w}.
#include <algorithm>

#include "../../include/katric_shard.h"
#include "kt_ctx.h"
#include "kt_device.h"

namespace kt {

constexpr int SH_THREADS = 256;
constexpr int SH_ITEMS = 16;
constexpr int SH_TILE = SH_THREADS * SH_ITEMS;

// Global id -> combined index (0xffffffff: unknown to this rank).  Ghosts are
// ranked in a bitmap over all global ids: rs[w] = {ghost bits of ids 32w ..
// 32w+31, ghosts below 32w}, so a lookup is one 8-byte gather and a popcount
// (n_all / 4 bytes in all, a table the caches hold far better than one index
// per id).
struct ShardMap {
    uint32_t from, to, nl, ng;
    const uint32_t* ghost_ids;
    const uint2* rs;
    uint32_t n_all;
    __device__ __forceinline__ uint32_t map(uint32_t u) const {
        if (u >= from && u < to) return u - from;
        if (u >= n_all) return 0xffffffffu;
        const uint2 e = rs[u >> 5];
        const uint32_t bit = 1u << (u & 31);
        // (the bound matters for a table that fails its check only)
        return (e.x & bit) ? nl + min(e.y + (uint32_t)__popc(e.x & (bit - 1)), ng - 1) : 0xffffffffu;
    }
    __device__ __forceinline__ uint32_t gid(uint32_t c) const { return c < nl ? from + c : ghost_ids[c - nl]; }
};

// One pass over the combined index space and the messages: degrees, the ghosts'
// rank-select table, the row bounds of the slot and message-entry tiles, and the
// checks of both offset arrays and of the ghost table.
//
// Ghost ids ascend, so the first ghost of a table word owns it: it reads the up
// to 31 ids after its own, and its index is the word's prefix.  Words without a
// ghost stay zero.  (The bits were set by atomics and counted, scanned and
// spread by six more launches, 37 us for 246,000 ghosts among 2^20 ids in the
// CeTriC shard of an R-MAT graph; this one takes 8 with all it does.)  Only
// strictly ascending ids are taken, so every index below is in range.
__global__ void k_shard_prepare(ShardMap M, uint64_t nnz, const uint64_t* __restrict__ off,
                                const uint64_t* __restrict__ ghost_degree, uint32_t* __restrict__ deg,
                                uint32_t* __restrict__ tbnd, uint2* __restrict__ rs, uint32_t nmsg, uint64_t mtot,
                                const uint64_t* __restrict__ moff, uint32_t* __restrict__ mbnd,
                                uint32_t* __restrict__ err) {
    const uint64_t X = (uint64_t)M.nl + M.ng, all = max(X, (uint64_t)nmsg);
    for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < all; c += (uint64_t)gridDim.x * blockDim.x) {
        if (c == 0) atomicOr(err, (off[0] != 0 || off[M.nl] != nnz) ? KT_ERR_OFFSETS | KT_FLAG_UNSORTED : KT_FLAG_UNSORTED);
        if (c < M.nl) {
            uint64_t a = off[c], b = off[c + 1];
            if (b < a || b - a > 0xffffffffull) {
                atomicOr(err, KT_ERR_OFFSETS);
                deg[c] = 0;
            } else {
                deg[c] = (uint32_t)(b - a);
                note_tiles((uint32_t)c, a, b, nnz, SH_TILE, tbnd);
            }
        } else if (c < X) {
            const uint32_t g = (uint32_t)(c - M.nl);
            const uint32_t id = M.ghost_ids[g];
            const uint32_t prev = g > 0 ? M.ghost_ids[g - 1] : 0u;
            if ((id >= M.from && id < M.to) || (g > 0 && prev >= id) || id >= M.n_all) atomicOr(err, KT_ERR_GHOST);
            uint64_t d = ghost_degree[g];
            deg[c] = d > 0xffffffffull ? 0xffffffffu : (uint32_t)d;
            if (id < M.n_all && (g == 0 || (prev >> 5) != (id >> 5))) {
                uint32_t bits = 1u << (id & 31), last = id;
                bool in = true;
#pragma unroll
                for (uint32_t j = 1; j < 32; ++j) {
                    const uint32_t x = M.ghost_ids[min((uint64_t)g + j, (uint64_t)M.ng - 1)];
                    in = in && x > last && (x >> 5) == (id >> 5);
                    bits |= in ? 1u << (x & 31) : 0u;
                    last = x;
                }
                rs[id >> 5] = make_uint2(bits, g);
            }
        }
        if (c < nmsg) {
            const uint64_t a = moff[c], b = moff[c + 1];
            if (b < a || b > mtot)
                atomicOr(err, KT_ERR_MESSAGE);
            else
                note_tiles((uint32_t)c, c ? a : 0, b, mtot, SH_TILE, mbnd);  // (entries before the first message: row 0)
        }
    }
}

__device__ __forceinline__ bool c_less(const ShardMap& M, const uint32_t* deg, uint32_t a, uint32_t b) {
    const uint32_t da = deg[a], db = deg[b];
    return da < db || (da == db && M.gid(a) < M.gid(b));
}

// Owned slots -> (tail, head) keys of N+ lists and (cetric-x) ghost lists,
// appended in any order, each with its rank among its tail's entries; the
// tails' counts are left in cnt (zeroed by the caller).  Every wave counts its
// keys over the tile's 16 slot rounds, and one atomic per workgroup reserves
// the workgroup's output range.  The ranks come from the counts' atomics: a
// run of a wave's slots with one owned tail takes one, a ghost list's entry its
// own (few per ghost: an entry's owned head follows the ghost in degree order).
// All of a thread's atomics are in flight together.
__global__ void __launch_bounds__(SH_THREADS)
    k_shard_entries(ShardMap M, uint64_t nnz, const uint64_t* __restrict__ off, const uint32_t* __restrict__ tbnd,
                    const uint32_t* __restrict__ heads, const uint32_t* __restrict__ deg, int bits, int ghost_lists,
                    uint64_t* __restrict__ keys, uint32_t* __restrict__ rank, uint64_t* __restrict__ cnt,
                    uint64_t* __restrict__ nkeys, uint32_t* __restrict__ err) {
    constexpr int NW = SH_THREADS / KT_WAVE;
    __shared__ uint32_t marks[SH_TILE];
    __shared__ uint32_t wmax[NW];
    __shared__ uint32_t bnd[2];
    __shared__ uint32_t wtot[NW];
    __shared__ uint64_t bbase;
    const uint64_t tile0 = (uint64_t)blockIdx.x * SH_TILE;
    const uint64_t tend = min(tile0 + SH_TILE, nnz);
    uint32_t lo, hi;
    tile_rows<SH_THREADS, SH_ITEMS>(off, M.nl, tile0, tend, marks, bnd, wmax, lo, hi, tbnd, err);
    const unsigned tid = threadIdx.x, wave = tid / KT_WAVE;
    uint32_t cs[SH_ITEMS];
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint64_t sl = tile0 + k * SH_THREADS + tid;
        cs[k] = sl < tend ? M.map(heads[sl]) : 0u;
    }
    uint32_t flags = 0, count = 0;
    uint64_t pm[SH_ITEMS], om[SH_ITEMS];
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const unsigned i = k * SH_THREADS + tid;
        bool out_e = false, in_e = false;
        const uint32_t v = lo + marks[i], c = cs[k];
        if (tile0 + i < tend) {
            if (c == 0xffffffffu) {
                flags |= KT_ERR_GHOST;
            } else if (c == v) {
                flags |= KT_ERR_SELF_LOOP;
            } else {
                out_e = c_less(M, deg, v, c);
                in_e = ghost_lists && !out_e && c >= M.nl;
            }
        }
        om[k] = __ballot(out_e);
        pm[k] = om[k] | __ballot(in_e);
        count += (uint32_t)__popcll(pm[k]);
    }
    // this lane's entries of round k: the owned ones before it in its row's run
    const uint64_t lt = lanemask_lt(), me = 1ull << lane_id();
    uint32_t base[SH_ITEMS];
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint32_t m = marks[k * SH_THREADS + tid], mp = __shfl_up(m, 1, 64);
        const uint64_t starts = __ballot(lane_id() == 0 || m != mp);
        const int s = 63 - __clzll((long long)(starts & (lt | me)));
        const uint64_t after = starts & ~(lt | me);
        const uint64_t run = om[k] & (~0ull << s) & (after ? (after & -after) - 1 : ~0ull);
        const bool own = (om[k] & me) != 0;
        const int lead = run ? __ffsll((unsigned long long)run) - 1 : 0;
        uint32_t got = 0;
        if ((pm[k] & me) && (!own || lead == (int)lane_id()))
            got = (uint32_t)atomic_add_u64(&cnt[own ? lo + m : cs[k]], own ? (uint64_t)__popcll(run) : 1ull);
        base[k] = __shfl(got, own ? lead : (int)lane_id(), 64) + (own ? (uint32_t)__popcll(run & lt) : 0u);
        if (pm[k] & me) flags |= (base[k] >= segsort_wave_len() ? KT_FLAG_OVER_WAVE : 0u) |
                                 (base[k] >= segsort_max_len() ? KT_FLAG_OVER_GROUP : 0u);
    }
    or_flags(err, flags);
    if (lane_id() == 0) wtot[wave] = count;
    __syncthreads();
    if (tid == 0) {
        uint64_t t = 0;
        for (int w = 0; w < NW; ++w) t += wtot[w];
        bbase = t ? atomic_add_u64(nkeys, t) : 0;
    }
    __syncthreads();
    uint64_t at = bbase;
    for (unsigned w = 0; w < wave; ++w) at += wtot[w];
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        if (pm[k] & me) {
            const uint64_t v = lo + marks[k * SH_THREADS + tid], c = cs[k], p = at + __popcll(pm[k] & lt);
            keys[p] = (om[k] & me) ? (v << bits) | c : (c << bits) | v;
            rank[p] = base[k];
        }
        at += __popcll(pm[k]);
    }
}

// Every entry to its rank's place in its tail's list.
__global__ void k_shard_place(uint64_t M, int bits, const uint64_t* __restrict__ keys,
                              const uint32_t* __restrict__ rank, const uint64_t* __restrict__ coff,
                              uint32_t* __restrict__ cheads) {
    const uint64_t mask = (1ull << bits) - 1;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < M; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t k = keys[i];
        cheads[coff[k >> bits] + rank[i]] = (uint32_t)(k & mask);
    }
}

// Sorted keys -> heads of the CSR (lists above the segmented sort's longest).
__global__ void k_keys_csr(uint64_t M, int bits, const uint64_t* __restrict__ keys, uint32_t* __restrict__ cheads,
                           uint32_t* __restrict__ err) {
    const uint64_t mask = (1ull << bits) - 1;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < M; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t k = keys[i];
        cheads[i] = (uint32_t)(k & mask);
        if (i > 0 && keys[i - 1] == k) atomicOr(err, KT_ERR_DUPLICATE);
    }
}

// First position of a ghost head (combined index >= nl) in each owned list.
__global__ void k_cut_begin(uint32_t nl, const uint64_t* __restrict__ coff, const uint32_t* __restrict__ cheads,
                            uint64_t* __restrict__ cut) {
    uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nl) return;
    uint64_t lo = coff[u], hi = coff[u + 1];
    while (lo < hi) {
        uint64_t mid = (lo + hi) >> 1;
        if (cheads[mid] < nl)
            lo = mid + 1;
        else
            hi = mid;
    }
    cut[u] = lo;
}

// Messages are taken as one flat run of entries, in tiles of SH_TILE: with O(p)
// and G(p) the owned and the ghost entries before entry p, and b, e a message's
// first entry and its end, an owned entry p goes to O(p) + G(b), a ghost entry
// to O(e) + G(p) -- the message's owned entries, then its ghosts, each in
// message order.  A count pass gives every 64 entries' bits and every tile's
// totals; a thread per message then ranks its b and e, and a write pass places
// the entries.  Short and long messages take the same time (8 lanes per message
// took 126 + 44 us for the 241,000 messages, 12 M ids, of an R-MAT CeTriC shard, the
// three passes take 111 + 8 + 34, the first at the rate of its gathers; 63 + 29 and
// 44 + 5 + 19 us for 6 M ids of a DiTriC shard).
struct MsgWord {
    uint64_t own, ghost;      // entry classes of 64 entries
    uint32_t pre_own, pre_ghost;  // those of the tile's words before
};

// No pass of the messages runs on offsets that fail their check, and none needs
// to where an entry was found bad.  Block-wide.
__device__ __forceinline__ bool messages_bad(const uint32_t* err, uint32_t* word) {
    if (threadIdx.x == 0) *word = *err;
    __syncthreads();
    return (*word & KT_ERR_MASK) != 0;
}

// Combined index of every entry (to mapped; entries of no message are unknown),
// order of the messages, and the entry classes.
__global__ void __launch_bounds__(SH_THREADS)
    k_msg_map(ShardMap M, uint32_t nmsg, uint64_t mtot, const uint64_t* __restrict__ moff,
              const uint32_t* __restrict__ mbnd, const uint32_t* __restrict__ mheads, uint32_t* __restrict__ mapped,
              MsgWord* __restrict__ words, uint64_t* __restrict__ tcnt, uint32_t* __restrict__ err) {
    constexpr int NW = SH_THREADS / KT_WAVE;
    static_assert(SH_ITEMS * NW == KT_WAVE, "a lane per word of a tile");
    __shared__ uint32_t marks[SH_TILE];
    __shared__ uint32_t wmax[NW];
    __shared__ uint32_t bnd[2];
    __shared__ uint64_t wo[KT_WAVE], wg[KT_WAVE];
    if (messages_bad(err, bnd)) return;
    const uint64_t tile0 = (uint64_t)blockIdx.x * SH_TILE;
    const uint64_t tend = min(tile0 + SH_TILE, mtot);
    uint32_t lo, hi;
    __syncthreads();  // bnd has been read
    tile_rows<SH_THREADS, SH_ITEMS>(moff, nmsg, tile0, tend, marks, bnd, wmax, lo, hi, mbnd);
    const uint64_t first = moff[0];
    const unsigned tid = threadIdx.x, wave = tid / KT_WAVE;
    uint32_t x[SH_ITEMS], nx[SH_ITEMS], c[SH_ITEMS];
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint64_t p = tile0 + k * SH_THREADS + tid;
        x[k] = p < tend ? mheads[p] : 0u;
        nx[k] = p + 1 < mtot ? mheads[p + 1] : 0xffffffffu;
    }
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint64_t p = tile0 + k * SH_THREADS + tid;
        c[k] = p < tend && p >= first ? M.map(x[k]) : 0xffffffffu;
    }
    uint32_t flags = 0;
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint32_t i = k * SH_THREADS + tid;
        const uint64_t p = tile0 + i;
        if (p < tend) {
            mapped[p] = c[k];
            const bool same = i + 1 < SH_TILE ? p + 1 < tend && marks[i + 1 < SH_TILE ? i + 1 : i] == marks[i]
                                              : p + 1 < moff[(uint64_t)lo + marks[i] + 1];
            if (p >= first && same && nx[k] <= x[k]) flags |= KT_ERR_MESSAGE;
        }
        const uint64_t ob = __ballot(c[k] < M.nl), gb = __ballot(c[k] != 0xffffffffu && c[k] >= M.nl);
        if (lane_id() == 0) {
            wo[k * NW + wave] = ob;
            wg[k * NW + wave] = gb;
        }
    }
    or_flags(err, flags);
    __syncthreads();
    if (wave != 0) return;
    MsgWord w{wo[tid], wg[tid], 0, 0};
    const uint64_t n = (uint64_t)__popcll(w.own) << 32 | (uint32_t)__popcll(w.ghost);
    const uint64_t incl = wave_incl_sum(n);
    w.pre_own = (uint32_t)((incl - n) >> 32);
    w.pre_ghost = (uint32_t)(incl - n);
    if (tile0 + tid * 64 < tend) words[tile0 / 64 + tid] = w;
    if (tid == KT_WAVE - 1) {
        tcnt[blockIdx.x] = incl >> 32;
        tcnt[gridDim.x + blockIdx.x] = (uint32_t)incl;
    }
}

// Owned and ghost entries before entry p; toff: scan of the tiles' owned, then
// ghost counts.
__device__ __forceinline__ void msg_ranks(uint64_t p, uint64_t mtot, uint64_t tiles, const MsgWord* __restrict__ words,
                                          const uint64_t* __restrict__ toff, uint64_t& own, uint64_t& ghost) {
    const uint64_t t = min(p / SH_TILE, tiles);
    own = toff[t];
    ghost = toff[tiles + t] - toff[tiles];
    if (p >= mtot) {
        own = toff[tiles];
        ghost = toff[2 * tiles] - toff[tiles];
        return;
    }
    const MsgWord w = words[p / 64];
    const uint64_t lt = (1ull << (p & 63)) - 1;
    own += w.pre_own + (uint32_t)__popcll(w.own & lt);
    ghost += w.pre_ghost + (uint32_t)__popcll(w.ghost & lt);
}

// Per message: its list in the output, the list's first ghost, the ghosts
// before it, and its sender's combined index.
__global__ void k_msg_place(ShardMap M, uint32_t nmsg, uint64_t mtot, uint64_t tiles, const uint32_t* __restrict__ src,
                            const uint64_t* __restrict__ moff, const MsgWord* __restrict__ words,
                            const uint64_t* __restrict__ toff, uint64_t* __restrict__ out_off,
                            uint64_t* __restrict__ split, uint64_t* __restrict__ gbeg, uint32_t* __restrict__ tail_id,
                            uint32_t* __restrict__ err) {
    if (*err & KT_ERR_MASK) return;
    uint32_t flags = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nmsg; i += gridDim.x * blockDim.x) {
        uint64_t o0, g0, o1, g1;
        msg_ranks(moff[i], mtot, tiles, words, toff, o0, g0);
        msg_ranks(moff[i + 1], mtot, tiles, words, toff, o1, g1);
        const uint32_t a = M.map(src[i]);
        if (a == 0xffffffffu || a < M.nl) flags |= KT_ERR_MESSAGE;
        if (o1 + g1 - o0 - g0 > segsort_wave_len()) flags |= KT_FLAG_LONG_MESSAGE;
        tail_id[i] = (a == 0xffffffffu) ? 0u : a;
        out_off[i] = o0 + g0;
        split[i] = o1 + g0;
        gbeg[i] = g0;
        if (i + 1 == nmsg) out_off[nmsg] = o1 + g1;
    }
    or_flags(err, flags);
}

__global__ void __launch_bounds__(SH_THREADS)
    k_msg_write(uint32_t nl, uint32_t nmsg, uint64_t mtot, const uint64_t* __restrict__ moff,
                const uint32_t* __restrict__ mbnd, const uint32_t* __restrict__ mapped,
                const uint64_t* __restrict__ toff, uint64_t tiles, const uint64_t* __restrict__ split,
                const uint64_t* __restrict__ gbeg, uint32_t* __restrict__ out, const uint32_t* __restrict__ err) {
    constexpr int NW = SH_THREADS / KT_WAVE;
    __shared__ uint32_t marks[SH_TILE];
    __shared__ uint32_t wmax[NW];
    __shared__ uint32_t bnd[2];
    __shared__ uint32_t pre[KT_WAVE];  // owned << 16 | ghost entries of the tile's words before
    if (messages_bad(err, bnd)) return;
    const uint64_t tile0 = (uint64_t)blockIdx.x * SH_TILE;
    const uint64_t tend = min(tile0 + SH_TILE, mtot);
    uint32_t lo, hi;
    __syncthreads();  // bnd has been read
    tile_rows<SH_THREADS, SH_ITEMS>(moff, nmsg, tile0, tend, marks, bnd, wmax, lo, hi, mbnd);
    const unsigned tid = threadIdx.x, wave = tid / KT_WAVE;
    uint32_t c[SH_ITEMS];
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint64_t p = tile0 + k * SH_THREADS + tid;
        c[k] = p < tend ? mapped[p] : 0xffffffffu;
    }
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const uint32_t o = (uint32_t)__popcll(__ballot(c[k] < nl));
        const uint32_t known = (uint32_t)__popcll(__ballot(c[k] != 0xffffffffu));
        if (lane_id() == 0) pre[k * NW + wave] = o << 16 | (known - o);
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t n = pre[tid];
        pre[tid] = wave_incl_sum(n) - n;
    }
    __syncthreads();
    const uint64_t obase = toff[blockIdx.x], gbase = toff[tiles + blockIdx.x] - toff[tiles], lt = lanemask_lt();
#pragma unroll
    for (int k = 0; k < SH_ITEMS; ++k) {
        const bool own = c[k] < nl, known = c[k] != 0xffffffffu;
        const uint64_t ob = __ballot(own), gb = __ballot(known) & ~ob;
        const uint32_t w = pre[k * NW + wave], i = lo + marks[k * SH_THREADS + tid];
        if (!known) continue;
        const uint64_t g0 = gbeg[i];
        const uint64_t p = own ? obase + (w >> 16) + (uint32_t)__popcll(ob & lt) + g0
                               : gbase + (w & 0xffffu) + (uint32_t)__popcll(gb & lt) + split[i] - g0;
        out[p] = c[k];
    }
}

}  // namespace kt

using namespace kt;

namespace {

int bits_for(uint64_t x) {
    int b = 0;
    while (b < 64 && (x >> b)) ++b;
    return b;
}

struct ShardBufs {
    uint64_t* small;
    const uint64_t* off;
    const uint32_t* heads;
    const uint32_t* ghost_ids;
    const uint64_t* ghost_degree;
    const uint32_t* msg_src;
    const uint64_t* msg_off;
    const uint32_t* msg_heads;
    uint32_t* deg;
    uint64_t* keys;
    uint64_t* alt;
    uint64_t* radix_tmp;
    uint64_t* coff;
    uint32_t* cheads;
    uint64_t* cut;
    uint64_t* mgbeg;
    uint64_t* moff;
    uint64_t* mtoff;
    uint32_t* mbnd;
    uint32_t* mtail;
    uint64_t* msplit;
    uint32_t* mheads2;
    uint32_t* mmapped;
    uint64_t* scan_tmp;
    uint64_t* tc_ws;
    uint64_t* pv;
    uint2* rs;
    uint32_t* tbnd;
    TcRoom room;
};


uint64_t shard_layout(void* base, const kt_shard_in* in, uint64_t nnz, uint64_t mtot, int num_cus, bool host_in,
                      bool want_pv, bool pv_dev, bool rich, ShardBufs& B) {
    Carver cv{base, 0};
    const uint64_t nloc = in->range_bounds[in->rank + 1] - in->range_bounds[in->rank];
    const uint64_t X = nloc + in->n_ghost;
    B.small = static_cast<uint64_t*>(cv.take(64 * 8));
    if (host_in) {
        B.off = static_cast<uint64_t*>(cv.take((nloc + 1) * 8));
        B.heads = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(nnz, 1) * 4));
        B.ghost_ids = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(in->n_ghost, 1) * 4));
        B.ghost_degree = static_cast<uint64_t*>(cv.take(std::max<uint64_t>(in->n_ghost, 1) * 8));
        B.msg_src = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(in->n_msg, 1) * 4));
        B.msg_off = static_cast<uint64_t*>(cv.take(((uint64_t)in->n_msg + 1) * 8));
        B.msg_heads = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(mtot, 1) * 4));
    }
    B.deg = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(X, 1) * 4));
    B.keys = static_cast<uint64_t*>(cv.take(std::max<uint64_t>(nnz, 1) * 8));
    B.alt = static_cast<uint64_t*>(cv.take(std::max<uint64_t>(nnz, 1) * 8));
    B.radix_tmp = static_cast<uint64_t*>(cv.take(radix_tmp_words(nnz) * 8));
    B.coff = static_cast<uint64_t*>(cv.take((X + 1) * 8));
    B.cheads = static_cast<uint32_t*>(cv.take((nnz + 4) * 4));
    B.cut = static_cast<uint64_t*>(cv.take(std::max<uint64_t>(nloc, 1) * 8));
    const uint64_t mtiles = (mtot + SH_TILE - 1) / SH_TILE;
    B.mgbeg = static_cast<uint64_t*>(cv.take(std::max<uint64_t>(in->n_msg, 1) * 8));
    B.moff = static_cast<uint64_t*>(cv.take(((uint64_t)in->n_msg + 1) * 8));
    B.mtoff = static_cast<uint64_t*>(cv.take((2 * mtiles + 1) * 8));
    B.mbnd = static_cast<uint32_t*>(cv.take((2 * mtiles + 1) * 4));
    B.mtail = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(in->n_msg, 1) * 4));
    B.msplit = static_cast<uint64_t*>(cv.take(std::max<uint64_t>(in->n_msg, 1) * 8));
    // (the entry classes sit here until the entries are written)
    static_assert(sizeof(MsgWord) <= 64 * sizeof(uint32_t), "words fit the entries' room");
    B.mheads2 = static_cast<uint32_t*>(cv.take(std::max((mtot + 4) * 4, (mtot + 63) / 64 * sizeof(MsgWord))));
    B.mmapped = static_cast<uint32_t*>(cv.take(std::max<uint64_t>(mtot, 1) * 4));
    const uint64_t n_all = in->range_bounds[in->num_ranks];
    const uint64_t rs_words = (n_all + 31) / 32;
    B.scan_tmp = static_cast<uint64_t*>(
        cv.take(scan_tmp_words(std::max<uint64_t>(X, 2 * mtiles) + 1) * 8));
    // both phases use it: the list of the larger set of tails, the parts of the longer walk
    B.room = rich ? tc_room(std::max(nnz, mtot), 0, want_pv ? X : 0) : TcRoom{};
    // hub lists for CeTriC's local phase, a plain view with at most nnz entries
    // (scale 21 / 2 ranks: count 6.6 ms without, 5.7 with)
    if (rich && in->algorithm == KT_SHARD_CETRIC) B.room.hub_slots = tc_room(nnz, nnz, 0).hub_slots;
    B.tc_ws = static_cast<uint64_t*>(
        cv.take(tc_ws_words((uint32_t)std::max<uint64_t>(X, in->n_msg), B.room, num_cus) * 8));
    B.pv = pv_dev ? static_cast<uint64_t*>(cv.take(std::max<uint64_t>(X, 1) * 8)) : nullptr;
    B.rs = static_cast<uint2*>(cv.take((rs_words + 1) * 8));
    B.tbnd = static_cast<uint32_t*>(cv.take((2 * ((nnz + SH_TILE - 1) / SH_TILE) + 1) * 4));
    return cv.used;
}

}  // namespace

// The body of kt_count_shard; the caller holds c->mu and has begun the call.
int kt::count_shard_locked(kt_ctx* c, const kt_shard_in* in, kt_shard_out* out, const ShardSizes* sizes) {
    int rc = KT_OK;
    if (!in || !out || !in->range_bounds || !in->offsets || in->num_ranks == 0 || in->rank >= in->num_ranks ||
        in->algorithm > KT_SHARD_DITRIC)
        return c->fail(KT_EINVAL, "bad shard arguments");
    // with pseudo2core the reference's senders also drop skipped interface
    // nodes from the distributed phase (cetric_edge_iterator.h:1247-1271),
    // and the messages are this call's inputs: not supported on shards
    if (c->prm.pseudo2core) return c->fail(KT_EINVAL, "pseudo2core applies to the shared-memory path only");
    const uint32_t P = in->num_ranks;
    const uint64_t* bd = in->range_bounds;
    if (bd[0] != 0) return c->fail(KT_EINVAL, "range_bounds[0] != 0");
    for (uint32_t r = 0; r < P; ++r)
        if (bd[r + 1] < bd[r] || bd[r + 1] > 0xffffffffull) return c->fail(KT_EINVAL, "range bounds not ascending");
    const uint32_t from = (uint32_t)bd[in->rank], to = (uint32_t)bd[in->rank + 1];
    const uint32_t nl = to - from, ng = in->n_ghost;
    const uint64_t X = (uint64_t)nl + ng;
    if (X >= 0xffffffffull) return c->fail(KT_EINVAL, "shard too large");
    out->local_triangles = out->type3_triangles = 0;
    const bool host_in = !(in->flags & KT_DEVICE_INPUT);
    const bool want_pv = out->per_vertex != nullptr;
    const bool pv_dev = want_pv && (in->flags & KT_DEVICE_OUTPUT);
    if (nl == 0 && ng == 0) return KT_OK;
    // sizes (read by a kernel from device arrays)
    if (in->n_msg && (!in->msg_src || !in->msg_offsets)) return c->fail(KT_EINVAL, "null shard array");
    uint64_t nnz = 0, mtot = 0;
    if (host_in) {
        if (in->offsets[0] != 0) return c->fail(KT_EINVAL, "offsets[0] != 0");
        nnz = in->offsets[nl];
        mtot = in->n_msg ? in->msg_offsets[in->n_msg] : 0;
        if (in->n_msg && in->msg_offsets[0] != 0) return c->fail(KT_EINVAL, "msg_offsets[0] != 0");
    } else {
        if (sizes) {
            nnz = sizes->slots;
            mtot = sizes->entries;
        } else {
            const uint64_t* at[2] = {in->offsets + nl, in->n_msg ? in->msg_offsets + in->n_msg : in->offsets + nl};
            uint64_t got[2];
            rc = c->read_words(at, 2, got, "D2H shard sizes");
            if (rc) return rc;
            nnz = got[0];
            mtot = in->n_msg ? got[1] : 0;
        }
    }
    if ((nnz && !in->heads) || (ng && (!in->ghost_ids || !in->ghost_degree)) ||
        (mtot && !in->msg_heads))
        return c->fail(KT_EINVAL, "null shard array");
    ShardBufs B;
    // the intersection's optional room is left out where only it does not fit
    bool rich = true;
    rc = c->reserve(shard_layout(nullptr, in, nnz, mtot, c->num_cus, host_in, want_pv, want_pv && !pv_dev, rich, B));
    if (rc == KT_ENOMEM) {
        rich = false;
        rc = c->reserve(shard_layout(nullptr, in, nnz, mtot, c->num_cus, host_in, want_pv, want_pv && !pv_dev, rich, B));
    }
    if (rc) return rc;
    shard_layout(c->arena, in, nnz, mtot, c->num_cus, host_in, want_pv, want_pv && !pv_dev, rich, B);
    hipStream_t st = c->stream;
    (void)hipEventRecord(c->ev[EV_START], st);
    if (host_in) {
        struct {
            const void* dst;
            const void* src;
            uint64_t bytes;
        } up[] = {{B.off, in->offsets, ((uint64_t)nl + 1) * 8},
                  {B.heads, in->heads, nnz * 4},
                  {B.ghost_ids, in->ghost_ids, (uint64_t)ng * 4},
                  {B.ghost_degree, in->ghost_degree, (uint64_t)ng * 8},
                  {B.msg_src, in->msg_src, (uint64_t)in->n_msg * 4},
                  {B.msg_off, in->msg_offsets, in->n_msg ? ((uint64_t)in->n_msg + 1) * 8 : 0},
                  {B.msg_heads, in->msg_heads, mtot * 4}};
        for (auto& u : up) {
            if (!u.bytes) continue;
            rc = c->hip_check(hipMemcpyAsync(const_cast<void*>(u.dst), u.src, u.bytes, hipMemcpyHostToDevice, st),
                              "H2D shard");
            if (rc) return rc;
        }
    } else {
        B.off = in->offsets;
        B.heads = in->heads;
        B.ghost_ids = in->ghost_ids;
        B.ghost_degree = in->ghost_degree;
        B.msg_src = in->msg_src;
        B.msg_off = in->msg_offsets;
        B.msg_heads = in->msg_heads;
    }
    (void)hipEventRecord(c->ev[EV_H2D], st);
    uint32_t* err = reinterpret_cast<uint32_t*>(B.small);
    uint64_t* nkeys = B.small + 1;
    const uint64_t n_all = bd[P];
    ShardMap M{from, to, nl, ng, B.ghost_ids, B.rs, (uint32_t)std::min<uint64_t>(n_all, 0xffffffffull)};
    {
        ClearList cl;
        cl.add(B.small, 64);
        cl.add(reinterpret_cast<uint64_t*>(B.rs), (n_all + 31) / 32);
        cl.add(B.coff, X + 1);
        clear(cl, st);
    }
    const int bits = std::max(1, bits_for(X));  // X itself is never a valid index: keys stay below 2^(2 bits)
    const bool cetric = in->algorithm == KT_SHARD_CETRIC;
    const uint64_t both = std::max<uint64_t>(X, in->n_msg);
    k_shard_prepare<<<(unsigned)std::min<uint64_t>((both + 255) / 256, 8192), 256, 0, st>>>(
        M, nnz, B.off, B.ghost_degree, B.deg, B.tbnd, B.rs, in->n_msg, mtot, B.msg_off, B.mbnd, err);
    const uint64_t tiles = (nnz + SH_TILE - 1) / SH_TILE;
    uint32_t* rank = reinterpret_cast<uint32_t*>(B.alt);
    if (tiles && nl)
        k_shard_entries<<<(unsigned)tiles, SH_THREADS, 0, st>>>(M, nnz, B.off, B.tbnd, B.heads, B.deg, bits,
                                                                cetric ? 1 : 0, B.keys, rank, B.coff, nkeys, err);
    // messages (on a malformed shard the later passes do nothing)
    if (in->n_msg) {
        const uint64_t mt = (mtot + SH_TILE - 1) / SH_TILE;
        MsgWord* words = reinterpret_cast<MsgWord*>(B.mheads2);
        if (mt)
            k_msg_map<<<(unsigned)mt, SH_THREADS, 0, st>>>(M, in->n_msg, mtot, B.msg_off, B.mbnd, B.msg_heads,
                                                           B.mmapped, words, B.mtoff, err);
        scan_u64(B.mtoff, B.mtoff, 2 * mt, B.scan_tmp, st);
        k_msg_place<<<(unsigned)std::min<uint64_t>(((uint64_t)in->n_msg + 255) / 256, 8192), 256, 0, st>>>(
            M, in->n_msg, mtot, mt, B.msg_src, B.msg_off, words, B.mtoff, B.moff, B.msplit, B.mgbeg, B.mtail, err);
        if (mt)
            k_msg_write<<<(unsigned)mt, SH_THREADS, 0, st>>>(nl, in->n_msg, mtot, B.msg_off, B.mbnd, B.mmapped,
                                                             B.mtoff, mt, B.msplit, B.mgbeg, B.mheads2, err);
    }
    rc = c->hip_check(hipMemcpyAsync(c->host_small, B.small, 16, hipMemcpyDeviceToHost, st), "D2H flags");
    if (rc) return rc;
    rc = c->hip_check(hipStreamSynchronize(st), "shard entries");
    if (rc) return rc;
    uint32_t flags = (uint32_t)c->host_small[0];
    const uint64_t Mk = c->host_small[1];
    if (flags & KT_ERR_MASK)
        return c->fail(KT_EINVAL, "malformed shard:%s%s%s%s%s", (flags & KT_ERR_OFFSETS) ? " bad offsets" : "",
                       (flags & KT_ERR_GHOST) ? " ghost table" : "", (flags & KT_ERR_SELF_LOOP) ? " self-loop" : "",
                       (flags & KT_ERR_DUPLICATE) ? " duplicate" : "",
                       (flags & KT_ERR_MESSAGE) ? " bad message" : "");
    // the lists: their offsets, then each entry to its rank's place and every
    // list sorted by itself, or, with one longer than that sort takes, all keys
    // by their bits.  (Five radix passes of five launches took 215 us for the
    // 1.9 M keys of an R-MAT CeTriC shard, place and sort 57.)
    const bool over_wave = (flags & KT_FLAG_OVER_WAVE) != 0, over_group = (flags & KT_FLAG_OVER_GROUP) != 0;
    scan_u64(B.coff, B.coff, X, B.scan_tmp, st);
    if (Mk) {
        const unsigned g = (unsigned)std::min<uint64_t>((Mk + 255) / 256, 16384);
        if (over_group) {
            radix_sort_u64(B.keys, B.alt, Mk, 2 * bits, B.radix_tmp, st);
            k_keys_csr<<<g, 256, 0, st>>>(Mk, bits, B.keys, B.cheads, err);
        } else {
            k_shard_place<<<g, 256, 0, st>>>(Mk, bits, B.keys, rank, B.coff, B.cheads);
            segsort_launch((uint32_t)X, B.coff, B.cheads, err, over_wave ? segsort_max_len() : segsort_wave_len(),
                           c->num_cus, st);
        }
    }
    if (nl) k_cut_begin<<<(nl + 255) / 256, 256, 0, st>>>(nl, B.coff, B.cheads, B.cut);
    rc = c->hip_check(hipMemcpyAsync(c->host_small, B.small, 8, hipMemcpyDeviceToHost, st), "D2H flags");
    if (rc) return rc;
    rc = c->hip_check(hipStreamSynchronize(st), "shard preprocessing");
    if (rc) return rc;
    flags = (uint32_t)c->host_small[0];
    if (flags & KT_ERR_MASK)
        return c->fail(KT_EINVAL, "malformed shard:%s", (flags & KT_ERR_DUPLICATE) ? " duplicate edge" : "");
    (void)hipEventRecord(c->ev[EV_PREP], st);
    uint64_t* pv = want_pv ? (pv_dev ? out->per_vertex : B.pv) : nullptr;
    if (pv) fill_u64(pv, X, 0, st);
    uint64_t* totals = B.small + 4;  // [4] local, [5] type3
    uint64_t* tstats = tc_stats_ptr(B.tc_ws);
    // local phase
    {
        TcView v{};
        v.sheads = B.cheads;
        v.s_off = B.coff;
        if (cetric) {
            v.X = (uint32_t)X;  // plain view over owned + ghost tails, by global degrees
            v.deg = B.deg;
            v.stripe = 1024;
        } else {
            v.X = nl;
            v.r_beg = B.coff;
            v.r_end = B.cut;
            v.rheads = B.cheads;
            v.t_beg = B.coff;
            v.t_end = B.coff + 1;
            v.theads = B.cheads;
        }
        v.room = B.room;
        v.longest = over_wave ? 0 : segsort_wave_len();
        TcOut o{pv, totals};
        rc = c->hip_check(tc_launch(v, o, c->prm, B.tc_ws, c->num_cus, st, c->ev[EV_TC0], c->ev[EV_TC1]),
                          "intersection launch");
        if (rc) return rc;
        rc = c->hip_check(hipMemcpyAsync(c->host_small + 8, tstats, 32, hipMemcpyDeviceToHost, st), "D2H stats");
        if (rc) return rc;
    }
    // contracted / distributed phase
    if (in->n_msg) {
        TcView v{};
        v.X = in->n_msg;
        v.sheads = B.mheads2;
        v.rheads = B.mheads2;
        v.r_beg = B.moff;
        v.r_end = B.msplit;
        if (cetric) {
            v.s_beg = B.msplit;
            v.s_end = B.moff + 1;
            v.t_beg = B.cut;
        } else {
            v.s_off = B.moff;
            v.t_beg = B.coff;
        }
        v.t_end = B.coff + 1;
        v.theads = B.cheads;
        v.tail_id = B.mtail;
        // counters as intersect_from_message keeps them (cetric_edge_iterator.h:1815-1856):
        // per local receiver u, |N+(u)| wedge checks and |message| + |N+(u)|
        // intersected ids; a CeTriC receiver without cut edges was compacted away
        v.stat_off = B.msg_off;
        v.stat_skip_empty = cetric ? 1u : 0u;
        v.room = B.room;
        v.longest = (flags & KT_FLAG_LONG_MESSAGE) ? 0 : segsort_wave_len();
        TcOut o{pv, totals + 1};
        // message tails have short owned parts: a whole workgroup on one of
        // them idles, so tails up to the largest wave table stay with one
        // wave (measured on RMAT-22 and RMAT-26 / 16 ranks); the workgroup
        // teams on the remaining (large) message tails share their receivers
        // 4 (CeTriC) or 2 (DiTriC) at a time, since a few long lists per
        // message make coarser grabs leave waves idle at the end on large
        // shards (with one list per step, RMAT-26 / 16: CeTriC contracted phase
        // 64.6 ms with 8 per grab, 58.4 with 4; with the present walk no
        // difference from 4 to 64 at scale 20 / 16)
        TcParams pm = c->prm;
        pm.wave_max_deg = std::max<uint32_t>(pm.wave_max_deg, 256u);
        pm.team_chunk = std::min<uint32_t>(pm.team_chunk, cetric ? 4u : 2u);
        // messages beyond the last-level cache (2^26 ids, 256 MB) are taken in
        // their order in memory, also by degree: R-MAT scale 26, rank 0 of 16 (906
        // M ids) DiTriC count phase 77.6 ms by degree, 69.4 so; scale 23 / 16 (110
        // M) 6.00 and 5.87, scale 22 / 16 (54 M) 2.63 and 2.61, scale 20 / 16 (13
        // M) 0.62 and 0.65
        if (mtot >= (1ull << 26)) pm.order = TC_BY_VERTEX;
        rc = c->hip_check(tc_launch(v, o, pm, B.tc_ws, c->num_cus, st, nullptr, nullptr), "intersection launch");
        if (rc) return rc;
        rc = c->hip_check(hipMemcpyAsync(c->host_small + 12, tstats, 32, hipMemcpyDeviceToHost, st), "D2H stats");
        if (rc) return rc;
    }
    (void)hipEventRecord(c->ev[EV_COUNT], st);
    rc = c->hip_check(hipMemcpyAsync(c->host_small + 4, totals, 16, hipMemcpyDeviceToHost, st), "D2H totals");
    if (rc) return rc;
    if (want_pv && !pv_dev) {
        rc = c->hip_check(hipMemcpyAsync(out->per_vertex, pv, X * 8, hipMemcpyDeviceToHost, st), "D2H per-vertex");
        if (rc) return rc;
    }
    (void)hipEventRecord(c->ev[EV_END], st);
    rc = c->hip_check(hipStreamSynchronize(st), "shard count");
    if (rc) return rc;
    out->local_triangles = c->host_small[4];
    out->type3_triangles = in->n_msg ? c->host_small[5] : 0;
    c->stats.local_triangles = out->local_triangles;
    c->stats.type3_triangles = out->type3_triangles;
    c->stats.wedge_checks = c->host_small[8] + (in->n_msg ? c->host_small[12] : 0);
    c->stats.intersection_size_local = c->host_small[9];
    c->stats.intersection_size_global = in->n_msg ? c->host_small[13] : 0;
    c->stats.streamed_ids = c->host_small[11] + (in->n_msg ? c->host_small[15] : 0);
    c->stats.oriented_edges = Mk;
    c->stats.vertices = X;
    c->stats.input_slots = nnz;
    c->timing.h2d_ms = c->elapsed(EV_START, EV_H2D);
    c->timing.prep_ms = c->elapsed(EV_H2D, EV_PREP);
    c->timing.count_ms = c->elapsed(EV_PREP, EV_COUNT);
    c->timing.intersect_ms = c->elapsed(EV_TC0, EV_TC1);
    c->timing.d2h_ms = c->elapsed(EV_COUNT, EV_END);
    c->timing.total_ms = c->elapsed(EV_START, EV_END);
    return KT_OK;
}

extern "C" int kt_count_shard(kt_ctx* c, const kt_shard_in* in, kt_shard_out* out) {
    if (!c) return KT_EINVAL;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = c->begin_call(true);
    if (rc) return rc;
    return count_shard_locked(c, in, out);
}
