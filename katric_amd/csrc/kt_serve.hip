// Serving loop: continuous batching of count requests on one GPU.
//
// A worker thread owns two device slots (own stream, own grow-only arena,
// pinned result buffers).  Requests are admitted FIFO into the next batch
// while the batch fits the slot's share of the HBM budget and the batch
// limits; the batch's CSRs are gathered into one disjoint-union CSR in the slot
// (device-resident for the batch's lifetime), by a kernel that reads page-locked
// requests where they are and from copies of the others, then counted by the
// batch pipeline.  Per-vertex counts for pageable memory leave the device as one
// copy into the slot's page-locked buffer and are handed out from there.  While one slot computes, the other uploads and
// launches the next batch, so requests arriving during a batch are admitted
// as soon as a slot frees up, and their work overlaps on the device.
//
// Every result equals the one-graph count: a batch whose validation fails is
// re-run one request per batch so that only the malformed request fails, and
// a batch with unsorted lists is re-run with its oriented lists sorted on the
// device.
#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <thread>
#include <unordered_map>
#include <vector>

#include "../../include/katric_serve.h"
#include "kt_ctx.h"
#include "kt_device.h"
#include "kt_pinned.h"

namespace kt {

static double now_ms() {
    using namespace std::chrono;
    return duration<double, std::milli>(steady_clock::now().time_since_epoch()).count();
}

// One request of a device batch: its CSR as the device reads it (the request's
// page-locked memory, or its copy at its place in the batch arena), its place in
// the batch, and its first work chunk.
struct GatherDesc {
    const uint64_t* off;
    const uint32_t* heads;
    uint64_t n, nnz;
    uint64_t vb, eb;  // vertex / edge base in the batch
    uint64_t c0;      // first chunk (offsets chunks, then heads chunks)
    uint64_t pad;
};
constexpr uint32_t GATHER_CHUNK = 4096;  // ids per chunk
constexpr size_t SERVE_LOOKAHEAD = 4096; // queued requests scanned when forming a batch

__host__ __device__ inline uint64_t gather_chunks(uint64_t n, uint64_t nnz) {
    return (n + GATHER_CHUNK - 1) / GATHER_CHUNK + (nnz + GATHER_CHUNK - 1) / GATHER_CHUNK;
}

// Writes the requests' CSRs into the batch's disjoint-union CSR in one launch:
// off[vb_g + i] = off_g[i] + eb_g, heads[eb_g + k] = heads_g[k] + vb_g (a head
// outside its own graph becomes an invalid id, flagged by the orientation pass),
// off[N] = nnz.  Blocks take chunks of one request's offsets or heads, every
// thread all its elements of a chunk at once: from page-locked memory the loads'
// way over PCIe is what takes the time.  A copied CSR is rebased in place (every
// element is read and written by the same thread).
__global__ void __launch_bounds__(256) k_serve_gather(uint32_t G, const GatherDesc* __restrict__ d,
                                                      uint64_t chunks, uint64_t* off, uint32_t* heads, uint64_t N,
                                                      uint64_t nnz) {
    constexpr int E = GATHER_CHUNK / 256;
    for (uint64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        uint32_t lo = 0, hi = G - 1;  // last request with c0 <= c
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) / 2;
            if (d[mid].c0 <= c)
                lo = mid;
            else
                hi = mid - 1;
        }
        const GatherDesc r = d[lo];
        const uint64_t oc = (r.n + GATHER_CHUNK - 1) / GATHER_CHUNK;
        const uint64_t k = c - r.c0;
        if (k < oc) {
            const uint64_t i0 = k * GATHER_CHUNK + threadIdx.x;
            uint64_t x[E];
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = i0 + j * 256 < r.n ? r.off[i0 + j * 256] : 0;
#pragma unroll
            for (int j = 0; j < E; ++j)
                if (i0 + j * 256 < r.n) off[r.vb + i0 + j * 256] = x[j] + r.eb;
        } else {
            const uint64_t e0 = (k - oc) * GATHER_CHUNK + threadIdx.x;
            uint32_t h[E];
#pragma unroll
            for (int j = 0; j < E; ++j) h[j] = e0 + j * 256 < r.nnz ? r.heads[e0 + j * 256] : 0;
#pragma unroll
            for (int j = 0; j < E; ++j)
                if (e0 + j * 256 < r.nnz)
                    heads[r.eb + e0 + j * 256] = (h[j] < r.n) ? (uint32_t)(h[j] + r.vb) : 0xffffffffu;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) off[N] = nnz;
}

// The device's address of host memory p[0, bytes) that is page-locked as a
// whole, or null.
static const void* device_view(const void* p, uint64_t bytes) {
    return pinned_view(p, bytes, [](const void* q) {
        hipPointerAttribute_t a{};
        hipDeviceptr_t base = nullptr;
        size_t size = 0;
        if (hipPointerGetAttributes(&a, q) != hipSuccess || a.type != hipMemoryTypeHost ||
            hipMemGetAddressRange(&base, &size, const_cast<void*>(q)) != hipSuccess) {
            (void)hipGetLastError();
            return PinnedAt{nullptr, nullptr, 0};
        }
        return PinnedAt{static_cast<const char*>(a.devicePointer), static_cast<const char*>(base), size};
    });
}

struct ServeReq {
    uint64_t ticket;
    uint32_t n;
    uint64_t nnz;
    const uint64_t* off;
    const uint32_t* heads;
    uint64_t* pv_out;
    double t_submit = 0, t_launch = 0, t_done = 0;
    int status = KT_ENOTREADY;
    uint64_t total = 0;
    uint64_t batch_id = 0;
    uint32_t batch_graphs = 0;
    bool staged = false;  // its per-vertex counts come through the slot's buffer
    bool isolate = false;
    bool cancelled = false;
    bool done = false;
};

struct ServeSlot {
    hipStream_t stream = nullptr;
    hipEvent_t ev = nullptr;
    void* arena = nullptr;
    uint64_t arena_bytes = 0;
    uint64_t* h_small = nullptr;  // pinned, 64 words
    uint64_t* h_meta = nullptr;   // pinned: vbase (cap + 1), then the gather descriptors (cap)
    uint64_t* h_totals = nullptr; // pinned, cap
    uint64_t meta_cap = 0;
    uint64_t* h_pv = nullptr;     // pinned, pv_cap: the batch's per-vertex counts
    uint64_t pv_cap = 0;
    bool staged = false;          // they are in h_pv when the batch is done
    std::vector<ServeReq*> reqs;
    bool busy = false;
    bool sorted = false;
    bool large = false;  // the batch is one large request
    bool rich = false;   // its layout has the intersection's optional room
    uint64_t batch_id = 0;
    uint64_t N = 0, nnz = 0;
};

struct ServeState {
    kt_serve_config cfg{};
    int device = 0;
    int num_cus = 0;
    TcParams prm{};
    uint64_t sym_key[2] = {0, 0};
    uint64_t slot_cap = 0;
    uint64_t large_edges = 0;  // requests above this many edges run alone
    std::thread worker;
    std::mutex mu;
    std::condition_variable cv_work, cv_done;
    std::deque<ServeReq*> pending;
    std::unordered_map<uint64_t, ServeReq*> all;
    uint64_t next_ticket = 1;
    uint64_t next_batch = 1;
    bool stop = false;
    ServeSlot slots[2];
    kt_serve_stats st{};
    char err[256] = {0};
};

// Device bytes of a slot's batch: the batch pipeline's buffers (with the
// radix-sort scratch for a relaunch of unsorted lists that needs it) and the
// gather descriptors after them.
static uint64_t slot_bytes(const ServeState* S, uint32_t G, uint64_t N, uint64_t nnz, bool radix, bool rich = false) {
    BatchBufs B;
    return ((batch_layout(nullptr, G, N, nnz, S->num_cus, true, true, radix, rich, B) + 255) & ~255ull) + (uint64_t)G * sizeof(GatherDesc);
}

static uint64_t req_bytes(const ServeState* S, const ServeReq* r) { return slot_bytes(S, 1, r->n, r->nnz, false); }

static int slot_grow(ServeSlot& s, uint64_t bytes, uint32_t G) {
    if (bytes > s.arena_bytes) {
        if (s.arena) (void)hipFree(s.arena);
        s.arena = nullptr;
        s.arena_bytes = 0;
        if (hipMalloc(&s.arena, bytes) != hipSuccess) {
            (void)hipGetLastError();
            s.arena = nullptr;
            return KT_ENOMEM;
        }
        s.arena_bytes = bytes;
    }
    if (G + 1 > s.meta_cap) {
        if (s.h_meta) (void)hipHostFree(s.h_meta);
        if (s.h_totals) (void)hipHostFree(s.h_totals);
        s.h_meta = s.h_totals = nullptr;
        s.meta_cap = 0;
        uint64_t cap = std::max<uint64_t>(2 * (uint64_t)G + 2, 64);
        if (hipHostMalloc(reinterpret_cast<void**>(&s.h_meta), (cap + 1) * 8 + cap * sizeof(GatherDesc),
                          hipHostMallocDefault) != hipSuccess ||
            hipHostMalloc(reinterpret_cast<void**>(&s.h_totals), cap * 8, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return KT_ENOMEM;
        }
        s.meta_cap = cap;
    }
    return KT_OK;
}

// Vertices whose counts are staged at most: 64 MiB of page-locked memory a slot.
constexpr uint64_t STAGE_MAX = 1ull << 23;

static bool stage_grow(ServeSlot& s, uint64_t n) {
    if (n <= s.pv_cap) return true;
    n = std::min(STAGE_MAX, std::max(n, 2 * s.pv_cap));
    if (s.h_pv) (void)hipHostFree(s.h_pv);
    s.h_pv = nullptr;
    s.pv_cap = 0;
    if (hipHostMalloc(reinterpret_cast<void**>(&s.h_pv), n * 8, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        s.h_pv = nullptr;
        return false;
    }
    s.pv_cap = n;
    return true;
}

// Gathers and enqueues one batch on the slot (worker thread, no lock).
static int launch(ServeState* S, ServeSlot& sl, uint32_t sort) {
    const uint32_t G = (uint32_t)sl.reqs.size();
    uint64_t N = 0, nnz = 0;
    for (auto* r : sl.reqs) {
        N += r->n;
        nnz += r->nnz;
    }
    BatchBufs B;
    const bool radix = sort == SORT_RADIX;
    // a slot never holds more than its share of the budget (a relaunch with
    // the radix-sort scratch can need more than admission counted); the
    // intersection's optional room, which admission leaves out, is taken
    // where it fits
    if (slot_bytes(S, G, N, nnz, radix) > S->slot_cap) return KT_ENOMEM;
    sl.rich = slot_bytes(S, G, N, nnz, radix, true) <= S->slot_cap;
    int rc = slot_grow(sl, slot_bytes(S, G, N, nnz, radix, sl.rich), G);
    if (rc == KT_ENOMEM && sl.rich) {
        sl.rich = false;
        rc = slot_grow(sl, slot_bytes(S, G, N, nnz, radix, false), G);
    }
    if (rc) return rc;
    const uint64_t used =
        (batch_layout(sl.arena, G, N, nnz, S->num_cus, true, true, radix, sl.rich, B) + 255) & ~255ull;
    GatherDesc* d_desc = reinterpret_cast<GatherDesc*>(static_cast<char*>(sl.arena) + used);
    uint64_t* vb = sl.h_meta;
    GatherDesc* desc = reinterpret_cast<GatherDesc*>(sl.h_meta + (sl.meta_cap + 1));
    hipStream_t st = sl.stream;
    uint64_t* d_off = const_cast<uint64_t*>(B.off);
    uint32_t* d_heads = const_cast<uint32_t*>(B.heads);
    const double t = now_ms();
    vb[0] = 0;
    uint64_t e = 0, chunks = 0;
    for (uint32_t g = 0; g < G; ++g) {
        ServeReq* r = sl.reqs[g];
        r->t_launch = t;
        GatherDesc& dg = desc[g];
        dg.n = r->n;
        dg.nnz = r->nnz;
        dg.vb = vb[g];
        dg.eb = e;
        dg.c0 = chunks;
        // k_serve_gather reads page-locked arrays itself (47 requests of 9,000
        // vertices on average: 94 copies took 1.2 ms, the kernel takes 0.7);
        // others are copied into their place in the batch and rebased there
        dg.off = static_cast<const uint64_t*>(device_view(r->off, (uint64_t)r->n * 8));
        dg.heads = static_cast<const uint32_t*>(device_view(r->heads, r->nnz * 4));
        if (!dg.off) {
            dg.off = d_off + vb[g];
            if (r->n &&
                hipMemcpyAsync(d_off + vb[g], r->off, (uint64_t)r->n * 8, hipMemcpyHostToDevice, st) != hipSuccess)
                return KT_EHIP;
        }
        if (!dg.heads) {
            dg.heads = d_heads + e;
            if (r->nnz && hipMemcpyAsync(d_heads + e, r->heads, r->nnz * 4, hipMemcpyHostToDevice, st) != hipSuccess)
                return KT_EHIP;
        }
        chunks += gather_chunks(r->n, r->nnz);
        vb[g + 1] = vb[g] + r->n;
        e += r->nnz;
    }
    if (hipMemcpyAsync(B.vbase, vb, ((uint64_t)G + 1) * 8, hipMemcpyHostToDevice, st) != hipSuccess) return KT_EHIP;
    if (hipMemcpyAsync(d_desc, desc, (uint64_t)G * sizeof(GatherDesc), hipMemcpyHostToDevice, st) != hipSuccess)
        return KT_EHIP;
    const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(chunks, (uint64_t)S->num_cus * 4));
    k_serve_gather<<<grid, 256, 0, st>>>(G, d_desc, chunks, d_off, d_heads, N, nnz);
    if (batch_pipeline(st, S->num_cus, S->prm, B, G, N, nnz, B.pv, sl.h_totals, sl.h_small, sort, S->sym_key) !=
        hipSuccess)
        return KT_EHIP;
    // per-vertex counts: a copy into pageable memory holds this thread until the
    // batch is done, so a batch with several such requests takes one copy to the
    // slot's buffer, which finish() hands out.  A single one is left to hold the
    // thread: the requests that arrive meanwhile make one batch (staged too, a
    // burst of 48 ran as three batches: 2.2 ms, with 1.6 ms in two)
    sl.staged = false;
    uint32_t pageable = 0;
    for (uint32_t g = 0; g < G; ++g) {
        ServeReq* r = sl.reqs[g];
        r->staged = r->pv_out && r->n && !device_view(r->pv_out, (uint64_t)r->n * 8);
        pageable += r->staged;
    }
    if (pageable > 1 && N <= STAGE_MAX) sl.staged = stage_grow(sl, N);
    if (sl.staged && hipMemcpyAsync(sl.h_pv, B.pv, N * 8, hipMemcpyDeviceToHost, st) != hipSuccess) return KT_EHIP;
    for (uint32_t g = 0; g < G; ++g) {
        ServeReq* r = sl.reqs[g];
        r->staged = r->staged && sl.staged;
        if (r->pv_out && r->n && !r->staged &&
            hipMemcpyAsync(r->pv_out, B.pv + vb[g], (uint64_t)r->n * 8, hipMemcpyDeviceToHost, st) != hipSuccess)
            return KT_EHIP;
    }
    if (hipEventRecord(sl.ev, st) != hipSuccess) return KT_EHIP;
    sl.N = N;
    sl.nnz = nnz;
    sl.sorted = sort != SORT_NONE;
    sl.busy = true;
    return KT_OK;
}

// Completion of a slot's batch (worker thread, lock held by the caller and
// released while counts are handed out).
static void finish(ServeState* S, ServeSlot& sl, std::unique_lock<std::mutex>& lk) {
    const uint32_t fl = (uint32_t)sl.h_small[0];
    const uint64_t kept = sl.h_small[1];
    const uint32_t G = (uint32_t)sl.reqs.size();
    const bool bad = (fl & KT_ERR_MASK) || 2 * kept != sl.nnz;
    if (sl.staged && !bad) {
        lk.unlock();
        for (uint32_t g = 0; g < G; ++g) {
            ServeReq* r = sl.reqs[g];
            if (r->staged) std::memcpy(r->pv_out, sl.h_pv + sl.h_meta[g], (uint64_t)r->n * 8);
        }
        lk.lock();
    }
    if (bad && G > 1) {
        // isolate: every request of the batch runs alone, at the queue front
        for (int g = (int)G - 1; g >= 0; --g) {
            sl.reqs[g]->isolate = true;
            S->pending.push_front(sl.reqs[g]);
        }
        S->st.isolation_reruns++;
    } else {
        const double t = now_ms();
        for (uint32_t g = 0; g < G; ++g) {
            ServeReq* r = sl.reqs[g];
            r->status = bad ? KT_EINVAL : (r->cancelled ? KT_ECANCELED : KT_OK);
            r->total = bad ? 0 : sl.h_totals[g];
            r->t_done = t;
            r->batch_id = sl.batch_id;
            r->batch_graphs = G;
            r->done = true;
        }
        if (!bad) {
            S->st.batches++;
            S->st.graphs += G;
            S->st.edges += sl.nnz / 2;
        }
    }
    sl.reqs.clear();
    sl.busy = false;
    S->cv_done.notify_all();
}

// A batch that could not be launched (lock held by the caller): a batch of
// several requests that ran out of device memory is re-run one request at a
// time, so that only a request too large on its own fails; any other error
// fails the batch's requests.
static void launch_failed(ServeState* S, ServeSlot& sl, int rc) {
    const uint32_t G = (uint32_t)sl.reqs.size();
    if (rc == KT_ENOMEM && G > 1) {
        for (int g = (int)G - 1; g >= 0; --g) {
            sl.reqs[g]->isolate = true;
            S->pending.push_front(sl.reqs[g]);
        }
        S->st.isolation_reruns++;
    } else {
        for (auto* r : sl.reqs) {
            r->status = rc;
            r->done = true;
        }
    }
    sl.reqs.clear();
    sl.busy = false;
    S->cv_done.notify_all();
}

static void worker_main(ServeState* S) {
    (void)hipSetDevice(S->device);
    std::unique_lock<std::mutex> lk(S->mu);
    while (true) {
        // publish finished batches
        for (auto& sl : S->slots) {
            if (!sl.busy) continue;
            if (hipEventQuery(sl.ev) != hipSuccess) continue;
            (void)hipGetLastError();
            const uint32_t fl = (uint32_t)sl.h_small[0];
            if (!(fl & KT_ERR_MASK) && (fl & KT_FLAG_UNSORTED) && !sl.sorted && 2 * sl.h_small[1] == sl.nnz) {
                lk.unlock();
                // same requests, with the oriented lists sorted (the sort
                // chosen from the longest list of the run that found them)
                BatchBufs B0;
                batch_layout(sl.arena, (uint32_t)sl.reqs.size(), sl.N, sl.nnz, S->num_cus, true, true, false, sl.rich, B0);
                uint32_t mode = SORT_RADIX;
                int rc = batch_sort_mode(sl.stream, B0, sl.N, sl.h_small, mode) == hipSuccess ? KT_OK : KT_EHIP;
                if (rc == KT_OK) rc = launch(S, sl, mode);
                lk.lock();
                if (rc != KT_OK) launch_failed(S, sl, rc);
                continue;
            }
            finish(S, sl, lk);
        }
        ServeSlot* free_slot = nullptr;
        for (auto& sl : S->slots)
            if (!sl.busy) {
                free_slot = &sl;
                break;
            }
        // drop cancelled requests at the queue front
        while (!S->pending.empty() && S->pending.front()->cancelled) {
            ServeReq* r = S->pending.front();
            S->pending.pop_front();
            r->status = KT_ECANCELED;
            r->done = true;
            S->cv_done.notify_all();
        }
        if (free_slot && !S->pending.empty()) {
            // Form the next batch.  A large request (more than large_edges
            // edges) or an isolated one runs alone, and at most one slot runs a
            // large request at a time: while the other slot holds one, a large
            // request at the queue front waits and the small requests behind
            // it form this slot's batch, so that they are not held up behind
            // it.  Small requests are taken in arrival order while the batch
            // fits the slot and the limits.
            ServeSlot& other = (free_slot == &S->slots[0]) ? S->slots[1] : S->slots[0];
            const bool other_large = other.busy && other.large;
            std::vector<ServeReq*> batch;
            bool blocked_large = false;
            uint64_t N = 0, nnz = 0;
            for (size_t i = 0; i < S->pending.size() && i < SERVE_LOOKAHEAD;) {
                ServeReq* r = S->pending[i];
                if (r->cancelled) {
                    S->pending.erase(S->pending.begin() + (ptrdiff_t)i);
                    r->status = KT_ECANCELED;
                    r->done = true;
                    S->cv_done.notify_all();
                    continue;
                }
                const bool large = r->nnz / 2 > S->large_edges;
                if (large || r->isolate) {
                    if (batch.empty() && !(large && other_large)) {
                        S->pending.erase(S->pending.begin() + (ptrdiff_t)i);
                        if (req_bytes(S, r) > S->slot_cap) {
                            r->status = KT_ENOMEM;
                            r->done = true;
                            S->cv_done.notify_all();
                            continue;
                        }
                        batch.push_back(r);
                        blocked_large = large;
                        break;
                    }
                    ++i;  // keeps its place; smaller requests behind it go ahead
                    continue;
                }
                const uint64_t bytes = slot_bytes(S, (uint32_t)batch.size() + 1, N + r->n, nnz + r->nnz, false);
                const bool limits = batch.size() + 1 <= S->cfg.max_batch_graphs &&
                                    (nnz + r->nnz) / 2 <= S->cfg.max_batch_edges;
                if (!batch.empty() && (bytes > S->slot_cap || !limits)) break;
                S->pending.erase(S->pending.begin() + (ptrdiff_t)i);
                if (bytes > S->slot_cap) {  // alone it does not fit the budget share
                    r->status = KT_ENOMEM;
                    r->done = true;
                    S->cv_done.notify_all();
                    continue;
                }
                batch.push_back(r);
                N += r->n;
                nnz += r->nnz;
            }
            if (!batch.empty()) {
                free_slot->reqs = batch;
                free_slot->large = blocked_large;
                free_slot->batch_id = S->next_batch++;
                lk.unlock();
                int rc = launch(S, *free_slot, SORT_NONE);
                lk.lock();
                if (rc != KT_OK) launch_failed(S, *free_slot, rc);
                continue;
            }
            // only a large request waits for the other slot's large one: poll below
        }
        bool any_busy = S->slots[0].busy || S->slots[1].busy;
        if (S->stop && S->pending.empty() && !any_busy) break;
        if (!any_busy) {
            S->cv_work.wait(lk);
        } else if (free_slot) {
            // a slot is free but nothing is pending: wake on a submission or
            // poll the busy slot again shortly
            S->cv_work.wait_for(lk, std::chrono::microseconds(100));
        } else {
            // both slots busy: wait for the earliest-launched one without the lock
            ServeSlot* w = nullptr;
            for (auto& sl : S->slots)
                if (sl.busy && (!w || sl.batch_id < w->batch_id)) w = &sl;
            hipEvent_t ev = w->ev;
            lk.unlock();
            (void)hipEventSynchronize(ev);
            lk.lock();
        }
    }
}

}  // namespace kt

using namespace kt;

static int serve_stop_impl(kt_ctx* c) {
    ServeState* S = c->serve;
    if (!S) return KT_OK;
    {
        std::lock_guard<std::mutex> lk(S->mu);
        S->stop = true;
    }
    S->cv_work.notify_all();
    if (S->worker.joinable()) S->worker.join();
    for (auto& sl : S->slots) {
        if (sl.stream) (void)hipStreamSynchronize(sl.stream);
        if (sl.arena) (void)hipFree(sl.arena);
        if (sl.h_small) (void)hipHostFree(sl.h_small);
        if (sl.h_meta) (void)hipHostFree(sl.h_meta);
        if (sl.h_totals) (void)hipHostFree(sl.h_totals);
        if (sl.h_pv) (void)hipHostFree(sl.h_pv);
        if (sl.ev) (void)hipEventDestroy(sl.ev);
        if (sl.stream) (void)hipStreamDestroy(sl.stream);
    }
    for (auto& kv : S->all) delete kv.second;
    delete S;
    c->serve = nullptr;
    return KT_OK;
}

void kt_serve_release(kt_ctx* c) { serve_stop_impl(c); }

extern "C" int kt_serve_start(kt_ctx* c, const kt_serve_config* cfg) {
    if (!c) return KT_EINVAL;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = c->begin_call(false);
    if (rc) return rc;
    if (c->serve) return c->fail(KT_ESTATE, "serving loop already running");
    ServeState* S = new ServeState();
    if (cfg) S->cfg = *cfg;
    if (S->cfg.max_batch_graphs == 0) S->cfg.max_batch_graphs = 4096;
    if (S->cfg.max_batch_edges == 0) S->cfg.max_batch_edges = 1ull << 25;
    S->large_edges = S->cfg.large_request_edges ? S->cfg.large_request_edges : S->cfg.max_batch_edges / 4;
    uint64_t budget = S->cfg.hbm_budget_bytes ? S->cfg.hbm_budget_bytes : c->budget;
    if (budget == 0) {
        size_t fr = 0, tot = 0;
        if (hipMemGetInfo(&fr, &tot) != hipSuccess) {
            (void)hipGetLastError();
            fr = 16ull << 30;
        }
        budget = fr / 2;
    }
    S->slot_cap = budget / 2;
    S->device = c->device;
    S->num_cus = c->num_cus;
    S->prm = c->prm;
    S->sym_key[0] = c->sym_key[0];
    S->sym_key[1] = c->sym_key[1];
    for (auto& sl : S->slots) {
        if (hipStreamCreateWithFlags(&sl.stream, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&sl.ev, hipEventDisableTiming) != hipSuccess ||
            hipHostMalloc(reinterpret_cast<void**>(&sl.h_small), 64 * 8, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            c->serve = S;
            serve_stop_impl(c);
            return c->fail(KT_EHIP, "serving loop: stream/event/pinned allocation failed");
        }
    }
    c->serve = S;
    S->worker = std::thread(worker_main, S);
    trace("serve: started, slot budget %llu bytes", (unsigned long long)S->slot_cap);
    return KT_OK;
}

extern "C" int kt_serve_stop(kt_ctx* c) {
    if (!c) return KT_EINVAL;
    std::lock_guard<std::mutex> lk(c->mu);
    return serve_stop_impl(c);
}

extern "C" int kt_serve_submit(kt_ctx* c, uint32_t n, const uint64_t* offsets, const uint32_t* heads,
                               uint64_t* per_vertex_out, uint64_t* ticket) {
    if (!c || !ticket || !offsets) return KT_EINVAL;
    ServeState* S = c->serve;
    if (!S) return KT_ESTATE;
    if (offsets[0] != 0) return KT_EINVAL;
    const uint64_t nnz = offsets[n];
    if ((nnz & 1) || (nnz && !heads)) return KT_EINVAL;
    ServeReq* r = new ServeReq();
    r->n = n;
    r->nnz = nnz;
    r->off = offsets;
    r->heads = heads;
    r->pv_out = per_vertex_out;
    r->t_submit = now_ms();
    {
        std::lock_guard<std::mutex> lk(S->mu);
        if (S->stop) {
            delete r;
            return KT_ESTATE;
        }
        r->ticket = S->next_ticket++;
        S->all[r->ticket] = r;
        if (req_bytes(S, r) > S->slot_cap) {
            r->status = KT_ENOMEM;
            r->done = true;
        } else {
            S->pending.push_back(r);
        }
        S->st.submitted++;
        *ticket = r->ticket;
    }
    S->cv_work.notify_all();
    return KT_OK;
}

static void fill_result(const ServeReq* r, kt_serve_result* out) {
    out->ticket = r->ticket;
    out->status = r->status;
    out->total = r->total;
    out->queue_ms = r->t_launch > 0 ? r->t_launch - r->t_submit : 0;
    out->latency_ms = r->t_done - r->t_submit;
    out->batch_id = r->batch_id;
    out->batch_graphs = r->batch_graphs;
}

extern "C" int kt_serve_poll(kt_ctx* c, uint64_t ticket, kt_serve_result* out) {
    if (!c || !out) return KT_EINVAL;
    ServeState* S = c->serve;
    if (!S) return KT_ESTATE;
    std::lock_guard<std::mutex> lk(S->mu);
    auto it = S->all.find(ticket);
    if (it == S->all.end()) return KT_ENOTFOUND;
    if (!it->second->done) return KT_ENOTREADY;
    fill_result(it->second, out);
    delete it->second;
    S->all.erase(it);
    return KT_OK;
}

extern "C" int kt_serve_wait(kt_ctx* c, uint64_t ticket, double timeout_ms, kt_serve_result* out) {
    if (!c || !out) return KT_EINVAL;
    ServeState* S = c->serve;
    if (!S) return KT_ESTATE;
    std::unique_lock<std::mutex> lk(S->mu);
    auto it = S->all.find(ticket);
    if (it == S->all.end()) return KT_ENOTFOUND;
    ServeReq* r = it->second;
    auto pred = [&] { return r->done; };
    if (timeout_ms < 0)
        S->cv_done.wait(lk, pred);
    else if (!S->cv_done.wait_for(lk, std::chrono::duration<double, std::milli>(timeout_ms), pred))
        return KT_ENOTREADY;
    fill_result(r, out);
    delete r;
    S->all.erase(ticket);
    return KT_OK;
}

extern "C" int kt_serve_cancel(kt_ctx* c, uint64_t ticket) {
    if (!c) return KT_EINVAL;
    ServeState* S = c->serve;
    if (!S) return KT_ESTATE;
    std::lock_guard<std::mutex> lk(S->mu);
    auto it = S->all.find(ticket);
    if (it == S->all.end()) return KT_ENOTFOUND;
    if (it->second->done) return KT_ESTATE;
    it->second->cancelled = true;
    S->cv_work.notify_all();
    return KT_OK;
}

extern "C" int kt_serve_get_stats(kt_ctx* c, kt_serve_stats* out) {
    if (!c || !out) return KT_EINVAL;
    ServeState* S = c->serve;
    if (!S) return KT_ESTATE;
    std::lock_guard<std::mutex> lk(S->mu);
    *out = S->st;
    out->pending = S->pending.size();
    return KT_OK;
}
