// Index plans of small inputs, built by one workgroup in one launch.
//
// A CSR build by the general kernels (plan_kernels.hip) is a chain of 8 to 14
// launches, an inverse build one of 4; below some ten thousand edges each of
// them runs for its latency only (2 to 12 us in a few workgroups) and the chain
// is what the build costs.  Here the whole build stays in the LDS of one
// workgroup.  The work grows with the edges and keys on one compute unit while
// the chain's latency does not, so larger inputs go to the general kernels
// (small_csr_plan, small_inv_plan).
//
// The plans are those of the general kernels, array for array; only the
// snapshot tiles flagged plain are stored here too (nothing reads them).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_utils.h"
#include "internal.h"

namespace relm_mp {

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int kDigitBits = 7;
constexpr int kDigits = 1 << kDigitBits;

constexpr int log2_of(int v) { return v <= 1 ? 0 : 1 + log2_of(v / 2); }

// One lane stores the validation status to the plan's status and, where the
// build waits on the host for it, to the host's mapped copy with `gen` behind it
// (system-scope release).
__device__ __forceinline__ void publish(const DevStatus& v, DevStatus* __restrict__ st,
                                        const StatusPublish& pub) {
    *st = v;
    if (pub.host == nullptr) return;
    *pub.host = v;
    __hip_atomic_store(pub.host_gen, pub.gen, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ DevStatus new_status(uint32_t bad_key, uint32_t bad_gather) {
    DevStatus v{};
    v.bad_key_edge = bad_key == ~0u ? kNoEdge : bad_key;
    v.bad_gather_edge = bad_gather == ~0u ? kNoEdge : bad_gather;
    return v;
}

// An index checked against its bound; 0 and the smallest bad edge if it fails.
__device__ __forceinline__ uint32_t narrow(int64_t v, int64_t bound, uint32_t p, uint32_t& bad) {
    const bool ok = static_cast<uint64_t>(v) < static_cast<uint64_t>(bound);
    bad = ok ? bad : min(bad, p);
    return ok ? static_cast<uint32_t>(v) : 0u;
}

// Totals over keys packed into one word, so that one scan adds them up: hub
// messages (15 bits), hubs (9), hubs of more than one chunk (4), chunks beyond
// one per hub (4).
constexpr int kHubShift = 15, kMultiShift = 24, kExtraShift = 28;
static_assert(kSmallPlanMax < (1 << kHubShift), "hub messages");
static_assert(kSmallPlanMax / (kHubThreshold + 1) < (1 << (kMultiShift - kHubShift)), "hubs");
static_assert(kSmallPlanMax / (kChunkSize + 1) < 16, "hubs of more than one chunk");
static_assert(kSmallPlanMax / kChunkSize < 16, "chunks beyond one per hub");

__device__ __forceinline__ uint32_t key_word(uint32_t deg) {
    if (deg <= kHubThreshold) return 0u;
    const uint32_t chunks = (deg + kChunkSize - 1) / kChunkSize;
    return deg | 1u << kHubShift | (chunks > 1 ? 1u : 0u) << kMultiShift | (chunks - 1) << kExtraShift;
}

// The CSR build for n <= kCap edges over key_bound <= kCap keys, kCap = 1024 *
// ITEMS: validation and snapshot, a stable LSD radix sort of (key, edge) packed
// into one word each (one pass of up to 7 bits, or two), offsets from a running
// maximum of the segments' ends, then the per-key index.  Bound by latency: some
// 15 barriers and, per sort pass and 64 edges of a wave, about a hundred
// instructions of ranking.  keys and gathers are read before the validation is
// published and not after it.  Wave w owns positions [w * per, w * per + per) in
// rounds of 64, so the order (wave, round, lane) is the edge order.
template <int ITEMS>
__global__ __launch_bounds__(kThreads) void k_csr_small(
    const int64_t* __restrict__ keys, int64_t key_bound, const int64_t* __restrict__ gathers,
    int64_t gather_bound, int n, int bits, SmallCsr a, DevStatus* __restrict__ st, StatusPublish pub) {
    constexpr int kCap = kThreads * ITEMS;
    constexpr int kPosBits = log2_of(kCap);
    constexpr uint32_t kPosMask = kCap - 1;
    static_assert(2 * kPosBits <= 32, "key and edge in one word");
    __shared__ uint32_t sk[kCap];      // key << kPosBits | edge
    __shared__ uint32_t sx[kCap + 1];  // per key: end of its segment, then hub messages before it
    __shared__ uint32_t wcnt[kWaves][kDigits];
    __shared__ uint32_t scan_lds[kWaves];
    __shared__ uint32_t s_bad[2], s_max;
    __shared__ uint32_t s_mis[kCap / kSnapTile];
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = lane_id(), wave = tid / kWave;
    const int nk = static_cast<int>(key_bound);
    const int rounds = (n + kThreads - 1) / kThreads;
    const int p0 = wave * rounds * kWave + lane;
    // rounds in which this lane has an edge: its positions are p0 + r * 64, r < mine
    const int mine = max(0, min(rounds, (n - p0 + kWave - 1) / kWave));
    if (tid < 2) s_bad[tid] = ~0u;
    if (tid == 2) s_max = 0;
    if (tid < kCap / kSnapTile) s_mis[tid] = 0;
    for (int k = tid; k <= nk; k += kThreads) sx[k] = 0;
    __syncthreads();

    // ---- validation, snapshot; four loads of a thread in flight
    {
        uint32_t bad_k = ~0u, bad_g = ~0u;
#pragma unroll 1
        for (int r0 = 0; r0 < mine; r0 += 4) {
            int64_t kv[4], gv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int p = p0 + (r0 + j) * kWave;
                kv[j] = r0 + j < mine ? keys[p] : 0;
                gv[j] = r0 + j < mine && gathers != nullptr ? gathers[p] : 0;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (r0 + j >= mine) continue;
                const int p = p0 + (r0 + j) * kWave;
                const uint32_t k = narrow(kv[j], key_bound, p, bad_k);
                a.snap_keys[p] = k;
                sk[p] = k << kPosBits | static_cast<uint32_t>(p);
                if (gathers != nullptr) {
                    a.snap_gathers[p] = narrow(gv[j], gather_bound, p, bad_g);
                    if (gv[j] != p) s_mis[p / kSnapTile] = 1;  // only ever 1
                }
            }
        }
        if (bad_k != ~0u) atomicMin(&s_bad[0], bad_k);
        if (bad_g != ~0u) atomicMin(&s_bad[1], bad_g);
    }
    __syncthreads();
    if (wave == kWaves - 1) {
        if (lane < (n + kSnapTile - 1) / kSnapTile) a.snap_plain[lane] = s_mis[lane] != 0u ? 0u : 1u;
        if (lane == 0) {
            DevStatus v = new_status(s_bad[0], s_bad[1]);
            for (int t = 0; t < kCap / kSnapTile; ++t) v.gather_mismatch |= s_mis[t];
            publish(v, st, pub);
        }
    }

    // ---- sort: digits of the keys from the lowest, stable
    const int passes = bits <= kDigitBits ? 1 : 2;
    int shift = kPosBits;
    for (int pass = 0; pass < passes; ++pass) {
        const int width = bits / passes + (pass < bits % passes ? 1 : 0);
        const uint32_t dmask = (1u << width) - 1u;
        for (int i = tid; i < kWaves * kDigits; i += kThreads) (&wcnt[0][0])[i] = 0;
        __syncthreads();
        uint32_t item[ITEMS], rank[ITEMS];
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) item[r] = r < mine ? sk[p0 + r * kWave] : 0u;
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            rank[r] = 0;
            if (r < rounds) {
                const bool active = r < mine;
                const uint32_t d = (item[r] >> shift) & dmask;
                const unsigned long long peers = match_digit<kDigitBits>(d, __ballot(active));
                const uint32_t below = __popcll(peers & lanemask_lt());
                const uint32_t before = active ? wcnt[wave][d] : 0u;
                rank[r] = before + below;
                if (active && below == 0) wcnt[wave][d] = before + __popcll(peers);
                wave_lds_sync();
            }
        }
        __syncthreads();
        // per digit: where each wave's elements start in the sorted order
        uint32_t run = 0;
        if (tid < kDigits) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const uint32_t c = wcnt[w][tid];
                wcnt[w][tid] = run;
                run += c;
            }
        }
        uint32_t total;
        const uint32_t start = block_inclusive_scan<kThreads>(run, scan_lds, total) - run;
        if (tid < kDigits) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) wcnt[w][tid] += start;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            if (r < mine) {
                const uint32_t d = (item[r] >> shift) & dmask;
                sk[(wcnt[wave][d] + rank[r]) & kPosMask] = item[r];
            }
        }
        __syncthreads();
        shift += width;
    }

    // ---- offsets: each segment's end, then a running maximum over the keys
    for (int p = tid; p < n; p += kThreads) {
        const uint32_t k = sk[p] >> kPosBits;
        if (p + 1 == n || sk[p + 1] >> kPosBits != k) sx[k] = static_cast<uint32_t>(p) + 1u;
    }
    __syncthreads();
    // consecutive keys per thread, key nk (the end) among them: an odd number, so
    // that the threads of a wave, which read kpt apart, hit different banks
    const int kpt = (nk / kThreads + 1) | 1;
    const int k0 = min(tid * kpt, nk + 1), k1 = min(k0 + kpt, nk + 1);
    uint32_t last = 0;
    for (int k = k0; k < k1; ++k) last = max(last, sx[k]);
    const uint32_t off0 = block_exclusive_max<kThreads>(last, scan_lds);
    // hubs among this thread's keys
    uint32_t word = 0, longest = 0, off = off0;
    for (int k = k0; k < k1; ++k) {
        const uint32_t end = max(off, sx[k]);
        word += key_word(end - off);
        longest = max(longest, end - off);
        off = end;
    }
    if (longest != 0) atomicMax(&s_max, longest);
    uint32_t total;
    uint32_t before = block_inclusive_scan<kThreads>(word, scan_lds, total) - word;

    // ---- per-key index
    off = off0;
    for (int k = k0; k < k1; ++k) {
        const uint32_t end = max(off, sx[k]);
        const uint32_t deg = end - off, w = key_word(deg);
        const uint32_t hub_edges = before & ((1u << kHubShift) - 1u);
        const int64_t S = static_cast<int64_t>(off) - hub_edges, W = k + S;
        a.offsets[k] = static_cast<int32_t>(off);
        a.short_off[k] = static_cast<int32_t>(S);
        if (k == 0) {
            a.item_first[0] = 0;
            a.item_short[0] = 0;
        }
        if (k < nk) {
            // the items that begin at key k + 1, whose weight is W1
            const int64_t S1 = S + (w == 0 ? deg : 0), W1 = k + 1 + S1;
            for (int64_t j = W / kItemSize + 1; j <= min(W1 / kItemSize, a.item_capacity); ++j) {
                a.item_first[j] = k + 1;
                a.item_short[j] = static_cast<int32_t>(S1);
            }
        } else {
            // the end closes the last item; the totals
            const int64_t j = W / kItemSize + 1;
            if (j <= a.item_capacity) {
                a.item_first[j] = nk;
                a.item_short[j] = static_cast<int32_t>(S);
            }
            const uint32_t hubs = (total >> kHubShift) & ((1u << (kMultiShift - kHubShift)) - 1u);
            const uint32_t multi = (total >> kMultiShift) & 15u;
            const uint32_t chunks = hubs + (total >> kExtraShift);
            const uint32_t degree = s_max;  // complete: barriers of the scan above
            a.counts->max_degree = st->max_degree = degree;
            a.counts->num_hubs = st->num_hubs = hubs;
            a.counts->num_chunks = st->num_chunks = chunks;
            a.counts->num_multi_hubs = st->num_multi_hubs = multi;
            a.counts->num_items = min(j, a.item_capacity);
            a.counts->num_short = S;
            st->total_weight = W;
        }
        if (w != 0) {
            const uint32_t slot = (before >> kHubShift) & ((1u << (kMultiShift - kHubShift)) - 1u);
            const uint32_t chunk = slot + (before >> kExtraShift);
            a.hub_key[slot] = k;
            a.hub_chunk_base[slot] = static_cast<int32_t>(chunk);
            if (w >> kMultiShift & 15u) a.multi_hubs[before >> kMultiShift & 15u] = static_cast<int32_t>(slot);
            for (uint32_t c = 0; c <= w >> kExtraShift; ++c) a.chunk_hub[chunk + c] = static_cast<int32_t>(slot);
        }
        sx[k] = hub_edges | (w != 0 ? 1u << 31 : 0u);
        before += w;
        off = end;
    }
    __syncthreads();

    // ---- the gathered rows in key order, and without the hubs' segments: from
    // the snapshot, for the caller may change its arrays once the validation is
    // published
    const bool any_hub = (total >> kHubShift) != 0u;
#pragma unroll 1
    for (int q = tid; q < n; q += 4 * kThreads) {
        uint32_t it[4], g[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            it[j] = sk[min(q + j * kThreads, n - 1)];
            g[j] = gathers != nullptr ? a.snap_gathers[it[j] & kPosMask] : it[j] & kPosMask;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int p = q + j * kThreads;
            if (p >= n) continue;
            const int32_t v = static_cast<int32_t>(g[j]);
            a.gather_sorted[p] = v;
            if (any_hub) {
                const uint32_t x = sx[it[j] >> kPosBits];
                if (!(x >> 31)) a.short_gather[p - static_cast<int>(x)] = v;
            }
        }
    }
}

// The inverse map for n <= kCap edges over key_bound <= kCap keys: inv[k] = max e
// with keys[e] == k, claimed in LDS; validation, snapshot, statistics and their
// publication as the general build's.
template <int ITEMS>
__global__ __launch_bounds__(kThreads) void k_inv_small(
    const int64_t* __restrict__ keys, int64_t key_bound, const int64_t* __restrict__ gathers,
    int64_t gather_bound, int n, int32_t* __restrict__ inv, SnapOut snap,
    relm_mp_plan_counts* __restrict__ counts, DevStatus* __restrict__ st, StatusPublish pub) {
    constexpr int kCap = kThreads * ITEMS;
    constexpr int kTiles = kCap / kSnapTile;
    __shared__ int32_t s_inv[kCap];
    __shared__ uint32_t s_bad[2], s_lost;
    __shared__ uint32_t s_mis[2 * kTiles];
    const int tid = static_cast<int>(threadIdx.x);
    const int nk = static_cast<int>(key_bound);
    if (tid < 2) s_bad[tid] = ~0u;
    if (tid == 2) s_lost = 0;
    if (tid < 2 * kTiles) s_mis[tid] = 0;
    int64_t kv[ITEMS], gv[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int p = r * kThreads + tid;
        kv[r] = p < n ? keys[p] : p;
        gv[r] = p < n && gathers != nullptr ? gathers[p] : p;
    }
    for (int k = tid; k < nk; k += kThreads) s_inv[k] = -1;
    __syncthreads();
    uint32_t bad_k = ~0u, bad_g = ~0u, lost = 0;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int p = r * kThreads + tid;
        if (p < n) {
            const uint32_t k = narrow(kv[r], key_bound, p, bad_k);
            if (kv[r] != p) s_mis[p / kSnapTile] = 1;
            if (static_cast<uint64_t>(kv[r]) < static_cast<uint64_t>(key_bound))
                lost += atomicMax(&s_inv[k], p) >= 0 ? 1u : 0u;
            if (snap.keys != nullptr) snap.keys[p] = k;
            if (gathers != nullptr) {
                const uint32_t g = narrow(gv[r], gather_bound, p, bad_g);
                if (gv[r] != p) s_mis[kTiles + p / kSnapTile] = 1;
                if (snap.gathers != nullptr) snap.gathers[p] = g;
            }
        }
    }
    if (bad_k != ~0u) atomicMin(&s_bad[0], bad_k);
    if (bad_g != ~0u) atomicMin(&s_bad[1], bad_g);
    if (lost != 0) atomicAdd(&s_lost, lost);
    __syncthreads();
    for (int k = tid; k < nk; k += kThreads) inv[k] = s_inv[k];
    if (tid < (n + kSnapTile - 1) / kSnapTile) {
        if (snap.key_plain != nullptr) snap.key_plain[tid] = s_mis[tid] != 0u ? 0u : 1u;
        if (snap.gather_plain != nullptr) snap.gather_plain[tid] = s_mis[kTiles + tid] != 0u ? 0u : 1u;
    }
    // Published behind the whole plan, as by the general build: the host's word
    // is all that a caller waits for before other streams read the map or its
    // memory is used again.  The barrier orders the workgroup's stores before the
    // publishing thread's system-scope release, which covers them all.
    __syncthreads();
    if (tid == 0) {
        DevStatus v = new_status(s_bad[0], s_bad[1]);
        for (int t = 0; t < kTiles; ++t) v.key_mismatch |= s_mis[t];
        v.collisions = s_lost;
        counts->collisions = static_cast<int64_t>(v.collisions);
        counts->identity = v.key_mismatch == 0 ? 1 : 0;
        publish(v, st, pub);
    }
}

}  // namespace

bool small_inv_plan(int64_t num_edges, int64_t num_keys) {
    return num_edges > 0 && num_edges <= kSmallPlanMax && num_keys <= kSmallPlanMax;
}

bool small_csr_plan(int64_t num_edges, int64_t num_keys) {
    return small_inv_plan(num_edges, num_keys) && num_edges + num_keys <= kSmallCsrMax;
}

// Builds back to back, here and by the general kernels: 3,200 edges over 200 keys
// 15 and 35 us, 8,192 over 8,192 32 and 44, 16,384 over 1,000 39 and 41, over 7,500
// 45 and 45, over 16,384 56 and 45; 12,288 over 12,288 44 and 45, over 15,500 49 and
// 45; 8,192 over 16,384 43 and 46.
hipError_t launch_csr_small(const int64_t* keys, int64_t key_bound, const int64_t* gathers,
                            int64_t gather_bound, int64_t n, const SmallCsr& a, DevStatus* st,
                            const StatusPublish& pub, hipStream_t s) {
    int bits = 0;
    while ((1ll << bits) < key_bound) ++bits;
    const auto kernel = std::max(n, key_bound) <= 4 * kThreads ? k_csr_small<4> : k_csr_small<16>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kThreads), 0, s, keys, key_bound, gathers, gather_bound,
                       static_cast<int>(n), bits, a, st, pub);
    return hipGetLastError();
}

// Builds back to back, here and by the general kernels: 3,200 edges over 200 keys
// 16 and 25 us, 8,192 over 8,192 20 and 32, 16,384 over 16,384 25 and 33: the limit
// is the LDS.
hipError_t launch_inv_small(const int64_t* keys, int64_t key_bound, const int64_t* gathers,
                            int64_t gather_bound, int64_t n, int32_t* inv, const SnapOut& snap,
                            relm_mp_plan_counts* counts, DevStatus* st, const StatusPublish& pub,
                            hipStream_t s) {
    const auto kernel = std::max(n, key_bound) <= 4 * kThreads ? k_inv_small<4> : k_inv_small<16>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kThreads), 0, s, keys, key_bound, gathers, gather_bound,
                       static_cast<int>(n), inv, snap, counts, st, pub);
    return hipGetLastError();
}

}  // namespace relm_mp
