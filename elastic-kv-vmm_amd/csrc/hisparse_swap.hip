// HiSparse hot-buffer swap-in with the calling convention of SGLang's
// load_blocks_to_device_buffer_mha (gfx950).
//
// The reference's decode path reaches that third-party kernel through its
// HiSparse coordinator (adaptive_sparse/request_residency.py:805-809,829-832).
// Its observable behaviour is pinned by the reference's own smoke test
// (tests/smoke_minimax_swap.py:18-67) and models:
//   - selected tokens: each Top-K block >= 0 expanded to block * bs + j,
//     kept when below the row's length, in Top-K order
//     (adaptive_sparse/hisparse_access_trace.py:59-64);
//   - the newest token (length - 1) always hits (:68-70), at the reserved
//     slot H (its data was written there by the decode step, so it is never
//     copied);
//   - any other token hits when one of the H hot slots holds it;
//   - batch-token LRU (benchmarks/hisparse_locality_replay.py:90-99): misses
//     are counted at entry, hits are touched in selection order, the misses
//     take the least recent slots (empty slots first) and are inserted in
//     selection order; their K and V rows are copied from the pinned host
//     cache into the device rows of their slots;
//   - the output lists the device location of every selected token in
//     selection order, then -1 (tests/smoke_minimax_swap.py:58-66).
// State per request r: device_buffer_tokens[r, i] (token in slot i, -1 =
// empty; column H untouched), lru_slots[r, 0..H) (slots from least to most
// recent), device_buffer_locs[r, i] (device row of slot i; column H is the
// reserved newest-token row), host_cache_locs[r, t] (host row of token t).
//
// One workgroup per batch row:
//   1. the hot tokens are hashed into LDS (open addressing, at least 2H
//      buckets holding slot ids, so every probe sequence meets an empty
//      bucket);
//   2. each lane probes the hash: a hit records its slot, a miss claims a
//      bucket for its token. A token repeated in a row (a repeated Top-K
//      block) is classified once, by its first lane (atomicMin), and its
//      other lanes reuse that lane's location, so the hot buffer never holds
//      a token twice;
//   3. ranks in selection order (output position, hit rank, miss rank): each
//      thread counts a contiguous run of lanes, one workgroup scan (DPP steps
//      in each wave + one LDS exchange) turns the counts into ranks;
//   4. the same scan over contiguous runs of the old LRU order gives each
//      slot's place in the new order and the victims (empty slots first, then
//      untouched slots);
//   5. the misses' rows are copied from mapped pinned host memory, 16 bytes
//      per lane when rows and bases allow: by the row's own workgroup, or by
//      a second launch where few batch rows miss much.
// Locations outside the device buffer are reported as -1 and never written.
#include "../../include/ekv_kernels.h"
#include "ekv_common.h"
#include "ekv_device.h"
#include "ekv_fastdiv.h"
#include "ekv_tensor_util.h"
#include "ekv_token.h"
#include "ekv_vec.h"
#include "ekv_wave.h"

#include <algorithm>
#include <atomic>
#include <climits>

namespace ekv {
namespace {

constexpr int64_t kMaxHot = 4096;     // hot slots per request (LDS holds the hash and the order)
constexpr int64_t kMaxLanes = 2048;   // selected lanes per row (Top-K blocks x block size)
constexpr int kLanesPerThread = 2;    // lanes per thread of the swap at most
constexpr int kBatch = 4;             // hot slots per thread of the swap at most
constexpr int kMaxWaves = 16;         // of the largest swap workgroup
static_assert(kMaxLanes <= kLanesPerThread * 64 * kMaxWaves && kMaxHot <= kBatch * 64 * kMaxWaves,
              "the largest workgroup holds the largest row");
constexpr int kSlotBits = 12;         // a miss left for the copy launch: -2 - (miss rank << kSlotBits | slot)
static_assert(kMaxHot <= 1 << kSlotBits && kMaxLanes << kSlotBits < int64_t{1} << 30, "slot and rank fit an entry");
constexpr int32_t kEmpty = -1;
constexpr int kMaxDevices = 64;

enum LaneKind : uint8_t { kInvalid = 0, kNewest = 1, kHit = 2, kMiss = 3 };

struct HsArgs {
    const void* topk;                  // [B, K] block ids
    int32_t topk64;
    int64_t topk_sb, topk_sk;
    int32_t* tokens;                   // device_buffer_tokens [R, >= H + 1] int32
    int64_t tok_sr, tok_ss;
    const void* host_locs;             // host_cache_locs [R, T]
    int32_t host_locs64;
    int64_t hl_sr, hl_st;
    const void* dev_locs;              // device_buffer_locs [R, >= H + 1]
    int32_t dev_locs64;
    int64_t dl_sr, dl_ss;
    void* lru;                         // lru_slots [R, H] int16 or int32
    int32_t lru32;
    int64_t lru_sr, lru_ss;
    int32_t* out;                      // top_k_device_locs [B, W] int32
    int64_t out_sb, out_so;
    IndexRef req, seq;                 // [B]
    IndexRef num_real;                 // [1] (data null: every row is real)
    const char* host_k;                // mapped pinned host rows
    int64_t host_kv, host_rs, host_rows;
    char* dev_k;                       // device rows
    int64_t dev_kv, dev_rs, dev_rows;
    int64_t row_bytes;
    int64_t batch, R, T, H, HB;
    uint32_t hb_shift;                 // 32 - log2(HB)
    uint32_t width;                    // W = K * block size
    uint32_t block_size;
    FastDiv block_div;
    FastDiv row_div;                   // pieces of one miss (K and V) in copy units
};

struct Lds {
    int32_t* hash;        // [HB] slot id (< H), H + lane (pending miss), or kEmpty
    int32_t* tok;         // [H] token per slot
    int32_t* first_touch; // [H] lowest lane that hit the slot (INT32_MAX: none)
    int16_t* hit_rank;    // [H] rank of the slot's first hit among first hits (-1: none)
    int16_t* order;       // [H] old LRU order
    int16_t* victim;      // [W] slot taken by the m-th miss (-1: none)
    int16_t* miss_lane;   // [W] lane of the m-th miss
    int16_t* lane_rank;   // [W] miss rank of a lane that owns its token's miss
    int32_t* lane_tok;    // [W]
    int32_t* lane_aux;    // [W] hit: slot; miss: hash bucket
    int32_t* lane_pos;    // [W] output position (-1: not selected)
    int32_t* lane_val;    // [W] hit: its device row (-1: outside the buffer); miss: its host row
    int32_t* miss_loc;    // [W] device row of the m-th miss (-1: none)
    uint8_t* lane_kind;   // [W]
    int32_t* scratch;     // [3 * kMaxWaves + 4]
};

// Exclusive prefix sums of N per-thread counts over the workgroup's threads
// in thread order, and their totals: a wave64 scan, then one LDS
// exchange of the wave totals. Every thread must call it (two barriers).
template <int N, int kWaves>
__device__ __forceinline__ void scan_counts(const int32_t (&count)[N], int32_t (&prefix)[N], int32_t (&total)[N],
                                            int32_t* scratch) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int32_t inclusive[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int32_t v = static_cast<int32_t>(wave_scan<kAdd>(static_cast<uint32_t>(count[k])));
        inclusive[k] = v;
        if (lane == 63) {
            scratch[k * kWaves + wave] = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
        int32_t before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int32_t c = scratch[k * kWaves + w];
            before += w < wave ? c : 0;
            all += c;
        }
        prefix[k] = before + inclusive[k] - count[k];
        total[k] = all;
    }
    __syncthreads();  // scratch is rewritten by the next call
}

__device__ __forceinline__ uint32_t bucket_of(const HsArgs& a, int32_t token) {
    return (static_cast<uint32_t>(token) * 0x9E3779B1u) >> a.hb_shift;
}

// A hash entry read while other lanes may be claiming buckets.
__device__ __forceinline__ int32_t load_entry(const Lds& s, uint32_t bucket) {
    return __hip_atomic_load(&s.hash[bucket], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Device row of slot `slot` (0..H), or -1 when outside the device buffer.
__device__ __forceinline__ int64_t device_row(const HsArgs& a, int64_t r, int64_t slot) {
    const int64_t row = load_index(a.dev_locs, a.dev_locs64, r * a.dl_sr + slot * a.dl_ss);
    return row >= 0 && row < a.dev_rows ? row : -1;
}

// The K and V rows of this row's misses, copied by its own workgroup: the
// pieces of all misses (both planes) are dealt to the threads in order,
// 16 KiB of them in flight with 16-byte pieces whatever the workgroup.
template <int kThreads, int kVecWidth>
__device__ __forceinline__ void copy_own_rows(const HsArgs& a, const Lds& s, int32_t misses) {
    using V = typename Vec<kVecWidth>::type;
    constexpr int kLoads = kThreads < 1024 ? 1024 / kThreads : 1;
    const uint32_t per_plane = static_cast<uint32_t>(a.row_bytes / kVecWidth);
    const uint32_t total = static_cast<uint32_t>(misses) * 2u * per_plane;
    for (uint32_t first = 0; first < total; first += kLoads * kThreads) {
        V v[kLoads];
        int64_t dst[kLoads];
        bool copies[kLoads];
#pragma unroll
        for (int k = 0; k < kLoads; ++k) {
            const uint32_t q = first + k * kThreads + threadIdx.x;
            const uint32_t m = q < total ? a.row_div.div(q) : 0u;   // miss rank
            const uint32_t p = q - m * 2u * per_plane;              // piece within the miss's K and V rows
            const int64_t kv = p >= per_plane ? 1 : 0;
            const int64_t within = (static_cast<int64_t>(p) - kv * per_plane) * kVecWidth;
            const int64_t row = s.miss_loc[m];
            copies[k] = q < total && row >= 0;
            dst[k] = kv * a.dev_kv + row * a.dev_rs + within;   // below 0 where V lies before K
            if (copies[k]) {
                const int64_t src = s.lane_val[s.miss_lane[m]];
                v[k] = *reinterpret_cast<const V*>(a.host_k + kv * a.host_kv + src * a.host_rs + within);
            }
        }
#pragma unroll
        for (int k = 0; k < kLoads; ++k) {
            if (copies[k]) {
                *reinterpret_cast<V*>(a.dev_k + dst[k]) = v[k];
            }
        }
    }
}

// One workgroup per batch row holds its CU nearly alone (134 KiB of LDS at the
// largest shape) and is a chain of barriers, so the more waves share its loops the
// shorter it is: kThreads is the smallest size whose threads hold four hot slots
// and two lanes each. 24 rows of 2048 lanes and 4096 slots, none missing: 41.4 us
// with 256 threads, 19.7 us with 1024.
// kCopyWidth: bytes per copy piece when the workgroup copies its row's misses
// itself, 0 when the copy launch does (copies_own_rows decides).
template <int kThreads, int kCopyWidth>
__global__ __launch_bounds__(kThreads) void hisparse_swap_kernel(const HsArgs a) {
    constexpr int kWaves = kThreads / 64;
    extern __shared__ __align__(16) unsigned char shared[];
    const int64_t b = blockIdx.x;
    const int64_t H = a.H, W = a.width;
    Lds s;
    {
        unsigned char* p = shared;
        auto take = [&p](int64_t bytes) {
            unsigned char* at = p;
            p += (bytes + 15) & ~int64_t{15};
            return at;
        };
        s.hash = reinterpret_cast<int32_t*>(take(a.HB * 4));
        s.tok = reinterpret_cast<int32_t*>(take(H * 4));
        s.first_touch = reinterpret_cast<int32_t*>(take(H * 4));
        s.hit_rank = reinterpret_cast<int16_t*>(take(H * 2));
        s.order = reinterpret_cast<int16_t*>(take(H * 2));
        s.victim = reinterpret_cast<int16_t*>(take(W * 2));
        s.miss_lane = reinterpret_cast<int16_t*>(take(W * 2));
        s.lane_rank = reinterpret_cast<int16_t*>(take(W * 2));
        s.lane_tok = reinterpret_cast<int32_t*>(take(W * 4));
        s.lane_aux = reinterpret_cast<int32_t*>(take(W * 4));
        s.lane_pos = reinterpret_cast<int32_t*>(take(W * 4));
        s.lane_val = reinterpret_cast<int32_t*>(take(W * 4));
        s.miss_loc = reinterpret_cast<int32_t*>(take(W * 4));
        s.lane_kind = reinterpret_cast<uint8_t*>(take(W));
        s.scratch = reinterpret_cast<int32_t*>(take((3 * kMaxWaves + 4) * 4));
    }
    int32_t* out = a.out + b * a.out_sb;
    const int64_t real = a.num_real.data != nullptr ? a.num_real[0] : a.batch;
    const int64_t r = a.req[b];
    const int64_t length = a.seq[b];
    if (b >= real || r < 0 || r >= a.R || length <= 0) {
        // Padding row (or a request outside the state): -1 only, state untouched.
        for (int64_t o = threadIdx.x; o < W; o += kThreads) {
            out[o * a.out_so] = -1;
        }
        return;  // uniform over the workgroup
    }
    int32_t* tokens = a.tokens + r * a.tok_sr;

    const void* topk_row = a.topk64 ? static_cast<const void*>(static_cast<const int64_t*>(a.topk) + b * a.topk_sb)
                                    : static_cast<const void*>(static_cast<const int32_t*>(a.topk) + b * a.topk_sb);
    // The row's Top-K ids are requested with its state, which they do not depend on.
    int64_t block[kLanesPerThread];
#pragma unroll
    for (int k = 0; k < kLanesPerThread; ++k) {
        const int64_t o = threadIdx.x + k * kThreads;
        const uint32_t at = static_cast<uint32_t>(o < W ? o : W - 1);
        block[k] = load_index(topk_row, a.topk64, a.block_div.div(at) * a.topk_sk);
    }

    // 1. Load the hot tokens and the LRU order (kBatch loads per thread in
    //    flight at once, clamped indices); build the hash.
    const int64_t reserved = device_row(a, r, H);
    for (int64_t first = 0; first < H; first += kThreads * kBatch) {
        int32_t held[kBatch];
        int64_t listed[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int64_t i = first + k * kThreads + threadIdx.x;
            const int64_t at = i < H ? i : H - 1;
            held[k] = tokens[at * a.tok_ss];
            listed[k] = a.lru32 ? static_cast<const int32_t*>(a.lru)[r * a.lru_sr + at * a.lru_ss]
                                : static_cast<const int16_t*>(a.lru)[r * a.lru_sr + at * a.lru_ss];
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int64_t i = first + k * kThreads + threadIdx.x;
            if (i < H) {
                s.tok[i] = held[k];
                s.first_touch[i] = INT_MAX;
                s.hit_rank[i] = -1;
                s.order[i] = static_cast<int16_t>(listed[k] >= 0 && listed[k] < H ? listed[k] : -1);
            }
        }
    }
    for (int64_t j = threadIdx.x; j < a.HB; j += kThreads) {
        s.hash[j] = kEmpty;
    }
    for (int64_t m = threadIdx.x; m < W; m += kThreads) {
        s.victim[m] = -1;
    }
    __syncthreads();
    for (int64_t i = threadIdx.x; i < H; i += kThreads) {
        const int32_t t = s.tok[i];
        if (t < 0) {
            continue;
        }
        uint32_t h = bucket_of(a, t);
        for (int64_t probe = 0; probe < a.HB; ++probe, h = (h + 1) & static_cast<uint32_t>(a.HB - 1)) {
            int32_t v = load_entry(s, h);
            if (v == kEmpty) {
                v = atomicCAS(&s.hash[h], kEmpty, static_cast<int32_t>(i));
                if (v == kEmpty) {
                    break;
                }
            }
            if (s.tok[v] == t) {
                // The token is in two slots (a state the coordinator does not
                // produce): the lowest slot is the one found.
                atomicMin(&s.hash[h], static_cast<int32_t>(i));
                break;
            }
        }
    }
    __syncthreads();

    // 2. Classify every lane (a thread holds lanes threadIdx.x + kThreads k):
    //    the hash probes (a hit marks its slot, a miss claims a bucket), then
    //    one batch of loads: the device row of each hit, the host row of each
    //    miss.
    {
        uint8_t kinds[kLanesPerThread];
        int32_t auxes[kLanesPerThread];
#pragma unroll
        for (int k = 0; k < kLanesPerThread; ++k) {
            const int64_t o = threadIdx.x + k * kThreads;
            const uint32_t kb = a.block_div.div(static_cast<uint32_t>(o < W ? o : 0));
            int64_t t;
            const bool named = token_position(block[k], a.block_size,
                                              static_cast<uint32_t>(o < W ? o : 0) - kb * a.block_size, a.T,
                                              length < a.T ? length : a.T, t);
            uint8_t kind = kInvalid;
            int32_t aux = -1;
            if (o < W && named) {
                if (t == length - 1) {
                    kind = kNewest;
                } else {
                    s.lane_tok[o] = static_cast<int32_t>(t);
                    __threadfence_block();  // the token is visible before this lane's claim is
                    uint32_t h = bucket_of(a, static_cast<int32_t>(t));
                    for (int64_t probe = 0; probe < a.HB; ++probe, h = (h + 1) & static_cast<uint32_t>(a.HB - 1)) {
                        int32_t v = load_entry(s, h);
                        if (v == kEmpty) {
                            v = atomicCAS(&s.hash[h], kEmpty, static_cast<int32_t>(H + o));
                            if (v == kEmpty) {
                                kind = kMiss;
                                aux = static_cast<int32_t>(h);
                                break;
                            }
                        }
                        // v is set: a resident slot, or a miss claimed by some lane
                        // (lane_tok of a claiming lane is written before its claim).
                        if (v < H) {
                            if (s.tok[v] == t) {
                                kind = kHit;
                                aux = v;
                                atomicMin(&s.first_touch[v], static_cast<int32_t>(o));
                                break;
                            }
                        } else if (s.lane_tok[v - H] == t) {
                            kind = kMiss;
                            aux = static_cast<int32_t>(h);
                            atomicMin(&s.hash[h], static_cast<int32_t>(H + o));
                            break;
                        }
                    }
                }
            }
            kinds[k] = kind;
            auxes[k] = aux;
        }
        // One unconditional load per lane, its address chosen by selects (a
        // branch per kind made the compiler wait for each load before the
        // next): a hit's device row, a miss's host row, otherwise the
        // request's first device row, read and not used.
        int64_t rows[kLanesPerThread];
#pragma unroll
        for (int k = 0; k < kLanesPerThread; ++k) {
            const int64_t o = threadIdx.x + k * kThreads;
            const bool hit = kinds[k] == kHit, miss = kinds[k] == kMiss;
            const int64_t token = s.lane_tok[miss ? o : 0];
            const void* base = miss ? a.host_locs : a.dev_locs;
            const int64_t at = miss ? r * a.hl_sr + token * a.hl_st : r * a.dl_sr + (hit ? int64_t{auxes[k]} : 0) * a.dl_ss;
            const int64_t row = load_index(base, miss ? a.host_locs64 : a.dev_locs64, at);
            rows[k] = hit || miss ? row : -1;
        }
#pragma unroll
        for (int k = 0; k < kLanesPerThread; ++k) {
            const int64_t o = threadIdx.x + k * kThreads;
            if (o < W) {
                uint8_t kind = kinds[k];
                int32_t value = -1;
                if (kind == kHit) {
                    value = rows[k] >= 0 && rows[k] < a.dev_rows ? static_cast<int32_t>(rows[k]) : -1;
                } else if (kind == kMiss) {
                    if (rows[k] >= 0 && rows[k] < a.host_rows) {
                        value = static_cast<int32_t>(rows[k]);
                    } else {
                        kind = kInvalid;  // no host row: every lane of this token sees the same row
                    }
                }
                s.lane_kind[o] = kind;
                s.lane_aux[o] = auxes[k];
                s.lane_val[o] = value;
            }
        }
    }
    __syncthreads();

    // 3. First lanes of each token, ranks in selection order, outputs of the
    //    newest token and of hits. A thread takes a contiguous run of lanes,
    //    counts, scans the counts once over the workgroup, then walks its run.
    int32_t selected, hits, misses;
    {
        const int64_t per = (W + kThreads - 1) / kThreads;
        const int64_t begin = threadIdx.x * per;
        const int64_t end = begin + per < W ? begin + per : W;
        auto first_hit = [&](int64_t o) { return s.lane_kind[o] == kHit && s.first_touch[s.lane_aux[o]] == o; };
        auto first_miss = [&](int64_t o) { return s.lane_kind[o] == kMiss && s.hash[s.lane_aux[o]] == H + o; };
        int32_t count[3] = {0, 0, 0};   // selected, first hits, first misses
        for (int64_t o = begin; o < end; ++o) {
            count[0] += s.lane_kind[o] != kInvalid;
            count[1] += first_hit(o);
            count[2] += first_miss(o);
        }
        int32_t prefix[3], total[3];
        scan_counts<3, kWaves>(count, prefix, total, s.scratch);
        int32_t pos = prefix[0], hit_rank = prefix[1], miss_rank = prefix[2];
        for (int64_t o = begin; o < end; ++o) {
            const uint8_t kind = s.lane_kind[o];
            const int32_t aux = s.lane_aux[o];
            const int32_t value = s.lane_val[o];   // device row of a hit, host row of a miss
            s.lane_pos[o] = kind != kInvalid ? pos : -1;
            if (kind == kNewest) {
                out[pos * a.out_so] = static_cast<int32_t>(reserved);
            } else if (kind == kHit) {
                out[pos * a.out_so] = value;
            }
            pos += kind != kInvalid;
            if (first_hit(o)) {
                s.hit_rank[aux] = static_cast<int16_t>(hit_rank++);
            }
            if (first_miss(o)) {
                s.lane_rank[o] = static_cast<int16_t>(miss_rank);
                s.miss_lane[miss_rank] = static_cast<int16_t>(o);
                ++miss_rank;
            }
        }
        selected = total[0];
        hits = total[1];
        misses = total[2];
    }
    __syncthreads();  // hit_rank and the miss lists are read by other threads below

    // 4. New LRU order and victims, when the row touched the hot buffer. A
    //    thread takes a contiguous run of the old order: counts of its empty
    //    and untouched slots, one scan, then the walk that places them.
    if (hits + misses > 0) {
        const int64_t per = (H + kThreads - 1) / kThreads;
        const int64_t begin = threadIdx.x * per;
        const int64_t end = begin + per < H ? begin + per : H;
        // 0: not listed, 1: touched (hit), 2: empty, 3: untouched occupied.
        auto class_of = [&](int32_t slot) {
            return slot < 0 ? 0 : (s.hit_rank[slot] >= 0 ? 1 : (s.tok[slot] < 0 ? 2 : 3));
        };
        int32_t count[2] = {0, 0};   // empty, untouched
        for (int64_t i = begin; i < end; ++i) {
            const int c = class_of(s.order[i]);
            count[0] += c == 2;
            count[1] += c == 3;
        }
        int32_t prefix[2], total[2];
        scan_counts<2, kWaves>(count, prefix, total, s.scratch);
        const int32_t empty = total[0], untouched = total[1];
        const int32_t taken_empty = misses < empty ? misses : empty;
        const int32_t taken_untouched = misses - taken_empty < untouched ? misses - taken_empty : untouched;
        const int32_t kept_empty = empty - taken_empty, kept_untouched = untouched - taken_untouched;
        const int32_t hit_base = kept_empty + kept_untouched, miss_base = hit_base + hits;
        int32_t e = prefix[0], u = prefix[1];
        for (int64_t i = begin; i < end; ++i) {
            const int32_t slot = s.order[i];
            const int c = class_of(slot);
            int64_t pos = -1;
            if (c == 2) {
                if (e < taken_empty) {
                    s.victim[e] = static_cast<int16_t>(slot);
                    pos = miss_base + e;
                } else {
                    pos = e - taken_empty;
                }
                ++e;
            } else if (c == 3) {
                if (u < taken_untouched) {
                    s.victim[taken_empty + u] = static_cast<int16_t>(slot);
                    pos = miss_base + taken_empty + u;
                } else {
                    pos = kept_empty + (u - taken_untouched);
                }
                ++u;
            } else if (c == 1) {
                pos = hit_base + s.hit_rank[slot];
            }
            if (pos >= 0 && pos < H) {
                if (a.lru32) {
                    static_cast<int32_t*>(a.lru)[r * a.lru_sr + pos * a.lru_ss] = slot;
                } else {
                    static_cast<int16_t*>(a.lru)[r * a.lru_sr + pos * a.lru_ss] = static_cast<int16_t>(slot);
                }
            }
        }
        __syncthreads();  // the victims are read by other threads below

        // 5. Misses take their victims: token table, locations.
        {
            int64_t loc[kLanesPerThread];
#pragma unroll
            for (int k = 0; k < kLanesPerThread; ++k) {
                const int64_t m = threadIdx.x + k * kThreads;
                const int32_t slot = m < misses ? s.victim[m] : -1;
                const int64_t row = device_row(a, r, slot >= 0 ? slot : 0);   // unconditional: loads in flight together
                loc[k] = slot >= 0 ? row : -1;
            }
#pragma unroll
            for (int k = 0; k < kLanesPerThread; ++k) {
                const int64_t m = threadIdx.x + k * kThreads;
                if (m < misses) {
                    const int32_t slot = s.victim[m];
                    if (slot >= 0) {
                        tokens[static_cast<int64_t>(slot) * a.tok_ss] = s.lane_tok[s.miss_lane[m]];
                    }
                    s.miss_loc[m] = static_cast<int32_t>(loc[k]);
                }
            }
        }
        __syncthreads();
    }

    // 6. Outputs of miss lanes and the -1 tail. Without copies of its own, a token's first lane leaves
    //    -2 - (miss rank << kSlotBits | slot) for the copy launch, which copies
    //    the slot's rows and puts its location there; a repeated token takes
    //    the location at once.
    for (int64_t o = threadIdx.x; o < W; o += kThreads) {
        if (s.lane_kind[o] == kMiss) {
            const int32_t owner = s.hash[s.lane_aux[o]] - static_cast<int32_t>(H);
            const int32_t m = s.lane_rank[owner];
            const int32_t loc = s.miss_loc[m];
            const bool left = kCopyWidth == 0 && owner == o && loc >= 0;
            out[s.lane_pos[o] * a.out_so] = left ? -2 - (m << kSlotBits | int32_t{s.victim[m]}) : loc;
        }
    }
    for (int64_t o = selected + threadIdx.x; o < W; o += kThreads) {
        out[o * a.out_so] = -1;
    }
    if constexpr (kCopyWidth > 0) {
        copy_own_rows<kThreads, kCopyWidth>(a, s, misses);
    }
}

// The misses' K and V rows of a few long batch rows, copied from the host cache
// by a launch of its own right behind the swap: the host link bounds it, and
// copy_own_rows keeps 16 KiB per batch row in flight, too little for so few.
// kCopyGroups workgroups of one 16-byte load per lane keep 192 KiB
// in flight, the amount that reached the link's rate for the row moves (57 GB/s).
// A miss to copy is an output entry -2 - (miss rank << kSlotBits | slot), left
// by the swap's step 6. The slot names its token, which names its host row,
// and its device row, which replaces the entry; so the launches share no memory
// beyond the caller's own, in a graph as well. Every workgroup reads all
// entries and takes the misses whose rank plus batch row is its own modulo
// the grid: a row's misses are dealt round robin, whatever block-sized runs
// they come in, and no workgroup acts on an entry that another one replaces.
constexpr int64_t kCopyRows = 8;                     // batch rows of a copy launch at most
constexpr uint32_t kCopyGroups = 48;
constexpr int kCopyThreads = 256;
constexpr int kScan = 16;                            // entries in flight per thread
constexpr uint32_t kRound = kCopyThreads * kScan;    // entries per round of the scan
// Misses a workgroup is dealt at most: every kCopyGroups-th of each row's.
constexpr uint32_t kListed = kCopyRows * ((kMaxLanes + kCopyGroups - 1) / kCopyGroups);
constexpr int kResolve = (kListed + kCopyThreads - 1) / kCopyThreads;   // per thread

template <typename V>
__global__ __launch_bounds__(kCopyThreads) void copy_missed_rows(const HsArgs a, uint32_t entries, FastDiv width_div,
                                                                 FastDiv group_div) {
    constexpr int64_t kWidth = sizeof(V);
    __shared__ uint32_t host_of[kListed];  // entry, then host row (all ones: none)
    __shared__ int32_t dev_of[kListed];    // slot, then device row (-1: none)
    __shared__ uint32_t listed;
    const uint32_t per_plane = static_cast<uint32_t>(a.row_bytes / kWidth);
    if (threadIdx.x == 0) {
        listed = 0;
    }
    __syncthreads();
    for (uint32_t base = 0; base < entries; base += kRound) {
        int32_t held[kScan];
#pragma unroll
        for (int k = 0; k < kScan; ++k) {
            const uint32_t e = base + k * kCopyThreads + threadIdx.x;
            const uint32_t at = e < entries ? e : 0u;
            const uint32_t row = width_div.div(at);
            held[k] = a.out[row * a.out_sb + (at - row * width_div.divisor) * a.out_so];
        }
#pragma unroll
        for (int k = 0; k < kScan; ++k) {
            const uint32_t e = base + k * kCopyThreads + threadIdx.x;
            if (e < entries && held[k] <= -2) {
                const uint32_t code = static_cast<uint32_t>(-2 - held[k]);
                const uint32_t deal = (code >> kSlotBits) + width_div.div(e);
                if (deal - group_div.div(deal) * group_div.divisor == blockIdx.x) {
                    const uint32_t i = atomicAdd(&listed, 1u);
                    host_of[i] = e;
                    dev_of[i] = static_cast<int32_t>(code & ((1u << kSlotBits) - 1));
                }
            }
        }
    }
    __syncthreads();
    const uint32_t n = listed;
    if (n == 0) {
        return;   // uniform
    }
    int64_t request[kResolve], loc[kResolve], host[kResolve];
    int32_t token[kResolve];
    uint32_t entry[kResolve];
#pragma unroll
    for (int k = 0; k < kResolve; ++k) {
        const uint32_t i = k * kCopyThreads + threadIdx.x;
        entry[k] = host_of[i < n ? i : 0u];
        request[k] = a.req[width_div.div(entry[k])];
    }
#pragma unroll
    for (int k = 0; k < kResolve; ++k) {
        const uint32_t i = k * kCopyThreads + threadIdx.x;
        const int64_t slot = dev_of[i < n ? i : 0u];
        token[k] = a.tokens[request[k] * a.tok_sr + slot * a.tok_ss];
        loc[k] = device_row(a, request[k], slot);
    }
#pragma unroll
    for (int k = 0; k < kResolve; ++k) {
        const bool known = token[k] >= 0 && token[k] < a.T;
        const int64_t row = load_index(a.host_locs, a.host_locs64,
                                       known ? request[k] * a.hl_sr + token[k] * a.hl_st : 0);
        host[k] = known && row >= 0 && row < a.host_rows ? row : -1;
    }
    __syncthreads();   // entry 0 stands in for threads past the list until all of them have read it
#pragma unroll
    for (int k = 0; k < kResolve; ++k) {
        const uint32_t i = k * kCopyThreads + threadIdx.x;
        if (i < n) {
            const uint32_t row = width_div.div(entry[k]);
            a.out[row * a.out_sb + (entry[k] - row * width_div.divisor) * a.out_so] = static_cast<int32_t>(loc[k]);
            host_of[i] = static_cast<uint32_t>(host[k]);
            dev_of[i] = static_cast<int32_t>(loc[k]);
        }
    }
    __syncthreads();
    const uint32_t pieces = n * 2u * per_plane;   // below 2^31 (kMaxLanes misses of any row are, checked by the host)
    for (uint32_t q = threadIdx.x; q < pieces; q += kCopyThreads) {
        const uint32_t m = a.row_div.div(q);
        const uint32_t p = q - m * 2u * per_plane;   // piece within the miss's K and V rows
        const int64_t kv = p >= per_plane ? 1 : 0;
        const int64_t within = (static_cast<int64_t>(p) - kv * per_plane) * kWidth;
        const uint32_t src = host_of[m];
        const int64_t dst = dev_of[m];
        if (src != ~0u && dst >= 0) {
            *reinterpret_cast<V*>(a.dev_k + kv * a.dev_kv + dst * a.dev_rs + within) =
                *reinterpret_cast<const V*>(a.host_k + kv * a.host_kv + src * a.host_rs + within);
        }
    }
}
static_assert(kListed <= kMaxLanes, "the listed misses' pieces fit 32 bits when kMaxLanes misses' do");

size_t lds_bytes(int64_t H, int64_t HB, int64_t W) {
    auto round = [](int64_t bytes) { return static_cast<size_t>((bytes + 15) & ~int64_t{15}); };
    return round(HB * 4) + round(H * 4) * 2 + round(H * 2) * 2 + round(W * 2) * 3 + round(W * 4) * 5 + round(W) +
           round((3 * kMaxWaves + 4) * 4);
}

template <int kThreads, int kCopyWidth>
void launch_swap_threads(const HsArgs& a, size_t lds, hipStream_t stream) {
    const auto kernel = hisparse_swap_kernel<kThreads, kCopyWidth>;
    // The LDS limit is raised once per device, to the largest size any call
    // needs, so calls recorded into a graph make no attribute call.
    static std::atomic<bool> raised[kMaxDevices];
    int device = 0;
    check_hip(hipGetDevice(&device), "hipGetDevice");
    if (device < 0 || device >= kMaxDevices) {
        throw std::invalid_argument("device ordinal out of range");
    }
    if (!raised[device].load(std::memory_order_acquire)) {
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds_bytes(kMaxHot, 2 * kMaxHot, kMaxLanes))),
                  "raise the swap-in LDS limit");
        raised[device].store(true, std::memory_order_release);
    }
    kernel<<<dim3(static_cast<uint32_t>(a.batch)), dim3(kThreads), lds, stream>>>(a);
    check_hip(hipGetLastError(), "launch hisparse swap-in");
}

template <int kCopyWidth>
void launch_swap(const HsArgs& a, size_t lds, hipStream_t stream) {
    const int64_t threads = std::max((a.H + kBatch - 1) / kBatch,
                                     (int64_t{a.width} + kLanesPerThread - 1) / kLanesPerThread);
    if (threads <= 256) {
        launch_swap_threads<256, kCopyWidth>(a, lds, stream);
    } else if (threads <= 512) {
        launch_swap_threads<512, kCopyWidth>(a, lds, stream);
    } else {
        launch_swap_threads<1024, kCopyWidth>(a, lds, stream);
    }
}

template <int kVecWidth>
void launch_copy(const HsArgs& a, hipStream_t stream) {
    // The bytes in flight are what counts: narrower pieces take more workgroups.
    const uint32_t groups = kCopyGroups * (16 / kVecWidth);
    copy_missed_rows<typename Vec<kVecWidth>::type><<<dim3(groups), dim3(kCopyThreads), 0, stream>>>(
        a, static_cast<uint32_t>(a.batch * a.width), FastDiv(a.width), FastDiv(groups));
    check_hip(hipGetLastError(), "launch hisparse row copies");
}

// Whether every batch row's workgroup copies its own misses, or a launch of
// its own does: with more than kCopyRows rows the workgroups keep the link busy by
// themselves, and up to kOwnBytes of rows per batch row are copied sooner than
// a second launch has scanned the entries. Measured (us; own copies / copy launch, most lanes
// missing and in brackets none; rows of 512 B):
//   1 x 256 lanes     31.4 / 19.3  (9.9 / 13.3)     1 x 128 lanes    18.5 / 15.9  (8.8 / 11.8)
//   1 x 2048 lanes     123 / 43.5  (17.9 / 20.4)    4 x 128 lanes    21.8 / 20.2  (8.7 / 11.9)
//   8 x 256 lanes     39.7 / 38.7  (11.7 / 14.9)    8 x 128 lanes    23.5 / 24.7  (8.7 / 11.9)
//   8 x 2048 lanes     188 / 169   (19.0 / 25.6)    8 x 64 lanes     18.0 / 19.4  (8.6 / 12.0)
//   16 x 256 lanes    53.6 / 59.9  (11.8 / 14.9)    128 x 256 lanes   307 / 338   (13.9 / 24.8)
//   16 x 2048 lanes    305 / 313   (19.8 / 32.5)    128 x 2048 lanes 2,099 / 2,184 (20.1 / 104)
//   24 x 2048 lanes    433 / 456   (19.7 / 36.6)    256 x 128 lanes   276 / 303   (9.6 / 21.4)
constexpr int64_t kOwnBytes = int64_t{128} << 10;

bool copies_own_rows(const HsArgs& a) {
    return a.batch > kCopyRows || a.width * 2 * a.row_bytes <= kOwnBytes;
}

void need_index2(const ekv_tensor& t, const char* name) {
    need_ndim(t, 2, name);
    need_index(t, name);
}

void need_plane_pair(const ekv_planes* p, const char* name) {
    if (p == nullptr || p->base == nullptr) {
        throw std::invalid_argument(std::string(name) + " is required");
    }
    if (p->layers != 1 || p->kv != 2 || p->rows < 0 || p->row_bytes <= 0 || p->row_stride < p->row_bytes) {
        throw std::invalid_argument(std::string(name) + " must be one layer of K and V planes of whole rows");
    }
    if (p->rows >= (int64_t{1} << 31)) {
        throw std::invalid_argument(std::string(name) + " has more than 2^31 - 1 rows");
    }
}

int hisparse_swap_in(const ekv_tensor* topk_p, const ekv_tensor* tokens_p, const ekv_tensor* host_locs_p,
                     const ekv_tensor* dev_locs_p, const ekv_planes* host, const ekv_planes* dev,
                     const ekv_tensor* out_p, const ekv_tensor* req_p, const ekv_tensor* seq_p,
                     const ekv_tensor* lru_p, int64_t hot, int64_t block_size, const ekv_tensor* num_real_p,
                     void* stream) {
    const ekv_tensor& topk = need(topk_p, "top_k_blocks");
    const ekv_tensor& tokens = need(tokens_p, "device_buffer_tokens");
    const ekv_tensor& host_locs = need(host_locs_p, "host_cache_locs");
    const ekv_tensor& dev_locs = need(dev_locs_p, "device_buffer_locs");
    const ekv_tensor& out = need(out_p, "top_k_device_locs");
    const ekv_tensor& req = need(req_p, "req_pool_indices");
    const ekv_tensor& seq = need(seq_p, "seq_lens");
    const ekv_tensor& lru = need(lru_p, "lru_slots");
    need_plane_pair(host, "host cache");
    need_plane_pair(dev, "device buffer");
    if (host->row_bytes != dev->row_bytes) {
        throw std::invalid_argument("host and device rows differ in size");
    }
    need_index2(topk, "top_k_blocks");
    const int64_t B = topk.shape[0], K = topk.shape[1];
    if (block_size < 1 || block_size > kMaxLanes) {
        throw std::invalid_argument("sparse_block_size must be 1.." + std::to_string(kMaxLanes));
    }
    const int64_t W = K * block_size;
    if (hot < 1 || hot > kMaxHot) {
        throw std::invalid_argument("hot_buffer_size must be 1.." + std::to_string(kMaxHot));
    }
    if (W > kMaxLanes || W > hot) {
        throw std::invalid_argument("Top-K blocks x block size must not exceed hot_buffer_size or " +
                                    std::to_string(kMaxLanes));
    }
    need_ndim(out, 2, "top_k_device_locs");
    if (out.dtype != EKV_INT32) {
        throw std::invalid_argument("top_k_device_locs must be int32");
    }
    need_dim(out, 0, B, "top_k_device_locs");
    need_dim(out, 1, W, "top_k_device_locs");
    need_ndim(tokens, 2, "device_buffer_tokens");
    if (tokens.dtype != EKV_INT32) {
        throw std::invalid_argument("device_buffer_tokens must be int32");
    }
    const int64_t R = tokens.shape[0];
    if (tokens.shape[1] < hot + 1) {
        throw std::invalid_argument("device_buffer_tokens needs hot_buffer_size + 1 columns");
    }
    need_index2(dev_locs, "device_buffer_locs");
    need_dim(dev_locs, 0, R, "device_buffer_locs");
    if (dev_locs.shape[1] < hot + 1) {
        throw std::invalid_argument("device_buffer_locs needs hot_buffer_size + 1 columns");
    }
    need_index2(host_locs, "host_cache_locs");
    need_dim(host_locs, 0, R, "host_cache_locs");
    const int64_t T = host_locs.shape[1];
    if (T >= (int64_t{1} << 31)) {
        throw std::invalid_argument("host_cache_locs has more than 2^31 - 1 tokens per request");
    }
    need_ndim(lru, 2, "lru_slots");
    if (lru.dtype != EKV_INT16 && lru.dtype != EKV_INT32) {
        throw std::invalid_argument("lru_slots must be int16 or int32");
    }
    need_dim(lru, 0, R, "lru_slots");
    need_dim(lru, 1, hot, "lru_slots");
    for (const auto* one : {&req, &seq}) {
        need_ndim(*one, 1, "req_pool_indices/seq_lens");
        need_index(*one, "req_pool_indices/seq_lens");
        need_dim(*one, 0, B, "req_pool_indices/seq_lens");
    }
    IndexRef num_real;
    if (num_real_p != nullptr) {
        const ekv_tensor& n = need(num_real_p, "num_real_reqs");
        need_index(n, "num_real_reqs");
        if (numel(n) != 1 || n.data == nullptr) {
            throw std::invalid_argument("num_real_reqs must hold one element");
        }
        num_real = index_ref(n, 0);
    }
    if (B == 0 || W == 0) {
        return 0;
    }
    if (B > 0x7fffffff) {
        throw std::invalid_argument("too many rows for one launch");
    }
    for (const auto* t : {&topk, &tokens, &host_locs, &dev_locs, &out, &req, &seq, &lru}) {
        need_data(*t, "tensor");
    }
    HsArgs a{};
    a.topk = topk.data;
    a.topk64 = topk.dtype == EKV_INT64;
    a.topk_sb = topk.stride[0], a.topk_sk = topk.stride[1];
    a.tokens = static_cast<int32_t*>(tokens.data);
    a.tok_sr = tokens.stride[0], a.tok_ss = tokens.stride[1];
    a.host_locs = host_locs.data;
    a.host_locs64 = host_locs.dtype == EKV_INT64;
    a.hl_sr = host_locs.stride[0], a.hl_st = host_locs.stride[1];
    a.dev_locs = dev_locs.data;
    a.dev_locs64 = dev_locs.dtype == EKV_INT64;
    a.dl_sr = dev_locs.stride[0], a.dl_ss = dev_locs.stride[1];
    a.lru = lru.data;
    a.lru32 = lru.dtype == EKV_INT32;
    a.lru_sr = lru.stride[0], a.lru_ss = lru.stride[1];
    a.out = static_cast<int32_t*>(out.data);
    a.out_sb = out.stride[0], a.out_so = out.stride[1];
    a.req = index_ref(req, 0);
    a.seq = index_ref(seq, 0);
    a.num_real = num_real;
    a.host_k = static_cast<const char*>(host->base);
    a.host_kv = host->kv_stride, a.host_rs = host->row_stride, a.host_rows = host->rows;
    a.dev_k = static_cast<char*>(dev->base);
    a.dev_kv = dev->kv_stride, a.dev_rs = dev->row_stride, a.dev_rows = dev->rows;
    a.row_bytes = dev->row_bytes;
    a.batch = B, a.R = R, a.T = T, a.H = hot;
    a.HB = 1;
    while (a.HB < 2 * hot) {
        a.HB <<= 1;
    }
    int log2 = 0;
    while ((int64_t{1} << log2) < a.HB) {
        ++log2;
    }
    a.hb_shift = static_cast<uint32_t>(32 - log2);
    if (log2 == 0) {
        a.hb_shift = 31;  // HB = 1 cannot happen (hot >= 1 gives HB >= 2); kept well defined
    }
    a.width = static_cast<uint32_t>(W);
    a.block_size = static_cast<uint32_t>(block_size);
    a.block_div = FastDiv(static_cast<uint32_t>(block_size));
    const size_t lds = lds_bytes(hot, a.HB, W);
    // Widest copy unit dividing the row size, the row strides, the plane
    // offsets and both base addresses.
    const int vw = pick_vector_width({a.row_bytes, a.host_rs, a.dev_rs, a.host_kv, a.dev_kv,
                                      static_cast<int64_t>(reinterpret_cast<uintptr_t>(a.host_k)),
                                      static_cast<int64_t>(reinterpret_cast<uintptr_t>(a.dev_k))});
    const auto st = static_cast<hipStream_t>(stream);
    const int64_t pieces = 2 * (a.row_bytes / vw);
    if (pieces * kMaxLanes >= (int64_t{1} << 31)) {
        throw std::invalid_argument("rows too large for one swap-in (copy pieces exceed 2^31)");
    }
    a.row_div = FastDiv(static_cast<uint32_t>(pieces));
    if (copies_own_rows(a)) {
        switch (vw) {
            case 16: launch_swap<16>(a, lds, st); break;
            case 8: launch_swap<8>(a, lds, st); break;
            case 4: launch_swap<4>(a, lds, st); break;
            case 2: launch_swap<2>(a, lds, st); break;
            default: launch_swap<1>(a, lds, st); break;
        }
        return 0;
    }
    launch_swap<0>(a, lds, st);
    if (R == 0 || T == 0) {
        return 0;   // no row has state or no token a host row: nothing missed
    }
    switch (vw) {
        case 16: launch_copy<16>(a, st); break;
        case 8: launch_copy<8>(a, st); break;
        case 4: launch_copy<4>(a, st); break;
        case 2: launch_copy<2>(a, st); break;
        default: launch_copy<1>(a, st); break;
    }
    return 0;
}

}  // namespace
}  // namespace ekv

extern "C" int ekv_hisparse_swap_in(const ekv_tensor* top_k_blocks, const ekv_tensor* device_buffer_tokens,
                                    const ekv_tensor* host_cache_locs, const ekv_tensor* device_buffer_locs,
                                    const ekv_planes* host_cache, const ekv_planes* device_buffer,
                                    const ekv_tensor* top_k_device_locs, const ekv_tensor* req_pool_indices,
                                    const ekv_tensor* seq_lens, const ekv_tensor* lru_slots,
                                    int64_t hot_buffer_size, int64_t sparse_block_size,
                                    const ekv_tensor* num_real_reqs, void* stream) {
    return ekv::guarded(-1, [&] {
        return ekv::hisparse_swap_in(top_k_blocks, device_buffer_tokens, host_cache_locs, device_buffer_locs,
                                     host_cache, device_buffer, top_k_device_locs, req_pool_indices, seq_lens,
                                     lru_slots, hot_buffer_size, sparse_block_size, num_real_reqs, stream);
    });
}

extern "C" int ekv_host_device_pointer(void* host, void** device) {
    return ekv::guarded(-1, [&] {
        if (host == nullptr || device == nullptr) {
            throw std::invalid_argument("host and device pointers are required");
        }
        ekv::check_hip(hipHostGetDevicePointer(device, host, 0),
                       "hipHostGetDevicePointer (the memory must be pinned host memory)");
        return 0;
    });
}
