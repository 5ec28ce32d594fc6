// Hot-buffer swap-in with batch-token LRU replacement (gfx950).
//
// Policy: benchmarks/hisparse_locality_replay.py:90-99 - per (request, layer)
// stream, misses are counted at entry, hits are touched (moved to most recent,
// in selection order), least-recent entries are evicted until the misses fit,
// then the misses are inserted in selection order. Here the hot buffer of a
// (layer, request) row is `capacity` slots; the reference's ordered dict is
// represented by one recency stamp per slot:
//   touched hit of lane o at step s: stamp = s * 8192 + o
//   inserted miss of lane o:         stamp = s * 8192 + 4096 + o
//   empty slot:                      stamp = INT32_MIN
// (a row has at most 4096 lanes, so every step's stamps lie above all of the
// steps before it whatever the width of each call), so sorting slots by
// (stamp, slot) reproduces the dict's order, and the m victims of a step
// (m = distinct missed tokens) are the slots of the m smallest keys: empty
// slots first, then the least recently used entries.
//
// Repeated tokens. The reference's replay refuses a selection that repeats a
// token (hisparse_locality_replay.py:55-56), but Top-K blocks expand to
// repeats when a block id appears twice (the access-trace KAT
// tests/test_hisparse_access_trace.py:170-199 selects [2, 3, 6, 2, 3]). This
// kernel defines a repeated token as one access by its first lane - the
// replay applied to the selection with later repeats dropped: a hit's stamp
// takes its lowest lane (atomicMin in LDS), a repeated miss takes one victim
// (an LDS hash of the miss tokens names each token's first miss), and its
// later lanes share that slot and record empty promotions.
//
// One workgroup per (row, layer): hits are touched in LDS, a
// radix select over the stamps finds the victims (the slots of the smallest
// (stamp, slot) keys), which one scan lists in slot order; the i-th distinct
// miss (in miss-list order) takes the i-th of them. (Which victim slot a
// miss takes is this kernel's own convention: the reference's LRU is an
// ordered dict of tokens, whose contents and order do not depend on it.)
// Each victim clears its old token from the token->slot table and residency
// summary, takes the new token, and writes one promotion (host row -> global
// slot) record. The lookup's slot output of every miss lane is patched to its
// new slot, so the gather that follows reads the promoted row.
//
// Residency summary. At bits_shift 0 a bit is one position: an evicted
// token clears it, an inserted token sets it. A coarser bit covers 2^shift
// positions; with per-bit resident counts the summary stays exact: a group's
// evictions and insertions change its count, and its bit is cleared when the
// count reaches zero and set when it leaves zero. Without counts a coarse
// bit is only ever set, and the summary is a superset of the table. A row's
// words (or changes of counts) are gathered in LDS and written once: the row
// belongs to this workgroup. As an atomic per eviction and insertion they
// were a quarter of the call at 2560 rows (178.6 against 133.5 us). Rows too
// long for LDS still take atomics, evictions before a barrier, insertions after it, so
// that no clear can follow a set.
//
// Refused rows. Two selected rows naming one request would race on its hot
// buffer, and a step whose stamps would overflow int32 cannot be ordered:
// such a row changes nothing, records empty promotions and ORs
// EKV_SWAP_SHARED_REQUEST or EKV_SWAP_STAMP_OVERFLOW into the caller's
// status word, which the host reads back.
#include "../../include/ekv_kernels.h"
#include "ekv_common.h"
#include "ekv_fastdiv.h"
#include "ekv_step.h"
#include "ekv_tensor_util.h"
#include "ekv_token.h"
#include "ekv_wave.h"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace ekv {
namespace {

constexpr int kMaxCapacity = 8192;   // slots per hot buffer (touches held in LDS; 16-bit scan fields)
constexpr int kMaxWidth = 4096;      // lanes per row whose miss tokens are hashed in LDS
constexpr int kDigits = 256;         // of one radix-select pass
// Summary words (bits_shift 0), or groups of a coarse summary, that a row's changes are gathered over in LDS: 8 KiB,
// contexts of 65,536 tokens at bits_shift 0 and 131,072 at 6. Longer rows take global atomics.
constexpr int64_t kMaxGathered = 2048;
// Stamps per LRU step: hits take step * kStepStamps + lane, misses
// step * kStepStamps + kMaxWidth + lane, so a call with fewer lanes than the
// one before still stamps above it.
constexpr int64_t kStepStamps = EKV_SWAP_STEP_STAMPS;
static_assert(kStepStamps == 2 * kMaxWidth, "hit and miss stamps of one step take 2 * kMaxWidth values");
constexpr int32_t kStatusStampOverflow = EKV_SWAP_STAMP_OVERFLOW;
constexpr int32_t kStatusSharedRequest = EKV_SWAP_SHARED_REQUEST;

struct SwapArgs {
    const void* topk;
    int32_t topk64;
    int64_t topk_sl, topk_sb, topk_sk;
    uint32_t block_size;
    FastDiv block_div;
    IndexRef rows, selected, slot_base;
    int64_t selected_count;
    int32_t* slots;                 // [L, B, W] lookup output, patched for misses
    int64_t sl_l, sl_b, sl_o;
    const int32_t* misses;          // [L, B, W] miss lanes
    int64_t mi_l, mi_b, mi_o;
    int32_t* counts;                // [L, B]
    IndexRef lengths;               // [B], when the lookup runs in the same launch
    int64_t ct_l, ct_b;
    void* table;                    // [L, R, T] token -> global slot (int32) or local slot + 1 (int16); 0 = not resident
    int32_t table16;
    int64_t tb_l, tb_r, tb_t, table_cols;
    int32_t* bits;                  // [L, R, words] residency summary (may be null)
    int64_t bt_l, bt_r, bt_w;
    uint32_t bits_shift;            // bit q covers positions [q << shift, (q + 1) << shift)
    int32_t* line_counts;           // [L, R, groups] resident positions per summary bit (bits_shift > 0; may be null)
    int64_t lc_l, lc_r, lc_q;
    int32_t* slot_token;            // [L, R, C] token held by each slot (-1 = empty)
    int64_t st_l, st_r, st_c;
    int32_t* stamps;                // [L, R, C] recency stamps
    int64_t sp_l, sp_r, sp_c;
    IndexRef host_table;            // [R, T] token -> host row, addressed with explicit strides
    int64_t host_sr, host_st;
    int32_t* promote_src;           // [L, B, W] host row per promotion
    int64_t ps_l, ps_b, ps_o;
    int32_t* promote_dst;           // [L, B, W] global slot per promotion
    int64_t pd_l, pd_b, pd_o;
    int64_t batch, table_rows, capacity;
    uint32_t width;
    int64_t step;
    const int64_t* step_counter;    // when set, the step is read from device memory (graph replays)
    int32_t* status;                // EKV_SWAP_* error bits, OR-ed in (may be null)
    uint32_t gathered;              // summary words (bits_shift 0) or line_counts groups kept in LDS (0: global atomics)
    uint32_t info_words;            // words of the info region
    uint32_t hash_size, hash_log2;  // miss-token hash buckets: a power of two >= 2W (and >= 2)
    uint32_t token_bitmap;          // 1: the region first serves as a token bitmap
    uint32_t bitmap_words;          // ceil(T / 32)
};

// Element i of a row at `row`. Dense rows (unit strides, byte extents below
// 4 GiB, checked by the host) take a 32-bit byte offset from the
// workgroup-uniform row; other rows a 64-bit product per access, of which a
// row of 4096 slots needs about sixty per thread.
template <bool kDense, typename T>
__device__ __forceinline__ T* element(T* row, int64_t stride, uint32_t i) {
    if constexpr (kDense) {
        using Byte = std::conditional_t<std::is_const_v<T>, const char, char>;
        return reinterpret_cast<T*>(reinterpret_cast<Byte*>(row) + i * static_cast<uint32_t>(sizeof(T)));
    } else {
        return row + static_cast<int64_t>(i) * stride;
    }
}

// The low 32 bits of element i of an int32 or int64 row, or (`high`) its high ones; no branch on the element type.
template <bool kDense>
__device__ __forceinline__ int32_t index_word(const void* row, int32_t is64, int64_t stride, uint32_t i, bool high) {
    const char* at = static_cast<const char*>(row);
    if constexpr (kDense) {
        return *reinterpret_cast<const int32_t*>(at + ((i << (is64 ? 3 : 2)) + (high ? 4u : 0u)));
    } else {
        return *reinterpret_cast<const int32_t*>(at + i * stride * (is64 ? 8 : 4) + (high ? 4 : 0));
    }
}

// Writes a token -> slot table entry (int32 global slot or int16 local slot + 1) of the row starting at element `row`.
template <bool kDense>
__device__ __forceinline__ void set_entry(const SwapArgs& a, int64_t row, uint32_t token, int32_t value) {
    if (a.table16) {
        *element<kDense>(static_cast<int16_t*>(a.table) + row, a.tb_t, token) = static_cast<int16_t>(value);
    } else {
        *element<kDense>(static_cast<int32_t*>(a.table) + row, a.tb_t, token) = value;
    }
}

// A workgroup barrier that orders LDS only: waves wait for their own LDS
// accesses, not for their outstanding global stores (which a full
// __syncthreads would also wait for).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Lanes of this wave below the calling lane whose bit is set in `mask`.
__device__ __forceinline__ int32_t lanes_below(uint64_t mask) {
    return static_cast<int32_t>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                                          __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u)));
}

// True in every thread when `value` is true in any. Every thread must call it
// (one LDS barrier); `cells` holds one word per wave, used by this call only.
template <int kWaves>
__device__ __forceinline__ bool workgroup_any(bool value, uint32_t* cells) {
    const uint32_t lane = threadIdx.x & 63;
    const bool any = __ballot(value) != 0;
    if (lane == 0) {
        cells[threadIdx.x >> 6] = any ? 1u : 0u;
    }
    lds_barrier();
    return __ballot(lane < kWaves && cells[lane < kWaves ? lane : 0] != 0) != 0;
}

// Sum, minimum and maximum of one value per thread over the workgroup, added
// to range[0..2] (starting at 0, all ones and 0) by each wave's last lane; read
// them after a barrier. Every thread must call it.
__device__ __forceinline__ void add_range(uint32_t sum, uint32_t lo, uint32_t hi, uint32_t* range) {
    sum = wave_scan<kAdd>(sum);
    lo = wave_scan<kMin>(lo);
    hi = wave_scan<kMax>(hi);
    if ((threadIdx.x & 63) == 63) {
        atomicAdd(&range[0], sum);
        atomicMin(&range[1], lo);
        atomicMax(&range[2], hi);
    }
}

__device__ __forceinline__ uint32_t token_hash(int32_t token, uint32_t log2_size) {
    return (static_cast<uint32_t>(token) * 2654435761u) >> (32 - log2_size);
}

// Packed 16-bit buckets of the miss-token hash: bucket h is the half
// (h & 1) of word h >> 1; 0xffff marks an empty bucket, otherwise the bucket
// holds a miss index (< 4096).
constexpr uint32_t kEmptyBucket = 0xffffu;

__device__ __forceinline__ uint32_t bucket_of(const uint32_t* words, uint32_t h) {
    return (words[h >> 1] >> ((h & 1u) * 16u)) & 0xffffu;
}

// Writes `value` into bucket h when the bucket holds `expected`; the other
// half of the word is preserved (retried while another lane changes it).
// Returns the bucket's value before the write, or its current value when it
// no longer held `expected`.
__device__ __forceinline__ uint32_t bucket_cas(uint32_t* words, uint32_t h, uint32_t expected, uint32_t value) {
    const uint32_t shift = (h & 1u) * 16u;
    uint32_t* word = words + (h >> 1);
    uint32_t seen = *word;
    while (true) {
        const uint32_t held = (seen >> shift) & 0xffffu;
        if (held != expected) {
            return held;
        }
        const uint32_t desired = (seen & ~(0xffffu << shift)) | (value << shift);
        const uint32_t previous = atomicCAS(word, seen, desired);
        if (previous == seen) {
            return expected;
        }
        seen = previous;   // the word changed (this bucket or its neighbour): look again
    }
}

// Lowers bucket h to `value` when that is smaller (a 16-bit atomicMin).
__device__ __forceinline__ void bucket_min(uint32_t* words, uint32_t h, uint32_t value) {
    uint32_t held = bucket_of(words, h);
    while (value < held) {
        const uint32_t seen = bucket_cas(words, h, held, value);
        if (seen == held) {
            return;
        }
        held = seen;
    }
}

// Open-addressing hash of the miss tokens: every token ends up in one bucket
// holding its lowest miss index. The table holds at least 2m buckets, so
// every probe meets its token or an empty bucket. Every thread must call it.
__device__ __forceinline__ void hash_miss_tokens(uint32_t* hash, const int32_t* info, int32_t m, uint32_t log2_size) {
    const uint32_t mask = (1u << log2_size) - 1u;
    for (int32_t i = threadIdx.x; i < m; i += blockDim.x) {
        const int32_t token = info[i];
        if (token < 0) {
            continue;
        }
        uint32_t h = token_hash(token, log2_size);
        while (true) {
            const uint32_t held = bucket_cas(hash, h, kEmptyBucket, static_cast<uint32_t>(i));
            if (held == kEmptyBucket) {
                break;   // claimed
            }
            if (info[held] == token) {
                bucket_min(hash, h, static_cast<uint32_t>(i));
                break;
            }
            h = (h + 1) & mask;
        }
    }
}

// Dynamic LDS of one workgroup (C = capacity, W = lanes per row):
//   touch    int32 [C]  lowest lane that hits the slot (INT32_MAX: none), then the new stamp of a victim;
//   info     int32 [W]  when tokens repeat: token of miss i (-1: an entry naming no valid lane),
//            then int16 [W], the victim's rank of a first miss, and behind it
//   summary  int32 [gathered]  the row's summary words, or the changes of its groups' counts;
//   region   the token bitmap, or hash_size 16-bit buckets (the miss-token hash), then the int16
//            list of the victims' slots in slot order;
//
// What bounds it. A row is a chain of about ten barrier-separated phases over
// a few KiB of LDS, so what counts is how short a phase's code is and how many waves
// share it: a thread holds kSlotRegs stamps and kLaneRegs lanes in registers,
// and the host picks the workgroup size that gives four and two (threads of
// 64 to 1024). With 256 threads for every shape a row of 4096 slots was 16
// and 8 registers of unrolled code, 53 KB of instructions fetched once per
// row, and the same code ran for a row of 256 slots. Scans are DPP steps,
// the summary is changed in LDS and written once, and dense rows are addressed
// with 32-bit offsets. The swap alone, against those 256 threads and global
// atomics: 48 rows of 1024 lanes (2048 slots) 23.1 -> 12.8 us, 2560 rows of 256 lanes
// 67.1 -> 24.7, of 2048 lanes 183.7 -> 115.0; 1280 rows of 4096 lanes and 8192 slots
// 262 -> 163 with the lookup. The 2560 x 2048 launch moves 246 MB from and
// 215 MB to HBM by the counters (scattered table entries as whole lines), 84 us
// at the rate of a copy.
//
// Global reads come in three batches, each issued as a fixed number of
// unrolled loads from clamped, in-bounds addresses and waited for once: the
// stamps, lookup slots and miss list (with the request checks); the Top-K
// ids of the miss entries; the victims' old tokens and host rows. (A loop
// with a run-time trip count waits for each load before issuing the next: a
// workgroup then spends most of its life on a chain of HBM round trips.)
//
// kLookup: the lookup of the rows runs here as well (the one-call decode step).
// A thread's lanes then are their own miss entries: their Top-K ids are read
// in the prologue, their table entries in place of the lookup's slots (no summary: what it
// could spare is the entry reads of the misses), the misses are ranked over the
// barrier of the request check, and slots and miss count are written here. It saves the
// lookup's launch and chain of reads, and the slots and miss list through memory.
// In the decode step of 8 rows of 64 lanes: 12.2 us, where the two kernels took
// 6.3 and 13.0.
template <int kThreads, int kSlotRegs, int kLaneRegs, bool kDense, bool kLookup>
__global__ __launch_bounds__(kThreads) void swap_in_kernel(const SwapArgs a) {
    constexpr int kWaves = kThreads / 64;
    constexpr uint32_t kReadAhead = 4;     // summary words or group counts per thread that are read ahead
    extern __shared__ __align__(16) unsigned char shared[];
    __shared__ __align__(16) int32_t digit_count[2 * kDigits];   // radix-select histograms of two passes
    __shared__ uint32_t key_range[3];      // empties, smallest and largest other key
    __shared__ uint32_t first_cells[kLaneRegs * kWaves], victim_cells[kSlotRegs * kWaves];
    __shared__ uint32_t any_cells[2][kWaves];
    __shared__ uint32_t miss_cells[kLookup ? kLaneRegs * kWaves : 1];
    int32_t* touch = reinterpret_cast<int32_t*>(shared);
    int32_t* info = touch + a.capacity;
    int16_t* owner = reinterpret_cast<int16_t*>(info);   // the tokens are in registers again by then
    int32_t* summary = info + (a.width + 1) / 2;
    uint32_t* hash = reinterpret_cast<uint32_t*>(info + a.info_words);
    int16_t* victims = reinterpret_cast<int16_t*>(hash);
    // The prologue's reads are vector loads issued together: as scalar loads
    // (uniform reads) the compiler waited for each before the next one, and
    // the selection entry, request row, miss count, step and slot base were a
    // chain of round trips. The request row and miss count are read on the
    // guess that the selection is the identity (entry j names batch row j:
    // every batch row, the decode default); a different entry re-reads them
    // for its row. The slot base is read beside batch 1, with whose results
    // it is first needed.
    const uint32_t zero = opaque_zero();
    const int64_t l = blockIdx.y;
    const int64_t guess = blockIdx.x < a.batch ? blockIdx.x : 0;
    const PendingIndex entry_read = issue_index(a.selected, blockIdx.x, zero);
    const PendingIndex req_read = issue_index(a.rows, guess, zero);
    int32_t counted_read = 0;
    PendingIndex length_read{0, 0};
    int32_t block_low[kLaneRegs], block_high[kLaneRegs];   // Top-K ids of this thread's lanes, or of its miss entries
    const auto topk_row_of = [&](int64_t row) {
        return a.topk64 ? static_cast<const void*>(static_cast<const int64_t*>(a.topk) + l * a.topk_sl + row * a.topk_sb)
                        : static_cast<const void*>(static_cast<const int32_t*>(a.topk) + l * a.topk_sl + row * a.topk_sb);
    };
    const auto read_id = [&](const void* topk_row, uint32_t lane, int k) {
        const uint32_t blk = a.block_size == 1 ? lane : a.block_div.div(lane);
        block_low[k] = index_word<kDense>(topk_row, a.topk64, a.topk_sk, blk, false);
        block_high[k] = index_word<kDense>(topk_row, a.topk64, a.topk_sk, blk, a.topk64 != 0);
    };
    if constexpr (kLookup) {
        length_read = issue_index(a.lengths, guess, zero);
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            read_id(topk_row_of(guess), min(threadIdx.x + k * kThreads, a.width - 1), k);
        }
    } else {
        counted_read = a.counts[l * a.ct_l + guess * a.ct_b + zero];
    }
    // The device step of a graph replay; without one, a word of the counts
    // stands in and is not used.
    const bool device_step = a.step_counter != nullptr;   // uniform
    const int32_t* step_words = device_step ? reinterpret_cast<const int32_t*>(a.step_counter) : a.counts;
    const int32_t step_lo = step_words[zero];
    const int32_t step_hi = step_words[(device_step ? 1u : 0u) + zero];
    // Every value is read back before the first early return, so the loads
    // stay together (the compiler moves a load whose uses all lie past a
    // return below it, where it waits for it alone).
    const int64_t b = index_value(a.selected, entry_read);
    int64_t req = index_value(a.rows, req_read);
    int32_t counted = __builtin_amdgcn_readfirstlane(counted_read);
    int64_t length = kLookup ? index_value(a.lengths, length_read) : 0;
    const int64_t step =
        device_step ? static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(
                                                __builtin_amdgcn_readfirstlane(step_hi))) << 32) |
                                           static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(step_lo)))
                    : a.step;   // uniform
    const bool live = b >= 0 && b < a.batch;   // uniform
    if (live && b != guess) {   // uniform: the selection is not the identity here
        req = a.rows.fetch(b);
        if constexpr (kLookup) {
            length = a.lengths.fetch(b);
#pragma unroll
            for (int k = 0; k < kLaneRegs; ++k) {
                read_id(topk_row_of(b), min(threadIdx.x + k * kThreads, a.width - 1), k);
            }
        } else {
            counted = a.counts[l * a.ct_l + b * a.ct_b];
        }
    }
    if (!live || req < 0 || req >= a.table_rows) {
        if constexpr (kLookup) {
            if (live) {   // uniform: no lane of it is valid
                for (uint32_t o = threadIdx.x; o < a.width; o += kThreads) {
                    *element<kDense>(a.slots + l * a.sl_l + b * a.sl_b, a.sl_o, o) = -1;
                }
                if (threadIdx.x == 0) {
                    a.counts[l * a.ct_l + b * a.ct_b] = 0;
                }
            }
        }
        return;  // uniform: a stray selection, or a row outside the tables (nothing resident)
    }
    const int64_t C = a.capacity;
    const int64_t W = a.width;
    const PendingIndex base_read = issue_index(a.slot_base, req, zero);
    int32_t* promote_src = a.promote_src + l * a.ps_l + b * a.ps_b;
    int32_t* promote_dst = a.promote_dst + l * a.pd_l + b * a.pd_b;
    int32_t* slots = a.slots + l * a.sl_l + b * a.sl_b;
    const int64_t table_row = l * a.tb_l + req * a.tb_r;   // element offset of this (layer, request) row
    int32_t* slot_token = a.slot_token + l * a.st_l + req * a.st_r;
    int32_t* stamps = a.stamps + l * a.sp_l + req * a.sp_r;
    const int32_t* misses = a.misses + l * a.mi_l + b * a.mi_b;

    // One workgroup owns each (layer, request) hot buffer: a second selected
    // row naming the same request would race on it, so both rows are refused.
    // Thread t checks selection entry t (and t + kThreads, ... for longer
    // selections). Vector loads complete in issue order, so entry t is read
    // before batch 1 and its request row right after batch 1 is issued: batch 2
    // then waits for batch 1 alone, not for two dependent reads behind it.
    const int64_t selected_count = a.selected_count;   // at least 1
    const int64_t first_j = threadIdx.x;
    const int64_t first_other = a.selected.fetch(first_j < selected_count ? first_j : selected_count - 1);
    // Batch 1: stamps, the lookup slots of this thread's lanes, its miss-list entries.
    int32_t held_stamp[kSlotRegs];
#pragma unroll
    for (int k = 0; k < kSlotRegs; ++k) {
        const uint32_t s = min(threadIdx.x + k * kThreads, static_cast<uint32_t>(C) - 1);
        held_stamp[k] = *element<kDense>(stamps, a.sp_c, s);
    }
    int32_t lane_slot[kLaneRegs];   // kLookup: the table entry until the base is known
    int32_t miss_lane[kLaneRegs];   // lane of this thread's k-th entry (kLookup: its k-th lane)
    bool valid_lane[kLaneRegs];     // kLookup
    int64_t lane_token[kLaneRegs];
    // The token of an entry: its block id times the block size, and the lane's place in the block; outside
    // [0, table_cols) when it names none.
    const auto token_at = [&](int k, int32_t lane) {
        const int32_t high = a.topk64 ? block_high[k] : block_low[k] >> 31;
        int64_t token = static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(high)) << 32 |
                                             static_cast<uint32_t>(block_low[k]));
        if (a.block_size != 1) {   // uniform
            const uint32_t offset =
                static_cast<uint32_t>(lane) - a.block_div.div(static_cast<uint32_t>(lane)) * a.block_size;
            int64_t position;
            token = token_position(token, a.block_size, offset, a.table_cols, a.table_cols, position) ? position : -1;
        }
        return token;
    };
    if constexpr (kLookup) {
        const int64_t bound = length < a.table_cols ? length : a.table_cols;
        uint32_t at[kLaneRegs];
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            miss_lane[k] = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            lane_token[k] = token_at(k, miss_lane[k]);
            valid_lane[k] = miss_lane[k] < W && lane_token[k] >= 0 && lane_token[k] < bound;
            at[k] = valid_lane[k] ? static_cast<uint32_t>(lane_token[k]) : 0u;
        }
        if (a.table16) {   // uniform
#pragma unroll
            for (int k = 0; k < kLaneRegs; ++k) {
                lane_slot[k] = *element<kDense>(static_cast<const int16_t*>(a.table) + table_row, a.tb_t, at[k]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < kLaneRegs; ++k) {
                lane_slot[k] = *element<kDense>(static_cast<const int32_t*>(a.table) + table_row, a.tb_t, at[k]);
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const uint32_t o = min(threadIdx.x + k * kThreads, a.width - 1);
            lane_slot[k] = *element<kDense>(slots, a.sl_o, o);
            miss_lane[k] = *element<kDense>(misses, a.mi_o, o);   // entries at or past the count are read but not used
        }
    }
    const bool first_in_range =
        first_j < selected_count && first_j != blockIdx.x && first_other >= 0 && first_other < a.batch;
    const int64_t first_req = a.rows.fetch(first_in_range ? first_other : b);   // b is a valid batch row
    bool shared_request = first_in_range && first_req == req;
    for (int64_t j = first_j + kThreads; j < selected_count; j += kThreads) {
        const int64_t other = a.selected[j];
        shared_request |= j != blockIdx.x && other >= 0 && other < a.batch && a.rows[other] == req;
    }
    // Batch 2: the Top-K ids of the miss entries.
    if constexpr (!kLookup) {
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            read_id(topk_row_of(b), static_cast<uint32_t>(min(max(miss_lane[k], 0), static_cast<int32_t>(W - 1))), k);
        }
    }
    int32_t m = counted < 0 ? 0 : (counted > W ? static_cast<int32_t>(W) : counted);
    // LDS starts, published by the barrier of the request check: nothing touched, the region a token bitmap (all clear)
    // when the tokens fit it, else the empty hash.
#pragma unroll
    for (int k = 0; k < kSlotRegs; ++k) {
        const uint32_t s = threadIdx.x + k * kThreads;
        if (s < C) {
            touch[s] = INT32_MAX;
        }
    }
    const uint32_t region_words = a.token_bitmap ? a.bitmap_words : a.hash_size / 2;
    const uint32_t region_fill = a.token_bitmap ? 0u : 0xffffffffu;
    for (uint32_t w = threadIdx.x; w < region_words; w += kThreads) {
        hash[w] = region_fill;
    }
    for (uint32_t d = threadIdx.x; d < 2 * kDigits; d += kThreads) {
        digit_count[d] = 0;
    }
    if (threadIdx.x < 3) {
        key_range[threadIdx.x] = threadIdx.x == 1 ? 0xffffffffu : 0u;
    }
    // The row's summary words, or its groups' counts, read ahead of their use.
    int32_t* bits = a.bits != nullptr ? a.bits + l * a.bt_l + req * a.bt_r : nullptr;
    // Group counts keep a coarse summary exact: their changes gathered in LDS and applied once per group, or
    // decremented and incremented in place around a barrier.
    int32_t* line_counts = bits != nullptr && a.bits_shift > 0 && a.line_counts != nullptr
                               ? a.line_counts + l * a.lc_l + req * a.lc_r
                               : nullptr;
    const uint32_t gathered = a.gathered;   // 0 without a summary
    int32_t* const state = line_counts != nullptr ? line_counts : bits;
    const int64_t state_stride = line_counts != nullptr ? a.lc_q : a.bt_w;
    int32_t held_state[kReadAhead];
#pragma unroll
    for (uint32_t g = 0; g < kReadAhead; ++g) {
        const uint32_t q = threadIdx.x + g * kThreads;
        held_state[g] = 0;
        if (gathered > 0) {   // uniform
            held_state[g] = *element<kDense>(state, state_stride, q < gathered ? q : gathered - 1);
        }
    }
    const int64_t base = index_value(a.slot_base, base_read);
    uint32_t list_at[kLaneRegs];   // place of this thread's k-th entry in the miss and promotion lists
    bool listed[kLaneRegs];        // it is a miss entry
    if constexpr (kLookup) {
        // The looked-up slots, and the misses' ranks in lane order (over the request check's barrier).
        uint32_t missed[kLaneRegs];
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const int32_t held = lane_slot[k];
            const int32_t slot = a.table16 ? (held > 0 ? static_cast<int32_t>(base + held - 1) : 0) : held;
            lane_slot[k] = valid_lane[k] ? slot : -1;
            listed[k] = valid_lane[k] && slot == 0;
            missed[k] = __popcll(__ballot(listed[k]));
        }
        pair_counts<kWaves, kLaneRegs>(missed, miss_cells);
    }
    shared_request = workgroup_any<kWaves>(shared_request, any_cells[0]);
    if constexpr (kLookup) {
        uint32_t total = 0;
        pair_bases<kWaves, kLaneRegs>(miss_cells, list_at, total);
        m = static_cast<int32_t>(total);
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            list_at[k] += lanes_below(__ballot(listed[k]));
            if (miss_lane[k] < W && !listed[k]) {   // a miss's slot is written with its victim below
                *element<kDense>(slots, a.sl_o, static_cast<uint32_t>(miss_lane[k])) = lane_slot[k];
            }
        }
        if (threadIdx.x == 0) {
            a.counts[l * a.ct_l + b * a.ct_b] = m;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            list_at[k] = threadIdx.x + k * kThreads;
            listed[k] = static_cast<int32_t>(list_at[k]) < m;
        }
    }
    const bool overflow = step < 0 || (step + 1) * kStepStamps >= (int64_t{1} << 31);
    if (shared_request || overflow) {
        // Change nothing, record empty promotions (the move that follows
        // copies nothing; the missed lanes keep slot 0) and flag the error.
        if (threadIdx.x == 0 && a.status != nullptr) {
            atomicOr(a.status, shared_request ? kStatusSharedRequest : kStatusStampOverflow);
        }
        for (int64_t i = threadIdx.x; i < m; i += kThreads) {
            promote_src[i * a.ps_o] = -1;
            promote_dst[i * a.pd_o] = -1;
        }
        if constexpr (kLookup) {
#pragma unroll
            for (int k = 0; k < kLaneRegs; ++k) {
                if (listed[k]) {
                    *element<kDense>(slots, a.sl_o, static_cast<uint32_t>(miss_lane[k])) = 0;
                }
            }
        }
        return;
    }
    const int32_t stamp_base = static_cast<int32_t>(step * kStepStamps);
    // Touch hits: a token repeated in the row is one access of its first lane. Repeated miss tokens: with the token
    // bitmap, each valid entry sets its token's bit; a bit found set means some token repeats, and only then is the
    // exact hash built (each token's lowest miss index). Without repeats every valid entry is its token's first miss.
    int32_t token_of[kLaneRegs];   // token of this thread's k-th miss entry, or -1
    int32_t first_of[kLaneRegs];   // the first miss of that token, or -1
    bool repeated = false;
#pragma unroll
    for (int k = 0; k < kLaneRegs; ++k) {
        const int32_t o = static_cast<int32_t>(threadIdx.x) + k * kThreads;
        const int64_t offset = static_cast<int64_t>(lane_slot[k]) - base;
        if (o < W && lane_slot[k] > 0 && offset >= 0 && offset < C) {
            atomicMin(&touch[static_cast<uint32_t>(offset)], o);
        }
        const int32_t lane = miss_lane[k];
        const int64_t token = kLookup ? lane_token[k] : token_at(k, lane);
        const bool valid = listed[k] && lane >= 0 && lane < W && token >= 0 && token < a.table_cols;
        token_of[k] = valid ? static_cast<int32_t>(token) : -1;
        first_of[k] = valid ? o : -1;
        if (a.token_bitmap && token_of[k] >= 0) {
            const uint32_t bit = 1u << (token_of[k] & 31);
            repeated |= (atomicOr(&hash[token_of[k] >> 5], bit) & bit) != 0u;
        }
    }
    const bool exact_hash = workgroup_any<kWaves>(repeated, any_cells[1]) || !a.token_bitmap;   // uniform
    if (exact_hash) {
        const int32_t entries = kLookup ? static_cast<int32_t>(W) : m;   // entries a thread may hold (-1: no miss)
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const int32_t i = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            if (i < entries) {
                info[i] = token_of[k];
            }
        }
        if (a.token_bitmap) {
            for (uint32_t w = threadIdx.x; w < a.hash_size / 2; w += kThreads) {
                hash[w] = 0xffffffffu;
            }
        }
        lds_barrier();
        hash_miss_tokens(hash, info, entries, a.hash_log2);
        lds_barrier();
        const uint32_t mask = a.hash_size - 1;
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            if (token_of[k] < 0) {
                continue;
            }
            for (uint32_t h = token_hash(token_of[k], a.hash_log2);; h = (h + 1) & mask) {
                const uint32_t held = bucket_of(hash, h);
                if (held == kEmptyBucket) {
                    break;   // not reached: every inserted token lies on its probe path
                }
                if (info[held] == token_of[k]) {
                    first_of[k] = static_cast<int32_t>(held);
                    break;
                }
            }
        }
    }
    // This thread's keys, slots t + k * kThreads, in the order-preserving
    // unsigned form of the stamps (an empty slot is key 0): a touched slot's
    // stamp is stamp_base + its first lane, any other keeps what it held.
    uint32_t key[kSlotRegs];
#pragma unroll
    for (int k = 0; k < kSlotRegs; ++k) {
        const uint32_t s = threadIdx.x + k * kThreads;
        const int32_t hit = s < C ? touch[s] : INT32_MAX;
        const int32_t stamp = hit != INT32_MAX ? stamp_base + hit : held_stamp[k];
        key[k] = s < C ? static_cast<uint32_t>(stamp) ^ 0x80000000u : 0xffffffffu;
    }
    uint32_t chosen = 0;   // bit k: slot t + k * kThreads is a victim
    if (m > 0) {   // uniform
        // Rank of each first miss among the first misses, in miss-list order,
        // and the range of the keys, over one barrier.
        uint32_t first_count[kLaneRegs], rank_of[kLaneRegs], unique = 0;
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const bool first = first_of[k] >= 0 && first_of[k] == static_cast<int32_t>(threadIdx.x) + k * kThreads;
            first_count[k] = __popcll(__ballot(first));
        }
        pair_counts<kWaves, kLaneRegs>(first_count, first_cells);
        uint32_t empties = 0, lo = 0xffffffffu, hi = 0;
#pragma unroll
        for (int k = 0; k < kSlotRegs; ++k) {
            const uint32_t v = key[k];
            const bool other = v != 0 && threadIdx.x + k * kThreads < C;
            empties += v == 0 ? 1u : 0u;
            lo = other ? min(lo, v) : lo;
            hi = other ? max(hi, v) : hi;
        }
        add_range(empties, lo, hi, key_range);
        lds_barrier();
        // The info region is free of tokens now: summary words are changed in
        // place, counts' changes start at zero (published by the victims' barrier).
#pragma unroll
        for (uint32_t g = 0; g < kReadAhead; ++g) {
            const uint32_t q = threadIdx.x + g * kThreads;
            if (q < gathered) {
                summary[q] = line_counts != nullptr ? 0 : held_state[g];
            }
        }
        for (uint32_t q = threadIdx.x + kReadAhead * kThreads; q < gathered; q += kThreads) {
            summary[q] = line_counts != nullptr ? 0 : *element<kDense>(state, state_stride, q);
        }
        pair_bases<kWaves, kLaneRegs>(first_cells, rank_of, unique);
        empties = key_range[0], lo = key_range[1], hi = key_range[2];
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const int32_t i = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            const bool first = first_of[k] >= 0 && first_of[k] == i;
            rank_of[k] += lanes_below(__ballot(first));
            if (exact_hash && first) {
                owner[i] = static_cast<int16_t>(rank_of[k]);   // read by repeats past the next barriers
            }
        }
        // The `unique` victims: the slots of the smallest (stamp, slot) keys,
        // empty slots (INT32_MIN) first, then the least recently used. When
        // the empties do not cover the victims, a radix select over the other
        // keys, as distances from the smallest of them (8-bit digits, most
        // significant first), finds the key T of the (unique - empties)-th
        // smallest and how many keys at T it takes; it starts at the highest
        // digit of the largest distance (the stamps of a buffer span a few
        // steps: two digits, where the digits in which plain keys
        // differ were three whenever a step crossed a multiple of 65,536). The
        // victims are then listed in slot order, and the i-th first miss takes
        // the i-th of them.
        if (unique > 0) {   // uniform
            uint32_t prefix = 0, prefix_mask = 0;   // of the distances from lo
            uint32_t threshold = 0;  // T
            uint32_t need = unique;  // keys still to take at the prefix (uniform)
            int first_shift = -8;    // no select: the empties alone, or every other key equal
            if (unique > empties) {
                need = unique - empties;
                if (hi != lo) {
                    first_shift = ((31 - __clz(hi - lo)) / 8) * 8;   // every higher digit is 0
                }
                threshold = lo;
            }
            for (int shift = first_shift, pass = 0; shift >= 0; shift -= 8, ++pass) {
                int32_t* count = digit_count + (pass & 1) * kDigits;
                if (pass >= 2) {   // uniform: the histogram of two passes ago, read by every wave before the last barrier
                    for (uint32_t d = threadIdx.x; d < kDigits; d += kThreads) {
                        count[d] = 0;
                    }
                    lds_barrier();
                }
                // Runs of one digit in a thread's slots count with one atomic:
                // recent stamps share their high digits, which would otherwise
                // serialize thousands of atomics on one counter.
                uint32_t run_digit = 0;
                int32_t run = 0;
#pragma unroll
                for (int k = 0; k < kSlotRegs; ++k) {
                    const uint32_t distance = key[k] - lo;
                    if (key[k] != 0 && (distance & prefix_mask) == prefix && threadIdx.x + k * kThreads < C) {
                        const uint32_t d = (distance >> shift) & 255u;
                        if (run > 0 && d != run_digit) {
                            atomicAdd(&count[run_digit], run);
                            run = 0;
                        }
                        run_digit = d;
                        ++run;
                    }
                }
                if (run > 0) {
                    atomicAdd(&count[run_digit], run);
                }
                lds_barrier();
                // Every wave scans the 256 counts itself (4 digits per lane)
                // and finds the digit holding the need-th key: no second barrier.
                const uint32_t lane = threadIdx.x & 63;
                const int4 c = reinterpret_cast<const int4*>(count)[lane];
                const uint32_t c0 = c.x, c1 = c0 + c.y, c2 = c1 + c.z, c3 = c2 + c.w;
                const uint32_t inclusive = wave_scan<kAdd>(c3);
                const uint32_t below = inclusive - c3;
                const uint64_t holds = __ballot(below < need && need <= inclusive);   // exactly one lane
                const int holder = __ffsll(static_cast<unsigned long long>(holds)) - 1;
                const uint32_t rest = need - below;   // in the holder: 1..c3
                const uint32_t j = rest <= c0 ? 0u : (rest <= c1 ? 1u : (rest <= c2 ? 2u : 3u));
                const uint32_t skipped = below + (j == 0 ? 0u : (j == 1 ? c0 : (j == 2 ? c1 : c2)));
                prefix |= (4u * holder + __builtin_amdgcn_readlane(j, holder)) << shift;
                prefix_mask |= 255u << shift;
                need -= __builtin_amdgcn_readlane(skipped, holder);
            }
            threshold += prefix;
            // T = threshold. Slot s is a victim when its key is below T (every
            // empty slot, when the empties do not cover the victims), or at T
            // and fewer than `need` slots below s hold T; its place in the list
            // is the number of victims below it. The slot-order counts of both
            // kinds (16 bits each) come from per-wave ballots.
            uint32_t kinds[kSlotRegs], before[kSlotRegs], all = 0;
#pragma unroll
            for (int k = 0; k < kSlotRegs; ++k) {
                const bool in = threadIdx.x + k * kThreads < C;
                kinds[k] = static_cast<uint32_t>(__popcll(__ballot(in && key[k] < threshold))) |
                           static_cast<uint32_t>(__popcll(__ballot(in && key[k] == threshold))) << 16;
            }
            pair_counts<kWaves, kSlotRegs>(kinds, victim_cells);
            lds_barrier();
            pair_bases<kWaves, kSlotRegs>(victim_cells, before, all);
#pragma unroll
            for (int k = 0; k < kSlotRegs; ++k) {
                const uint32_t s = threadIdx.x + k * kThreads;
                const bool lower = s < C && key[k] < threshold;
                const bool tie = s < C && key[k] == threshold;
                const uint32_t lower_before = (before[k] & 0xffffu) + lanes_below(__ballot(lower));
                const uint32_t ties_before = (before[k] >> 16) + lanes_below(__ballot(tie));
                if (lower || (tie && ties_before < need)) {
                    victims[lower_before + min(ties_before, need)] = static_cast<int16_t>(s);
                    chosen |= 1u << k;
                }
            }
        }
        lds_barrier();   // the victims (and the ranks of repeated tokens) are read by other threads below
        // Batch 3: each entry's victim (from LDS), then the victims' old
        // tokens and the promoted tokens' host rows, all loads issued before
        // any is used.
        const char* host_row = static_cast<const char*>(a.host_table.data) +
                               req * a.host_sr * (a.host_table.is64 ? 8 : 4);
        int32_t victim_of[kLaneRegs];
        int32_t old_of[kLaneRegs];
        int32_t host_row_of[kLaneRegs];
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const int32_t i = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            const bool valid = token_of[k] >= 0;
            const uint32_t rank = first_of[k] == i ? rank_of[k] : (valid ? static_cast<uint32_t>(owner[first_of[k]]) : 0u);
            victim_of[k] = valid ? static_cast<int32_t>(victims[rank]) : 0;
            old_of[k] = *element<kDense>(slot_token, a.st_c, static_cast<uint32_t>(victim_of[k]));
            host_row_of[k] = index_word<kDense>(host_row, a.host_table.is64, a.host_st,
                                                valid ? static_cast<uint32_t>(token_of[k]) : 0u, false);
        }
#pragma unroll
        for (int k = 0; k < kLaneRegs; ++k) {
            const int32_t i = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            if (!listed[k]) {
                continue;
            }
            const int32_t lane = miss_lane[k];
            const int32_t victim = victim_of[k];
            const int32_t token = token_of[k];
            const int32_t global = static_cast<int32_t>(static_cast<uint32_t>(base) + static_cast<uint32_t>(victim));
            if (token >= 0) {
                *element<kDense>(slots, a.sl_o, static_cast<uint32_t>(lane)) = global;
            }
            if (first_of[k] != i) {
                // Not an entry of a miss list written by the lookup, or a repeat of an earlier miss (which shares that
                // miss's slot and promotion): record an empty promotion so the move that follows skips it.
                *element<kDense>(promote_src, a.ps_o, list_at[k]) = -1;
                *element<kDense>(promote_dst, a.pd_o, list_at[k]) = -1;
                continue;
            }
            const int32_t old = old_of[k];
            if (old >= 0 && old < a.table_cols) {
                set_entry<kDense>(a, table_row, old, 0);
                if (gathered > 0 && a.bits_shift == 0) {
                    atomicAnd(reinterpret_cast<unsigned int*>(&summary[old >> 5]), ~(1u << (old & 31)));
                } else if (gathered > 0) {
                    atomicSub(&summary[old >> a.bits_shift], 1);
                } else if (bits != nullptr && a.bits_shift == 0) {
                    atomicAnd(reinterpret_cast<unsigned int*>(bits + (old >> 5) * a.bt_w), ~(1u << (old & 31)));
                } else if (line_counts != nullptr) {
                    // The group's last resident position leaves: clear its bit.
                    const int64_t q = old >> a.bits_shift;
                    if (atomicSub(line_counts + q * a.lc_q, 1) == 1) {
                        atomicAnd(reinterpret_cast<unsigned int*>(bits + (q >> 5) * a.bt_w), ~(1u << (q & 31)));
                    }
                }
                // Without counts a coarse bit stays set (other positions of
                // its group may still be resident): a superset.
            }
            set_entry<kDense>(a, table_row, token, a.table16 ? victim + 1 : global);
            if (gathered > 0 && a.bits_shift == 0) {
                atomicOr(reinterpret_cast<unsigned int*>(&summary[token >> 5]), 1u << (token & 31));
            } else if (gathered > 0) {
                atomicAdd(&summary[token >> a.bits_shift], 1);
            } else if (bits != nullptr && line_counts == nullptr) {
                const int64_t q = token >> a.bits_shift;
                atomicOr(reinterpret_cast<unsigned int*>(bits + (q >> 5) * a.bt_w), 1u << (q & 31));
            }
            *element<kDense>(slot_token, a.st_c, static_cast<uint32_t>(victim)) = token;
            touch[victim] = stamp_base + kMaxWidth + lane;
            *element<kDense>(promote_src, a.ps_o, list_at[k]) = host_row_of[k];
            *element<kDense>(promote_dst, a.pd_o, list_at[k]) = global;
        }
        if (gathered > 0 || line_counts == nullptr) {   // uniform
            lds_barrier();     // the victims' stamps and the summary's changes are read by other threads below
        } else {
            __syncthreads();   // the evictions' count decrements (global atomics) precede the increments
            // Insertions: after every eviction's clear above, so a group that
            // both loses and gains positions ends with its bit set.
#pragma unroll
            for (int k = 0; k < kLaneRegs; ++k) {
                if (token_of[k] >= 0 && first_of[k] == static_cast<int32_t>(threadIdx.x) + k * kThreads) {
                    const int64_t q = static_cast<int64_t>(token_of[k]) >> a.bits_shift;
                    if (atomicAdd(line_counts + q * a.lc_q, 1) == 0) {
                        atomicOr(reinterpret_cast<unsigned int*>(bits + (q >> 5) * a.bt_w), 1u << (q & 31));
                    }
                }
            }
        }
        // The summary words, or each group's count and the bits of the groups that empty or fill (a wave's 64 groups are
        // two words).
        for (uint32_t g = 0; g * kThreads < gathered; ++g) {   // uniform over the workgroup
            const uint32_t q = threadIdx.x + g * kThreads;
            const int32_t mine = q < gathered ? summary[q] : 0;
            if (line_counts == nullptr) {   // uniform
                if (q < gathered) {
                    *element<kDense>(bits, a.bt_w, q) = mine;
                }
                continue;
            }
            int32_t held = held_state[0];
#pragma unroll
            for (uint32_t r = 1; r < kReadAhead; ++r) {
                held = g == r ? held_state[r] : held;
            }
            if (g >= kReadAhead) {   // uniform
                held = line_counts[(q < gathered ? q : gathered - 1) * a.lc_q];
            }
            if (mine != 0) {
                line_counts[q * a.lc_q] = held + mine;
            }
            const uint64_t clears = __ballot(mine != 0 && held > 0 && held + mine <= 0);
            const uint64_t sets = __ballot(mine != 0 && held <= 0 && held + mine > 0);
            if ((threadIdx.x & 31) == 0) {
                const uint32_t clear = static_cast<uint32_t>(clears >> (threadIdx.x & 32));
                const uint32_t set = static_cast<uint32_t>(sets >> (threadIdx.x & 32));
                auto* word = reinterpret_cast<unsigned int*>(bits + (q >> 5) * a.bt_w);
                if (clear != 0) {
                    atomicAnd(word, ~clear);
                }
                if (set != 0) {
                    atomicOr(word, set);
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kSlotRegs; ++k) {
        const uint32_t s = threadIdx.x + k * kThreads;
        if (s < C) {
            *element<kDense>(stamps, a.sp_c, s) = (chosen >> k) & 1u ? touch[s] : static_cast<int32_t>(key[k] ^ 0x80000000u);
        }
    }
}

// One thread advances the device step counter after the swap-in of a replay.
__global__ void advance_step_kernel(int64_t* counter) {
    if (threadIdx.x == 0) {
        counter[0] += 1;
    }
}

template <int kThreads, int kSlotRegs, int kLaneRegs>
void launch_swap(const SwapArgs& a, bool dense, dim3 grid, size_t lds, hipStream_t stream) {
    auto* kernel = a.lengths.data != nullptr ? swap_in_kernel<kThreads, kSlotRegs, kLaneRegs, true, true>
                   : dense                   ? swap_in_kernel<kThreads, kSlotRegs, kLaneRegs, true, false>
                                             : swap_in_kernel<kThreads, kSlotRegs, kLaneRegs, false, false>;
    if (lds > 60 * 1024) {   // with the static 3 KiB, past the default 64
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)),
                  "raise the swap-in LDS limit");
    }
    kernel<<<grid, dim3(kThreads), lds, stream>>>(a);
}

// swap_in's answer when it was asked to run the lookup too and the layouts need the lookup's own kernels.
constexpr int kNeedsLookup = 1;

void need_i32(const ekv_tensor& t, const char* name) {
    if (t.dtype != EKV_INT32) {
        throw std::invalid_argument(std::string(name) + " must be int32");
    }
}

int swap_in(const ekv_tensor* topk_p, int64_t block_size, const ekv_tensor* rows_p, const ekv_tensor* selected_p,
            const ekv_tensor* slots_p, const ekv_tensor* misses_p, const ekv_tensor* counts_p,
            const ekv_tensor* table_p, const ekv_tensor* bits_p, int64_t bits_shift, const ekv_tensor* counts_q_p,
            const ekv_tensor* slot_token_p,
            const ekv_tensor* stamps_p, const ekv_tensor* slot_base_p, const ekv_tensor* host_table_p,
            const ekv_tensor* promote_src_p, const ekv_tensor* promote_dst_p, int64_t step,
            const ekv_tensor* step_counter_p, const ekv_tensor* status_p, void* stream,
            const ekv_tensor* lengths_p = nullptr) {
    const ekv_tensor& topk = need(topk_p, "topk");
    const ekv_tensor& rows = need(rows_p, "rows");
    const ekv_tensor& selected = need(selected_p, "selected");
    const ekv_tensor& slots = need(slots_p, "slots");
    const ekv_tensor& misses = need(misses_p, "misses");
    const ekv_tensor& counts = need(counts_p, "miss_count");
    const ekv_tensor& table = need(table_p, "table");
    const ekv_tensor& slot_token = need(slot_token_p, "slot_token");
    const ekv_tensor& stamps = need(stamps_p, "stamps");
    const ekv_tensor& slot_base = need(slot_base_p, "slot_base");
    const ekv_tensor& host_table = need(host_table_p, "host_table");
    const ekv_tensor& promote_src = need(promote_src_p, "promote_src");
    const ekv_tensor& promote_dst = need(promote_dst_p, "promote_dst");
    need_ndim(topk, 3, "topk");
    need_index(topk, "topk");
    const int64_t L = topk.shape[0], B = topk.shape[1], K = topk.shape[2];
    if (block_size < 1 || block_size >= (int64_t{1} << 31)) {
        throw std::invalid_argument("block_size must be positive");
    }
    const int64_t W = K * block_size;
    for (const auto* t : {&slots, &misses, &promote_src, &promote_dst}) {
        need_ndim(*t, 3, "slots/misses/promote lists");
        need_i32(*t, "slots/misses/promote lists");
        need_dim(*t, 0, L, "slots/misses/promote lists");
        need_dim(*t, 1, B, "slots/misses/promote lists");
        need_dim(*t, 2, W, "slots/misses/promote lists");
    }
    need_ndim(counts, 2, "miss_count");
    need_i32(counts, "miss_count");
    need_dim(counts, 0, L, "miss_count");
    need_dim(counts, 1, B, "miss_count");
    for (const auto* t : {&table, &slot_token, &stamps}) {
        need_ndim(*t, 3, "table/slot_token/stamps");
        if (t != &table || table.dtype != EKV_INT16) {
            need_i32(*t, "table/slot_token/stamps");
        }
        need_dim(*t, 0, L, "table/slot_token/stamps");
    }
    const int64_t R = table.shape[1], T = table.shape[2], C = slot_token.shape[2];
    need_dim(slot_token, 1, R, "slot_token");
    need_dim(stamps, 1, R, "stamps");
    need_dim(stamps, 2, C, "stamps");
    if (C < 1 || C > kMaxCapacity) {
        throw std::invalid_argument("capacity must be 1.." + std::to_string(kMaxCapacity));
    }
    static_assert(kMaxCapacity < 32768, "int16 tables hold local slot + 1");
    if (W > C) {
        throw std::invalid_argument("lanes per row exceed the hot capacity");
    }
    if (W > kMaxWidth) {
        throw std::invalid_argument("at most " + std::to_string(kMaxWidth) + " lanes per row");
    }
    if (T >= (int64_t{1} << 31) || step < 0 || (step + 1) * kStepStamps >= (int64_t{1} << 31)) {
        throw std::invalid_argument("token count or step outside the 32-bit stamp range");
    }
    int32_t* status = nullptr;
    if (status_p != nullptr) {
        const ekv_tensor& st = need(status_p, "status");
        if (st.dtype != EKV_INT32 || numel(st) != 1 || st.data == nullptr) {
            throw std::invalid_argument("status must be one int32 element in device memory");
        }
        status = static_cast<int32_t*>(st.data);
    }
    int64_t* counter = nullptr;
    if (step_counter_p != nullptr) {
        const ekv_tensor& c = need(step_counter_p, "step_counter");
        if (c.dtype != EKV_INT64 || numel(c) != 1 || c.data == nullptr) {
            throw std::invalid_argument("step_counter must be one int64 element in device memory");
        }
        counter = static_cast<int64_t*>(c.data);
    }
    need_ndim(rows, 1, "rows");
    need_ndim(selected, 1, "selected");
    need_ndim(slot_base, 1, "slot_base");
    need_index(rows, "rows");
    need_index(selected, "selected");
    need_index(slot_base, "slot_base");
    need_dim(rows, 0, B, "rows");
    need_dim(slot_base, 0, R, "slot_base");
    need_ndim(host_table, 2, "host_table");
    need_index(host_table, "host_table");
    need_dim(host_table, 0, R, "host_table");
    need_dim(host_table, 1, T, "host_table");
    if (bits_p != nullptr) {
        const ekv_tensor& bits = need(bits_p, "resident_bits");
        need_ndim(bits, 3, "resident_bits");
        need_i32(bits, "resident_bits");
        need_dim(bits, 0, L, "resident_bits");
        need_dim(bits, 1, R, "resident_bits");
        if (bits_shift < 0 || bits_shift > 20) {
            throw std::invalid_argument("bits_shift must be 0..20");
        }
        const int64_t summary_bits = (T + (int64_t{1} << bits_shift) - 1) >> bits_shift;
        if (bits.shape[2] < (summary_bits + 31) / 32) {
            throw std::invalid_argument("resident_bits needs ceil(ceil(T / 2^bits_shift) / 32) words per row");
        }
        if (counts_q_p != nullptr) {
            const ekv_tensor& groups = need(counts_q_p, "resident_counts");
            if (bits_shift == 0) {
                throw std::invalid_argument("resident_counts serve a summary with bits_shift > 0");
            }
            need_ndim(groups, 3, "resident_counts");
            need_i32(groups, "resident_counts");
            need_dim(groups, 0, L, "resident_counts");
            need_dim(groups, 1, R, "resident_counts");
            need_dim(groups, 2, summary_bits, "resident_counts");
            need_data(groups, "resident_counts");
        }
    } else if (counts_q_p != nullptr) {
        throw std::invalid_argument("resident_counts need resident_bits");
    }
    const int64_t count = selected.shape[0];
    if (L > 65535 || count > 0x7fffffff) {
        throw std::invalid_argument("too many layers or rows for one launch");
    }
    // An empty batch leaves every selection entry stray: nothing to launch
    // (the kernel's first reads assume batch row 0 exists).
    const bool launches = count > 0 && L > 0 && W > 0 && B > 0;
    if (launches) {
        for (const auto* t : {&topk, &rows, &selected, &slots, &misses, &counts, &table, &slot_token, &stamps,
                              &slot_base, &host_table, &promote_src, &promote_dst}) {
            need_data(*t, "tensor");
        }
        if (T == 0) {
            throw std::invalid_argument("the token table has no positions");   // host rows are read at position 0
        }
    }
    if (check_only()) {
        return 0;
    }
    if (!launches) {
        if (counter != nullptr) {
            advance_step_kernel<<<dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream)>>>(counter);
            check_hip(hipGetLastError(), "launch step advance");
        }
        return 0;
    }
    SwapArgs a{};
    a.topk = topk.data;
    a.topk64 = topk.dtype == EKV_INT64;
    a.topk_sl = topk.stride[0];
    a.topk_sb = topk.stride[1];
    a.topk_sk = topk.stride[2];
    a.block_size = static_cast<uint32_t>(block_size);
    a.block_div = FastDiv(static_cast<uint32_t>(block_size));
    a.rows = index_ref(rows, 0);
    a.selected = index_ref(selected, 0);
    a.slot_base = index_ref(slot_base, 0);
    a.slots = static_cast<int32_t*>(slots.data);
    a.sl_l = slots.stride[0], a.sl_b = slots.stride[1], a.sl_o = slots.stride[2];
    a.misses = static_cast<const int32_t*>(misses.data);
    a.mi_l = misses.stride[0], a.mi_b = misses.stride[1], a.mi_o = misses.stride[2];
    a.counts = static_cast<int32_t*>(counts.data);
    a.ct_l = counts.stride[0], a.ct_b = counts.stride[1];
    a.table = table.data;
    a.table16 = table.dtype == EKV_INT16;
    a.tb_l = table.stride[0], a.tb_r = table.stride[1], a.tb_t = table.stride[2], a.table_cols = T;
    if (bits_p != nullptr) {
        a.bits = static_cast<int32_t*>(bits_p->data);
        a.bt_l = bits_p->stride[0], a.bt_r = bits_p->stride[1], a.bt_w = bits_p->stride[2];
        a.bits_shift = static_cast<uint32_t>(bits_shift);
        if (counts_q_p != nullptr) {
            a.line_counts = static_cast<int32_t*>(counts_q_p->data);
            a.lc_l = counts_q_p->stride[0], a.lc_r = counts_q_p->stride[1], a.lc_q = counts_q_p->stride[2];
        }
    }
    a.selected_count = count;
    a.status = status;
    a.slot_token = static_cast<int32_t*>(slot_token.data);
    a.st_l = slot_token.stride[0], a.st_r = slot_token.stride[1], a.st_c = slot_token.stride[2];
    a.stamps = static_cast<int32_t*>(stamps.data);
    a.sp_l = stamps.stride[0], a.sp_r = stamps.stride[1], a.sp_c = stamps.stride[2];
    a.host_table = index_ref(host_table, 0);
    a.host_table.stride = 1;
    a.host_sr = host_table.stride[0];
    a.host_st = host_table.stride[1];
    a.promote_src = static_cast<int32_t*>(promote_src.data);
    a.ps_l = promote_src.stride[0], a.ps_b = promote_src.stride[1], a.ps_o = promote_src.stride[2];
    a.promote_dst = static_cast<int32_t*>(promote_dst.data);
    a.pd_l = promote_dst.stride[0], a.pd_b = promote_dst.stride[1], a.pd_o = promote_dst.stride[2];
    a.batch = B;
    a.table_rows = R;
    a.capacity = C;
    a.width = static_cast<uint32_t>(W);
    a.step = step;
    a.step_counter = counter;
    a.hash_size = 2;
    a.hash_log2 = 1;
    while (a.hash_size < 2 * W) {
        a.hash_size <<= 1;
        ++a.hash_log2;
    }
    // A bitmap of the tokens in up to 8 KiB of LDS, whatever the hash takes: it
    // is one LDS atomic per miss, the hash a probe chain behind two more barriers
    // (0.8 of 9.2 us in a row of 64 lanes over 4096 tokens).
    a.token_bitmap = T <= std::max<int64_t>(int64_t{16} * a.hash_size, int64_t{1} << 16) ? 1u : 0u;
    a.bitmap_words = static_cast<uint32_t>(a.token_bitmap ? (T + 31) / 32 : 0);
    if (a.line_counts != nullptr || (a.bits != nullptr && bits_shift == 0)) {
        const int64_t cover = bits_shift == 0 ? 32 : int64_t{1} << bits_shift;   // positions per word or group
        const int64_t entries = (T + cover - 1) / cover;
        a.gathered = entries <= kMaxGathered ? static_cast<uint32_t>(entries) : 0u;
    }
    // touches; the miss tokens, then the ranks (2 bytes each) and the summary;
    // the 16-bit hash buckets or the token bitmap, then the victim list
    // (2 bytes per victim: at most W <= hash_size / 2)
    static_assert(kMaxWidth <= 0x7fff && kMaxCapacity <= 0x7fff, "miss indices and slots fit 16 bits");
    a.info_words = static_cast<uint32_t>(std::max<int64_t>(W, (W + 1) / 2 + a.gathered));
    const size_t lds = (static_cast<size_t>(C) + a.info_words + std::max(a.hash_size / 2, a.bitmap_words)) * 4;
    const dim3 grid(static_cast<uint32_t>(count), static_cast<uint32_t>(L));
    const auto s = static_cast<hipStream_t>(stream);
    // The workgroup size: the smallest whose threads hold four slots and two
    // lanes each, so that the most waves share a row's phases, while such workgroups
    // fill no more than half of the CUs' threads; past that the smallest whose threads
    // hold eight and four, since what each wave repeats (scans, ranges) then
    // costs the rows beside it. Measured (us, the swap alone; lanes and slots of a row):
    //   rows x lanes, slots     four and two   eight and four
    //   48 x 1024, 2048             13.0           15.2
    //   256 x 2048, 4096            21.0           22.6
    //   512 x 1024, 2048            19.4           21.2
    //   512 x 512, 1024             14.8           18.7
    //   384 x 2048, 4096            33.3           26.6
    //   1024 x 1024, 2048           33.6           27.8
    //   2560 x 256, 1024            31.0           28.6
    //   2560 x 512, 1024            38.9           43.1   (on the wrong side of the line)
    //   2560 x 768, 1536            60.5           48.3
    //   2560 x 1024, 2048           67.0           62.0
    //   2560 x 2048, 4096          162.9          115.0
    // (2560 x 256, 512: 24.7 against 27.8, so rows of up to 512 slots stay with four.)
    constexpr int64_t kHalfOfThreads = 256 * 1024;
    const bool dense = a.topk_sk == 1 && a.sl_o == 1 && a.mi_o == 1 && a.st_c == 1 && a.sp_c == 1 && a.ps_o == 1 &&
                       a.pd_o == 1 && a.tb_t == 1 && a.host_st == 1 && (a.bits == nullptr || a.bt_w == 1) &&
                       (a.line_counts == nullptr || a.lc_q == 1) && T < (int64_t{1} << 29);
    if (lengths_p != nullptr) {
        if (!dense) {
            return kNeedsLookup;
        }
        a.lengths = index_ref(*lengths_p, 0);
    }
    const int64_t four = std::max((C + 3) / 4, (W + 1) / 2), eight = std::max((C + 7) / 8, (W + 3) / 4);
    int64_t threads = 64;   // of the four-and-two workgroup
    while (threads < four) {
        threads *= 2;
    }
    const bool crowded = count * L * threads > kHalfOfThreads && four > 128;
    if (four <= 64) {
        launch_swap<64, 4, 2>(a, dense, grid, lds, s);
    } else if (four <= 128) {
        launch_swap<128, 4, 2>(a, dense, grid, lds, s);
    } else if (crowded && eight <= 128) {
        launch_swap<128, 8, 4>(a, dense, grid, lds, s);
    } else if (four <= 256) {
        launch_swap<256, 4, 2>(a, dense, grid, lds, s);
    } else if (crowded && eight <= 256) {
        launch_swap<256, 8, 4>(a, dense, grid, lds, s);
    } else if (four <= 512) {
        launch_swap<512, 4, 2>(a, dense, grid, lds, s);
    } else if (crowded && eight <= 512) {
        launch_swap<512, 8, 4>(a, dense, grid, lds, s);
    } else if (four <= 1024) {
        launch_swap<1024, 4, 2>(a, dense, grid, lds, s);
    } else {
        launch_swap<1024, 8, 4>(a, dense, grid, lds, s);
    }
    check_hip(hipGetLastError(), "launch swap-in");
    if (counter != nullptr) {
        advance_step_kernel<<<dim3(1), dim3(64), 0, s>>>(counter);
        check_hip(hipGetLastError(), "launch step advance");
    }
    return 0;
}

}  // namespace

bool lookup_swap_in(const ekv_step_args& s, const ekv_tensor& misses, const ekv_tensor& counts, const ekv_tensor& src,
                    const ekv_tensor& dst, void* stream) {
    const bool counted = s.step_counter != nullptr;
    return swap_in(s.topk, s.block_size, s.rows, s.selected, s.slots, &misses, &counts, s.table, s.resident_bits,
                   s.bits_shift, s.resident_counts, s.slot_token, s.stamps, s.slot_base, s.host_table, &src, &dst,
                   counted ? 0 : s.step, s.step_counter, s.status, stream, s.lengths) != kNeedsLookup;
}

}  // namespace ekv

extern "C" int ekv_swap_in(const ekv_tensor* topk, int64_t block_size, const ekv_tensor* rows,
                           const ekv_tensor* selected, const ekv_tensor* slots, const ekv_tensor* misses,
                           const ekv_tensor* miss_count, const ekv_tensor* table, const ekv_tensor* resident_bits,
                           int64_t bits_shift, const ekv_tensor* resident_counts, const ekv_tensor* slot_token,
                           const ekv_tensor* stamps,
                           const ekv_tensor* slot_base, const ekv_tensor* host_table, const ekv_tensor* promote_src,
                           const ekv_tensor* promote_dst, int64_t step, const ekv_tensor* status, void* stream) {
    return ekv::guarded(-1, [&] {
        return ekv::swap_in(topk, block_size, rows, selected, slots, misses, miss_count, table, resident_bits,
                            bits_shift, resident_counts, slot_token, stamps, slot_base, host_table, promote_src,
                            promote_dst, step, nullptr, status, stream);
    });
}

extern "C" int ekv_swap_in_counted(const ekv_tensor* topk, int64_t block_size, const ekv_tensor* rows,
                                   const ekv_tensor* selected, const ekv_tensor* slots, const ekv_tensor* misses,
                                   const ekv_tensor* miss_count, const ekv_tensor* table,
                                   const ekv_tensor* resident_bits, int64_t bits_shift,
                                   const ekv_tensor* resident_counts, const ekv_tensor* slot_token,
                                   const ekv_tensor* stamps,
                                   const ekv_tensor* slot_base, const ekv_tensor* host_table,
                                   const ekv_tensor* promote_src, const ekv_tensor* promote_dst,
                                   const ekv_tensor* step_counter, const ekv_tensor* status, void* stream) {
    return ekv::guarded(-1, [&] {
        if (step_counter == nullptr) {
            throw std::invalid_argument("step_counter is required");
        }
        return ekv::swap_in(topk, block_size, rows, selected, slots, misses, miss_count, table, resident_bits,
                            bits_shift, resident_counts, slot_token, stamps, slot_base, host_table, promote_src,
                            promote_dst, 0, step_counter, status, stream);
    });
}
