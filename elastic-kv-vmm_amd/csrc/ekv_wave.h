// Scans over the wave64 and over a workgroup whose threads hold strided registers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ekv {

// Inclusive scan of one value per lane over the wave, in six DPP steps (within
// rows of 16 lanes, then row 0 to 1 and 2 to 3, then lane 31 to rows 2 and 3)
// instead of six LDS permutes of a round trip each.
enum WaveOp { kAdd, kMin, kMax };

template <WaveOp kOp>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    constexpr uint32_t kNone = kOp == kMin ? 0xffffffffu : 0u;   // what a lane without a source combines
    const auto combine = [](uint32_t a, int b) {
        const uint32_t other = static_cast<uint32_t>(b);
        return kOp == kAdd ? a + other : (kOp == kMin ? min(a, other) : max(a, other));
    };
    constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143;   // DPP controls
    v = combine(v, __builtin_amdgcn_update_dpp(static_cast<int>(kNone), static_cast<int>(v), kRowShr + 1, 0xf, 0xf, false));
    v = combine(v, __builtin_amdgcn_update_dpp(static_cast<int>(kNone), static_cast<int>(v), kRowShr + 2, 0xf, 0xf, false));
    v = combine(v, __builtin_amdgcn_update_dpp(static_cast<int>(kNone), static_cast<int>(v), kRowShr + 4, 0xf, 0xf, false));
    v = combine(v, __builtin_amdgcn_update_dpp(static_cast<int>(kNone), static_cast<int>(v), kRowShr + 8, 0xf, 0xf, false));
    v = combine(v, __builtin_amdgcn_update_dpp(static_cast<int>(kNone), static_cast<int>(v), kRowBcast15, 0xa, 0xf, false));
    v = combine(v, __builtin_amdgcn_update_dpp(static_cast<int>(kNone), static_cast<int>(v), kRowBcast31, 0xc, 0xf, false));
    return v;
}

// Elements are held as register k of thread t = element t + k * threads, so
// wave w's registers k cover consecutive elements. Each wave leaves its counts
// (two 16-bit fields per word) of every register in `cells`; after a barrier,
// pair_bases gives the count of all elements before register k of this wave.
template <int kWaves, int kRegs>
__device__ __forceinline__ void pair_counts(const uint32_t (&count)[kRegs], uint32_t* cells) {
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < kRegs; ++k) {
            cells[k * kWaves + (threadIdx.x >> 6)] = count[k];
        }
    }
}

template <int kWaves, int kRegs>
__device__ __forceinline__ void pair_bases(const uint32_t* cells, uint32_t (&base)[kRegs], uint32_t& total) {
    constexpr int kPairs = kWaves * kRegs;
    constexpr int kPer = (kPairs + 63) / 64;
    static_assert(kPer <= 2, "at most two cells per lane");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    uint32_t cell[kPer], sum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int at = lane * kPer + j;
        cell[j] = cells[at < kPairs ? at : 0];
        cell[j] = at < kPairs ? cell[j] : 0u;
        sum += cell[j];
    }
    const uint32_t inclusive = wave_scan<kAdd>(sum);
    const uint32_t before = inclusive - sum;
    total = __builtin_amdgcn_readlane(inclusive, (kPairs - 1) / kPer);
#pragma unroll
    for (int k = 0; k < kRegs; ++k) {
        const int pair = k * kWaves + wave;
        base[k] = __builtin_amdgcn_readlane(before, pair / kPer);
        if (kPer > 1 && (pair & 1)) {
            base[k] += __builtin_amdgcn_readlane(cell[0], pair / kPer);
        }
    }
}

}  // namespace ekv
