// Cross-lane reductions of a 64-lane wave by data-parallel primitives (no LDS traffic).

#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <type_traits>

namespace gmm {

// v of the lane that the DPP control word names, the lane's own v where there is none.
template<int Ctrl>
__device__ inline uint32_t dpp(uint32_t v)
{
    return uint32_t(__builtin_amdgcn_update_dpp(int(v), int(v), Ctrl, 0xf, 0xf, false));
}

constexpr int DPP_XOR1 = 0xb1;            // lane ^ 1, lane ^ 2 (permutations within groups of 4)
constexpr int DPP_XOR2 = 0x4e;
constexpr int DPP_QUAD0 = 0x00;           // the first lane of the group of 4
constexpr int DPP_HALF_MIRROR = 0x141;    // lane 7 - i of the group of 8
constexpr int DPP_ROW_SHR = 0x110;        // + n: lane - n of the row of 16
constexpr int DPP_BCAST15 = 0x142;        // lane 15 of a row to the next row
constexpr int DPP_BCAST31 = 0x143;        // lane 31 to lanes 32..63

// op over the wave's 64 values, for an idempotent op (min, max, or); the same in every lane.
template<typename Op>
__device__ inline uint32_t wave_reduce(uint32_t v, Op op)
{
    v = op(v, dpp<DPP_ROW_SHR + 1>(v));
    v = op(v, dpp<DPP_ROW_SHR + 2>(v));
    v = op(v, dpp<DPP_ROW_SHR + 4>(v));
    v = op(v, dpp<DPP_ROW_SHR + 8>(v));
    v = op(v, dpp<DPP_BCAST15>(v));
    v = op(v, dpp<DPP_BCAST31>(v));
    return uint32_t(__builtin_amdgcn_readlane(int(v), 63));
}

__device__ inline uint32_t wave_min_u32(uint32_t v)
{
    return wave_reduce(v, [](uint32_t a, uint32_t b) { return min(a, b); });
}

__device__ inline uint32_t wave_max_u32(uint32_t v)
{
    return wave_reduce(v, [](uint32_t a, uint32_t b) { return max(a, b); });
}

// Inclusive sum over the wave's lanes.
__device__ inline uint32_t wave_inclusive_sum(uint32_t v)
{
    auto shifted = [](uint32_t x, auto ctrl, auto rows) {
        return uint32_t(__builtin_amdgcn_update_dpp(0, int(x), decltype(ctrl)::value, decltype(rows)::value, 0xf, false));
    };
    using std::integral_constant;
    v += shifted(v, integral_constant<int, DPP_ROW_SHR + 1>(), integral_constant<int, 0xf>());
    v += shifted(v, integral_constant<int, DPP_ROW_SHR + 2>(), integral_constant<int, 0xf>());
    v += shifted(v, integral_constant<int, DPP_ROW_SHR + 4>(), integral_constant<int, 0xf>());
    v += shifted(v, integral_constant<int, DPP_ROW_SHR + 8>(), integral_constant<int, 0xf>());
    v += shifted(v, integral_constant<int, DPP_BCAST15>(), integral_constant<int, 0xa>());
    v += shifted(v, integral_constant<int, DPP_BCAST31>(), integral_constant<int, 0xc>());
    return v;
}

// op over the 8 lanes of each aligned group of 8, the same in all of them. (Permutations have a source
// for every lane, so the compiler can fold the move into an integer op.)
template<typename Op>
__device__ inline uint32_t group8_reduce(uint32_t v, Op op)
{
    v = op(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), DPP_XOR1, 0xf, 0xf, true)));
    v = op(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), DPP_XOR2, 0xf, 0xf, true)));
    v = op(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), DPP_HALF_MIRROR, 0xf, 0xf, true)));
    return v;
}

// Exclusive scan over a block of NT threads (NT/64 waves), returns the block total too;
// s_wave: a word per wave.
template<int NT>
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t *s_wave, uint32_t &total)
{
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    uint32_t inc = wave_inclusive_sum(v);
    if (lane == 63)
        s_wave[wave] = inc;
    __syncthreads();
    uint32_t before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        uint32_t t = s_wave[w];
        before += (w < wave) ? t : 0u;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return before + inc - v;
}

}  // namespace gmm
