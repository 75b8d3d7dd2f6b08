// Cross-lane reductions of a 64-lane wave by data-parallel primitives (no LDS traffic).

#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace gmm {

// v of the lane that the DPP control word names, the lane's own v where there is none.
template<int Ctrl>
__device__ inline uint32_t dpp(uint32_t v)
{
    return uint32_t(__builtin_amdgcn_update_dpp(int(v), int(v), Ctrl, 0xf, 0xf, false));
}

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

}  // namespace gmm
