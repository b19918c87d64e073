// Small operations over the lanes of a wave.
#pragma once
#include "hd.hpp"

namespace mptg {
namespace {

template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_or_self(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(
        (int)__float_as_uint(v), (int)__float_as_uint(v), CTRL, ROWS, 0xf, false));
}
// Minimum over the wave (no NaN), the same on every lane.
__device__ __forceinline__ float wave_min_f32(float v) {
    v = __builtin_fminf(v, dpp_or_self<0x128, 0xf>(v));  // rows of 16: rotate by 8, 4, 2, 1
    v = __builtin_fminf(v, dpp_or_self<0x124, 0xf>(v));
    v = __builtin_fminf(v, dpp_or_self<0x122, 0xf>(v));
    v = __builtin_fminf(v, dpp_or_self<0x121, 0xf>(v));
    v = __builtin_fminf(v, dpp_or_self<0x142, 0xa>(v));  // lane 15 to row 1, 47 to row 3
    v = __builtin_fminf(v, dpp_or_self<0x143, 0xc>(v));  // lane 31 to rows 2 and 3
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}

__device__ __forceinline__ float lane_f32(float v, int src) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), src));
}

}  // namespace
}  // namespace mptg
