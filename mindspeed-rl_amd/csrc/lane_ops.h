// Reductions inside a wavefront by lane operands and scalar registers, without the LDS crossbar that a shuffle goes
// through, for values of 4 and 8 bytes.
#pragma once

#include "mrl_internal.h"

namespace mrl {

// 32 bits of the lane that step kStep of a reduction inside 16 lanes pairs with this one: quad_perm [1,0,3,2],
// [2,3,0,1], row_half_mirror and row_mirror, each of which pairs groups that already agree.  A VALU operand.
template <int kStep>
__device__ __forceinline__ uint32_t lane_partner_bits(uint32_t x) {
    constexpr int kControl[4] = {0xB1, 0x4E, 0x141, 0x140};
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kControl[kStep], 0xf, 0xf, true);
}

template <int kStep>
__device__ __forceinline__ float lane_partner(float x) {
    return __uint_as_float(lane_partner_bits<kStep>(__float_as_uint(x)));
}

template <int kStep>
__device__ __forceinline__ double lane_partner(double x) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const uint32_t lo = lane_partner_bits<kStep>((uint32_t)u), hi = lane_partner_bits<kStep>((uint32_t)(u >> 32));
    return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}

// Over the 2^kSteps lanes around this one, kSteps up to 4.
template <int kSteps>
__device__ __forceinline__ float lanes_max(float x) {
    x = fmaxf(x, lane_partner<0>(x));
    if (kSteps > 1) x = fmaxf(x, lane_partner<1>(x));
    if (kSteps > 2) x = fmaxf(x, lane_partner<2>(x));
    if (kSteps > 3) x = fmaxf(x, lane_partner<3>(x));
    return x;
}

template <int kSteps, typename F>
__device__ __forceinline__ F lanes_sum(F x) {
    x += lane_partner<0>(x);
    if (kSteps > 1) x += lane_partner<1>(x);
    if (kSteps > 2) x += lane_partner<2>(x);
    if (kSteps > 3) x += lane_partner<3>(x);
    return x;
}

// x of lane `lane`, the same in every lane.
__device__ __forceinline__ float lane_value(float x, int lane) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), lane));
}

__device__ __forceinline__ double lane_value(double x, int lane) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}

}  // namespace mrl
