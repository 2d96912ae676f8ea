// What the k-NN kernels share: candidate keys and exact distances (device
// side).
#pragma once

#include <float.h>

#include "tbvh_internal.hpp"

namespace tbvh {

constexpr float kFar = FLT_MAX;

template <int D>
__device__ __forceinline__ float box_distance(const float* q, const float* box) {
    float s = 0.0f;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const float delta = fmaxf(box[d] - q[d], fmaxf(0.0f, q[d] - box[D + d]));
        s = d == 0 ? delta * delta : __builtin_fmaf(delta, delta, s);
    }
    return s;
}

__device__ __forceinline__ uint64_t candidate_key(float dist, uint32_t idx) {
    return (static_cast<uint64_t>(__float_as_uint(dist)) << 32) | idx;
}

// Minimum / maximum of two candidate keys by f64 min / max.  A key read as
// an IEEE double is never negative and never NaN: its sign bit is the sign
// of a distance >= 0, and an all-ones exponent field would need a float
// distance with an all-ones exponent (inf/NaN), which is never inserted
// (the largest key holds FLT_MAX).  Such doubles order exactly like the
// 64-bit unsigned keys, and with f64 denormals kept (the default mode;
// distance-0 keys read as denormals) v_min_f64 / v_max_f64 return one
// operand bit for bit.  Written as instructions: the compiler's fmin/fmax
// would first canonicalise each operand, one more instruction per slot.
__device__ __forceinline__ uint64_t key_min(uint64_t a, uint64_t b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(__longlong_as_double(a)), "v"(__longlong_as_double(b)));
    return static_cast<uint64_t>(__double_as_longlong(r));
}
__device__ __forceinline__ uint64_t key_max(uint64_t a, uint64_t b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(__longlong_as_double(a)), "v"(__longlong_as_double(b)));
    return static_cast<uint64_t>(__double_as_longlong(r));
}

// The key of an empty slot, (FLT_MAX, -1): also what a candidate that may
// not enter the list (distance FLT_MAX, inf or NaN) becomes before a merge.
constexpr uint64_t kEmptyKey = (static_cast<uint64_t>(0x7f7fffffu) << 32) | 0xffffffffu;

// Exact distance to a point stored as float4, bit-identical to box_distance
// on the point's degenerate box (lo = hi = p) for every input, NaN and inf
// included.  There, delta = max(p - q, max(0, q - p)); IEEE subtraction is
// sign-symmetric (q - p = -(p - q), also for inf, and NaN for NaN), so
// delta = |p - q| when p - q is not NaN and 0 when it is (max returns the
// non-NaN operand: a NaN query coordinate, or equal infinities, count 0 on
// that axis).  max(|e|, 0) with e = p - q gives exactly that in one
// instruction (abs is a source modifier; arithmetic NaNs are quiet).
template <int D>
__device__ __forceinline__ float point_distance(const float* q, const float4 p) {
    const float pc[3] = {p.x, p.y, p.z};
    float s = 0.0f;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const float e = fmaxf(fabsf(pc[d] - q[d]), 0.0f);
        s = d == 0 ? e * e : __builtin_fmaf(e, e, s);
    }
    return s;
}

}  // namespace tbvh
