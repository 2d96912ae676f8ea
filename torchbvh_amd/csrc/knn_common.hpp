// What the k-NN kernels share (device side): candidate keys, exact
// distances, launch positions.
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

// One wave per work-group: measured against 256 threads, -3.5% at cfg2 and
// -14% at cfg5, whose waves differ most in cost (finer-grained balancing
// over the CUs); 128 falls between, 512 is 13-24% slower.
constexpr int kKnnBlock = 64;
constexpr int kXcds = 8;               // MI355X: work-groups are dealt round-robin over 8 XCDs

// The cell-block search's failure lists (launch positions left for the next
// stage) are cut into kXcds * kGridSubLists sub-lists, each with its own
// count, filled by one atomic add per wave.  Work-group b's sub-list is that
// of its XCD share (b % kXcds, as in the tile map) and of the residue of its
// local tile index (b / kXcds) mod kGridSubLists; the next stage's
// work-group b reads chunk (b / kXcds) / kGridSubLists of the same
// sub-list, so that it takes failures of tiles near its own.  One count per
// XCD share measured 375 us for the first pass at cfg3, where every wave
// fails at once: same-address atomics serialise (about 90 ns each).  The
// counts lie kCountStride words apart, each on a 128-byte line of its own.
constexpr int kGridSubLists = 64;
constexpr int kCountStride = 32;
constexpr int kGridCounts = kXcds * kGridSubLists;  // per list
__device__ __forceinline__ int grid_sublist() {
    return static_cast<int>(blockIdx.x % kXcds) * kGridSubLists + static_cast<int>(blockIdx.x / kXcds) % kGridSubLists;
}
__device__ __forceinline__ int64_t grid_chunk_start() {
    return static_cast<int64_t>(blockIdx.x / kXcds / kGridSubLists) * kKnnBlock;
}

// Where query `gid` of the launch reads and writes: its cloud, its input row
// and output row, and the structure it searches.
struct QueryLoc {
    int64_t row;           // input row (queries), -1 for a corrupt order entry
    int64_t out_row;       // result row
    int64_t pstart;        // the cloud's first point row
    int64_t nstart;        // the cloud's first node row (implicit tree)
    int64_t index_offset;  // added to result indices (false route)
    int n;                 // the cloud's points
    bool second;           // false route: the second structure
};

template <bool kOrdered, bool kRagged, bool kRouted, bool kAccel>
__device__ __forceinline__ QueryLoc locate(const KnnArgs& a, int64_t gid) {
    QueryLoc l;
    int64_t seg, qbase, qcount;
    if constexpr (kRagged) {
        seg = find_segment([&](int i) { return a.query_offsets[i]; }, static_cast<int>(a.B), gid);
        qbase = a.query_offsets[seg];
        qcount = a.query_offsets[seg + 1] - qbase;
        l.pstart = a.point_offsets[seg];
        l.n = static_cast<int>(a.point_offsets[seg + 1] - l.pstart);
        l.nstart = kAccel ? 0 : a.node_offsets[seg];
    } else {
        seg = gid / a.M;
        qbase = seg * a.M;
        qcount = a.M;
        l.n = a.num_leaves;
        l.pstart = seg * static_cast<int64_t>(l.n);
        l.nstart = seg * static_cast<int64_t>(a.num_real_nodes);
    }
    const int64_t local = gid - qbase;
    const int64_t qi = kOrdered ? a.order[qbase + local] : local;
    l.row = qi < 0 || qi >= qcount ? -1 : qbase + qi;  // a corrupt order never indexes out of range
    // Spatial output (knn_query.cu:147-148) keeps the launch (Morton) order.
    l.out_row = a.spatial_output ? gid : l.row;
    l.second = false;
    l.index_offset = 0;
    if (kRouted && l.row >= 0 && a.routes[l.row] == 0) {
        // False route (knn_query.cu:205-217): the second structure, indices
        // after the first's points.
        l.second = true;
        l.index_offset = l.n;
        l.n = a.num_leaves2;
        l.pstart = seg * static_cast<int64_t>(l.n);
        l.nstart = seg * static_cast<int64_t>(a.num_real_nodes2);
    }
    return l;
}

}  // namespace tbvh
