// Neighbour-value accumulation of interpolate_displaced.
//
// The reference loops over the k neighbour ranks in Python, each step a
// gather of the neighbours' rows and two broadcast multiply-adds over the
// whole (B, N, H, Ch) tensor, and finally, after asking the host whether any
// exact hit exists, swaps in the plain mean of the exact hits
// (torchbvh/_multihead.py:123-144).  Here one thread owns V channels of one
// query row and walks the ranks in the same order with the same two
// roundings per step (product, then sum; the library is built with
// -ffp-contract=off), so both sums are bit-identical, the exact-hit count
// is a sum of ones and the mean is one correctly rounded division, as in
// the reference.  No gathered rows are materialised and no host
// synchronisation decides whether any exact hit exists.
#include "tbvh_internal.hpp"

namespace tbvh {
namespace {

constexpr int64_t kMaxGrid = int64_t{1} << 20;  // work-groups per launch

template <int V>
struct Vec;
template <>
struct Vec<1> {
    using T = float;
};
template <>
struct Vec<4> {
    using T = float4;
};

template <int V>
__device__ __forceinline__ float lane(const typename Vec<V>::T& v, int i) {
    if constexpr (V == 1) {
        return v;
    } else {
        return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
    }
}

template <int V>
__device__ __forceinline__ void interpolate_item(const float* __restrict__ values,
                                                 const int64_t* __restrict__ indices,
                                                 const float* __restrict__ weights,
                                                 const uint8_t* __restrict__ exact, int64_t t, int64_t groups,
                                                 int64_t N, int64_t H, int64_t C, int K, float* __restrict__ out) {
    using T = typename Vec<V>::T;
    const int64_t r = t / groups;              // query row (b, n, h)
    const int64_t c = (t - r * groups) * V;    // first channel
    const int64_t h = r % H;
    const int64_t b = r / (N * H);
    float acc[V], ex[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = ex[i] = 0.0f;
    float hits = 0.0f;
    for (int j = 0; j < K; ++j) {
        const int64_t idx = indices[r * K + j];
        const float w = weights[r * K + j];
        const float e = exact[r * K + j] ? 1.0f : 0.0f;
        hits = hits + e;
        T v{};
        if (idx >= 0 && idx < N) v = *reinterpret_cast<const T*>(values + ((b * N + idx) * H + h) * C + c);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const float x = lane<V>(v, i);
            acc[i] = acc[i] + x * w;
            ex[i] = ex[i] + x * e;
        }
    }
    T res;
    float* o = reinterpret_cast<float*>(&res);
#pragma unroll
    for (int i = 0; i < V; ++i) o[i] = hits > 0.0f ? ex[i] / hits : acc[i];
    *reinterpret_cast<T*>(out + r * C + c) = res;
}

// Grid-stride over (row, channel group) items: the grid is capped, since a
// launch holds fewer than 2^32 work-items.
template <int V>
__global__ __launch_bounds__(kBlock) void interpolate_kernel(const float* __restrict__ values,
                                                             const int64_t* __restrict__ indices,
                                                             const float* __restrict__ weights,
                                                             const uint8_t* __restrict__ exact, int64_t rows,
                                                             int64_t N, int64_t H, int64_t C, int K,
                                                             float* __restrict__ out) {
    const int64_t groups = C / V;  // V-channel groups per row
    const int64_t items = rows * groups;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; t < items; t += stride) {
        interpolate_item<V>(values, indices, weights, exact, t, groups, N, H, C, K, out);
    }
}

// First launch of the backward: for entry e = (n * H + h) * K + j of a cloud its
// target row idx * H + h (the sort key), its coefficient - the weight, or, in a
// row with exact hits, minus their count for a hit (the gradient is divided by
// it, as the forward divides) and 0 for the others - and every tile's count of
// the first sort digit.
__global__ __launch_bounds__(kBlock) void interpolate_keys_kernel(const int64_t* __restrict__ indices,
                                                                  const float* __restrict__ weights,
                                                                  const uint8_t* __restrict__ exact, Segment* segs,
                                                                  int S, int N, int H, int K,
                                                                  uint32_t* __restrict__ keys,
                                                                  float* __restrict__ coef,
                                                                  uint32_t* __restrict__ tile_hist,
                                                                  int64_t tstride) {
    __shared__ int s_seg;
    __shared__ uint32_t s_cnt[kRadix];
    const int per_cloud = N * H * K;
    store_uniform_table(segs, S, per_cloud, false);
    int seg;
    const Segment g = first_launch_segment(segs, S, UniformPlan{segs, per_cloud, false}, blockIdx.x, &s_seg, &seg);
    for (int i = threadIdx.x; i < kRadix; i += kBlock) s_cnt[i] = 0u;
    __syncthreads();
    const bool words = K % 4 == 0 && reinterpret_cast<uintptr_t>(exact) % 4 == 0;
    const int lt = static_cast<int>(blockIdx.x - g.tile_first);
    const int count = lt < g.tiles ? min(kSortTile, g.n - lt * kSortTile) : 0;
    for (int i = threadIdx.x; i < count; i += kBlock) {
        const int e = lt * kSortTile + i;
        const int row = e / K;
        const int64_t first = g.start + static_cast<int64_t>(row) * K;
        // The row's flags (bytes of 0 or 1) as words where they allow it.
        int hits = 0;
        if (words) {
            for (int j = 0; j < K; j += 4) hits += __popc(*reinterpret_cast<const uint32_t*>(exact + first + j));
        } else {
            for (int j = 0; j < K; ++j) hits += exact[first + j] ? 1 : 0;
        }
        const int64_t idx = indices[g.start + e];
        const bool valid = idx >= 0 && idx < N;
        const uint32_t key = valid ? static_cast<uint32_t>(idx) * H + row % H : 0u;
        const float c = hits == 0 ? weights[g.start + e] : exact[g.start + e] ? -static_cast<float>(hits) : 0.0f;
        keys[g.start + e] = key;
        coef[g.start + e] = valid ? c : 0.0f;
        atomicAdd(&s_cnt[key & (kRadix - 1)], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kRadix; i += kBlock) tile_hist[hist_at(i, blockIdx.x, tstride)] = s_cnt[i];
}

// One thread per V channels of a target row: its run of sorted entries, found
// by a binary search of the row's cloud, summed in order.
template <int V>
__global__ __launch_bounds__(kBlock) void interpolate_collect_kernel(const float* __restrict__ grad,
                                                                     const uint32_t* __restrict__ keys,
                                                                     const int64_t* __restrict__ order,
                                                                     const float* __restrict__ coef, int64_t rows,
                                                                     int cloud_rows, int C, int K,
                                                                     float* __restrict__ out) {
    using T = typename Vec<V>::T;
    const int groups = C / V;
    const int64_t items = rows * groups;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlock;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; t < items; t += stride) {
        const int64_t r = t / groups;
        const int c = static_cast<int>(t - r * groups) * V;
        const int64_t b = r / cloud_rows;
        const uint32_t target = static_cast<uint32_t>(r - b * cloud_rows);
        const int n = cloud_rows * K;
        const int64_t first = b * n;
        const uint32_t* k = keys + first;
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = lo + ((hi - lo) >> 1);
            if (k[mid] < target) lo = mid + 1;
            else hi = mid;
        }
        float acc[V];
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = 0.0f;
        for (; lo < n && k[lo] == target; ++lo) {
            const int e = static_cast<int>(order[first + lo]);
            const float w = coef[first + e];
            const int64_t src = b * cloud_rows + e / K;
            const T g = *reinterpret_cast<const T*>(grad + src * C + c);
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float x = lane<V>(g, i);
                acc[i] = acc[i] + (w < 0.0f ? x / -w : x * w);
            }
        }
        T res;
        float* o = reinterpret_cast<float*>(&res);
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = acc[i];
        *reinterpret_cast<T*>(out + r * C + c) = res;
    }
}

}  // namespace

hipError_t launch_interpolate_backward(const float* grad, const int64_t* indices, const float* weights,
                                       const uint8_t* exact, int64_t B, int64_t N, int64_t H, int64_t C, int K,
                                       Segment* segs, int64_t tiles, const SortBuffers& sb, int64_t* order,
                                       float* coef, float* out, hipStream_t stream) {
    const int64_t cloud_rows = N * H;
    int bits = 1;
    while ((int64_t{1} << bits) < cloud_rows) ++bits;
    const SortBits range{0, bits};
    interpolate_keys_kernel<<<static_cast<unsigned>(tiles), kBlock, 0, stream>>>(
        indices, weights, exact, segs, static_cast<int>(B), static_cast<int>(N), static_cast<int>(H), K, sb.keys_a,
        coef, sb.tile_hist, sb.tstride);
    // The buffer that the last pass does not read.
    uint32_t* sorted = range.passes() % 2 == 0 ? sb.keys_a : sb.keys_b;
    hipError_t e = launch_sort(segs, B, tiles, range, sb, order, sorted, stream);
    if (e != hipSuccess) return e;
    const bool vec = C % 4 == 0 && reinterpret_cast<uintptr_t>(grad) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(out) % 16 == 0;
    const int64_t items = B * cloud_rows * (vec ? C / 4 : C);
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>((items + kBlock - 1) / kBlock, kMaxGrid));
    if (vec) {
        interpolate_collect_kernel<4><<<grid, kBlock, 0, stream>>>(grad, sorted, order, coef, B * cloud_rows,
                                                                   static_cast<int>(cloud_rows), static_cast<int>(C),
                                                                   K, out);
    } else {
        interpolate_collect_kernel<1><<<grid, kBlock, 0, stream>>>(grad, sorted, order, coef, B * cloud_rows,
                                                                   static_cast<int>(cloud_rows), static_cast<int>(C),
                                                                   K, out);
    }
    return hipGetLastError();
}

hipError_t launch_interpolate(const float* values, const int64_t* indices, const float* weights,
                              const uint8_t* exact, int64_t rows, int64_t N, int64_t H, int64_t C, int K,
                              float* out, hipStream_t stream) {
    const bool vec = C % 4 == 0 && reinterpret_cast<uintptr_t>(values) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(out) % 16 == 0;
    const int64_t items = rows * (vec ? C / 4 : C);
    if (items == 0) return hipSuccess;
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>((items + kBlock - 1) / kBlock, kMaxGrid));
    if (vec) {
        interpolate_kernel<4><<<grid, kBlock, 0, stream>>>(values, indices, weights, exact, rows, N, H, C, K, out);
    } else {
        interpolate_kernel<1><<<grid, kBlock, 0, stream>>>(values, indices, weights, exact, rows, N, H, C, K, out);
    }
    return hipGetLastError();
}

}  // namespace tbvh
