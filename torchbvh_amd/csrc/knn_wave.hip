// Exact k-NN with one wave per query, for calls of few queries.
//
// A traversal with one query per lane (knn.hip) is a chain of about 140
// dependent steps per wave whatever the call's size: 1,000 queries are 16
// waves on a chip of 256 CUs, and the call takes that chain's latency.  Here
// a wave's 64 lanes work on one query: a step tests 64 boxes of the implicit
// tree or 64 points at once, and the chain is about ten steps.
//
// Boxes.  The implicit tree's node at depth L - s covers 2^s consecutive
// Morton-ordered points, and the nodes of a level are consecutive rows, so
// the boxes of 64 sibling runs are one contiguous read.  The wave descends
// six levels at a time: runs of 16 points ("blocks") at the bottom, then of
// 1,024, 65,536, ..., up to a top level of at most 64 nodes.  These boxes
// overlap more than the radix tree's (a run may straddle a large Morton
// cell's border), which costs 64-wide tests little.
//
// List.  One key per lane, ascending over the lanes: the 64 smallest keys
// seen (the first K are the result).  The first four blocks (64 points,
// nearest first) fill it by one bitonic sort over the lanes; later points
// below the k-th key are inserted, or merged 64 at a time.  Keys and
// distances are the traversal's, so the result is the same k smallest
// (distance, index) pairs, bit for bit; a box is skipped only when its
// distance exceeds the k-th distance.
//
// Bound: a lone query takes the chain of dependent reads and exchanges (about
// 15 us for 50,000 points); many, about 1,500 issue slots each.  Measured, call
// time against the traversal: 1,000 queries of 50,000 3-D points at k = 8
// 73 -> 23 us, 10,000 of 10,000 at k = 4 64 -> 31 us (kernel); which calls take
// it: WAVE_MAX_QUERIES in _native.py.
#include <algorithm>

#include "knn_common.hpp"

namespace tbvh {
namespace {

constexpr int kBlockBits = 4;   // points per block: 16
constexpr int kFanBits = 6;     // levels per step: 64 children
constexpr int kInsertMost = 24; // accepted keys of a step inserted one by one

template <int kCtrl>
__device__ __forceinline__ uint64_t dpp_key(uint64_t k) {
    const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(static_cast<uint32_t>(k)), kCtrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(static_cast<uint32_t>(k >> 32)), kCtrl, 0xf, 0xf, true);
    return (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kXor3 = 0x1B;                // quad_perm
constexpr int kXor7 = 0x141, kXor15 = 0x140, kRor8 = 0x128;            // row mirrors, rotate by half a row

// Keys of the two 16-lane rows (kRow16) or two wave halves of each pair, as
// (even / low one's, odd / high one's) in every lane.
template <bool kRow16>
__device__ __forceinline__ void pair_keys(uint64_t k, uint64_t& even, uint64_t& odd) {
    const uint32_t lo = static_cast<uint32_t>(k), hi = static_cast<uint32_t>(k >> 32);
    const auto l = kRow16 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                          : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = kRow16 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                          : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    even = (static_cast<uint64_t>(h[0]) << 32) | l[0];
    odd = (static_cast<uint64_t>(h[1]) << 32) | l[1];
}

// This lane's key becomes the smaller (lane bit kBit clear) or larger of it
// and `other`.
template <int kBit>
__device__ __forceinline__ uint64_t keep(uint64_t k, uint64_t other) {
    const uint64_t mn = key_min(k, other), mx = key_max(k, other);
    return (lane_id() & kBit) ? mx : mn;
}

// Compare-exchange with the lane kStride away.
template <int kStride>
__device__ __forceinline__ uint64_t exchange(uint64_t k) {
    if constexpr (kStride == 1) return keep<1>(k, dpp_key<kXor1>(k));
    else if constexpr (kStride == 2) return keep<2>(k, dpp_key<kXor2>(k));
    else if constexpr (kStride == 4) return keep<4>(k, dpp_key<kXor3>(dpp_key<kXor7>(k)));
    else if constexpr (kStride == 8) return keep<8>(k, dpp_key<kRor8>(k));
    else {
        uint64_t even, odd;
        pair_keys<kStride == 16>(k, even, odd);
        return keep<kStride>(even, odd);
    }
}

// The key of lane 31 - l (of its half) and of lane 63 - l.
__device__ __forceinline__ uint64_t reversed32(uint64_t k) {
    uint64_t even, odd;
    pair_keys<true>(dpp_key<kXor15>(k), even, odd);
    return (lane_id() & 16) ? even : odd;
}
__device__ __forceinline__ uint64_t reversed64(uint64_t k) {
    uint64_t even, odd;
    pair_keys<false>(reversed32(k), even, odd);
    return (lane_id() & 32) ? even : odd;
}

// key_max with a wave-uniform second operand.  A vector instruction may read a
// scalar register only two wait states after another vector instruction (the
// v_readlane that `add` has the key from) wrote it; the compiler inserts them
// for its own instructions and not for those in inline assembly.
__device__ __forceinline__ uint64_t key_max_uniform(uint64_t a, uint64_t b) {
    double r;
    asm("s_nop 1\n\tv_max_f64 %0, %1, %2" : "=v"(r) : "v"(__longlong_as_double(a)), "s"(__longlong_as_double(b)));
    return static_cast<uint64_t>(__double_as_longlong(r));
}

// The next lower lane's key; lane 0 reads 0.
__device__ __forceinline__ uint64_t shifted(uint64_t k) {
    return dpp_key<0x138>(k);  // wave_shr:1
}

// Bitonic sequence over the 64 lanes -> ascending.
__device__ __forceinline__ uint64_t clean64(uint64_t k) {
    k = exchange<32>(k);
    k = exchange<16>(k);
    k = exchange<8>(k);
    k = exchange<4>(k);
    k = exchange<2>(k);
    return exchange<1>(k);
}

// Ascending over the 64 lanes (bitonic sort whose merges start with the
// second run reversed, so every exchange is ascending).
__device__ __forceinline__ uint64_t sort64(uint64_t k) {
    k = keep<1>(k, dpp_key<kXor1>(k));
    k = keep<2>(k, dpp_key<kXor3>(k));
    k = exchange<1>(k);
    k = keep<4>(k, dpp_key<kXor7>(k));
    k = exchange<2>(k);
    k = exchange<1>(k);
    k = keep<8>(k, dpp_key<kXor15>(k));
    k = exchange<4>(k);
    k = exchange<2>(k);
    k = exchange<1>(k);
    k = keep<16>(k, reversed32(k));
    k = exchange<8>(k);
    k = exchange<4>(k);
    k = exchange<2>(k);
    k = exchange<1>(k);
    k = keep<32>(k, reversed64(k));
    k = exchange<16>(k);
    k = exchange<8>(k);
    k = exchange<4>(k);
    k = exchange<2>(k);
    return exchange<1>(k);
}

// Smallest value over the wave.
__device__ __forceinline__ uint32_t wave_least(uint32_t v) {
    const auto step = [&](auto shifted) { v = min(v, static_cast<uint32_t>(shifted)); };
    step(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x111, 0xf, 0xf, false));  // row_shr:1
    step(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x112, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x114, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x118, 0xf, 0xf, false));
    step(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x142, 0xa, 0xf, false));  // row_bcast:15
    step(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), 0x143, 0xc, 0xf, false));  // row_bcast:31
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// Lane (set in `mask`) with the smallest distance, ties within 2^-17 of each
// other to the lower lane.
__device__ __forceinline__ int nearest_lane(float d, uint64_t mask) {
    const bool in = (mask >> lane_id()) & 1ull;
    const uint32_t k = in ? (__float_as_uint(d) & ~63u) | static_cast<uint32_t>(lane_id()) : 0xffffffffu;
    return static_cast<int>(wave_least(k) & 63u);
}

template <int D, int K>
struct WaveQuery {
    const float* nodes;   // this cloud's rows of 2 * D floats
    const float4* pts;    // this cloud's Morton-ordered points
    int n, L, vl, bl;     // points, leaf level, virtual leaves, block level
    float q[D];
    bool filled;          // the first blocks are in the list
    uint64_t list;        // this lane's key, ascending over the lanes
    uint64_t kth;         // key of lane K - 1, or the starting bound's (wave-uniform)
    float worst;          // its distance

    // `bound`: at least K points lie within it (kFar: unknown).
    __device__ __forceinline__ void init(const float* nodes_, const float4* pts_, int n_, float bound) {
        nodes = nodes_;
        pts = pts_;
        n = n_;
        L = tree::leaf_level(n);
        vl = tree::virtual_leaves(n);
        bl = L > kBlockBits ? L - kBlockBits : 0;
        restart(bound);
    }

    // Entries (bound, -1) in every lane: K points displace those below K.
    __device__ __forceinline__ void restart(float bound) {
        filled = false;
        list = candidate_key(bound, 0xffffffffu);
        kth = list;
        worst = bound;
    }

    __device__ __forceinline__ void set_kth() {
        const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(list), K - 1);
        const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(list >> 32), K - 1);
        kth = (static_cast<uint64_t>(hi) << 32) | lo;
        worst = __uint_as_float(hi);
    }

    // Adds the lanes' keys below the k-th one (`in`, the lanes of mask `m`).
    // Few are inserted one by one: the lanes from the key's rank on take
    // their lower neighbour's, 6 instructions (a key past the k-th by then
    // lands past lane K - 1).  Many are sorted over the lanes and merged:
    // the smaller of list and reversed keys is a bitonic sequence of the 64
    // smallest (28 exchanges, about 200 instructions).
    __device__ __forceinline__ void add(uint64_t key, bool in, uint64_t m) {
        if (__popcll(m) > kInsertMost) {
            list = clean64(key_min(list, reversed64(sort64(in ? key : kEmptyKey))));
        } else {
            do {
                const int from = __builtin_ctzll(m);
                m &= m - 1;
                const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(key), from);
                const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(key >> 32), from);
                list = key_min(list, key_max_uniform(shifted(list), (static_cast<uint64_t>(hi) << 32) | lo));
            } while (m != 0);
        }
        set_kth();
    }

    // Distance from the query to node `i` of `level`; +inf past the level's
    // real nodes.
    __device__ __forceinline__ float node_distance(int level, int i) const {
        const int real = tree::real_at_level(vl, L, level);
        if (i >= real) return INFINITY;
        const int row0 = tree::level_first(level) - tree::virtual_above(vl, L, level);
        float box[2 * D];
        const float* b = nodes + static_cast<int64_t>(row0 + i) * (2 * D);
#pragma unroll
        for (int d = 0; d < 2 * D; ++d) box[d] = b[d];
        return box_distance<D>(q, box);
    }

    // The points of the blocks first + (bits of mask), `d` each lane's block
    // distance.
    __device__ __forceinline__ void scan_blocks(int first, uint64_t mask, float d) {
        const int bits = L - bl;
        const int slot = lane_id() & 15;
        while (mask != 0) {
            // Four blocks, 16 lanes each: the nearest four while the list is
            // empty, then in storage order.
            int b[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                b[g] = mask == 0 ? -1 : filled ? static_cast<int>(__builtin_ctzll(mask)) : nearest_lane(d, mask);
                mask = mask == 0 ? 0 : mask & ~(1ull << b[g]);
            }
            const int pick = lane_id() < 32 ? (lane_id() < 16 ? b[0] : b[1]) : (lane_id() < 48 ? b[2] : b[3]);
            const int mine = pick < 0 ? -1 : first + pick;
            const int at = (mine << bits) + slot;
            const bool valid = mine >= 0 && slot < (1 << bits) && at < n;
            const float4 p = pts[valid ? at : 0];
            const float dist = point_distance<D>(q, p);
            const uint64_t key = valid && dist < kFar ? candidate_key(dist, __float_as_uint(p.w)) : kEmptyKey;
            if (!filled) {
                filled = true;
                list = key_min(list, sort64(key));
                set_kth();
            } else {
                const bool in = key < kth;
                const uint64_t m = __ballot(in);
                if (m == 0) continue;
                add(key, in, m);
            }
            mask &= __ballot(d <= worst);
        }
    }

    // Visits the children (at `level`) of node `parent`, six levels up; the
    // level is bl - 6 * kBelow.
    template <int kBelow>
    __device__ __forceinline__ void expand(int parent) {
        const int level = bl - kBelow * kFanBits;
        const int first = parent << kFanBits;
        const float d = node_distance(level, first + lane_id());
        uint64_t mask = __ballot(d <= worst && d < INFINITY);
        if constexpr (kBelow == 0) {
            scan_blocks(first, mask, d);
        } else {
            while (mask != 0) {
                const int c = nearest_lane(d, mask);
                expand<kBelow - 1>(first + c);
                mask &= ~(1ull << c);
                mask &= __ballot(d <= worst);
            }
        }
    }
};

// Wide steps from a top level of at most 64 nodes down to the blocks: four
// cover the accel's largest cloud (2^28 points).
__host__ __device__ inline int wave_steps(int n) {
    const int L = tree::leaf_level(n);
    const int bl = L > kBlockBits ? L - kBlockBits : 0;
    return bl <= kFanBits ? 1 : (bl + kFanBits - 1) / kFanBits;
}

// The list's first K entries (and their rows) into result row `out_row`.
template <int D, int K>
__device__ __forceinline__ void write_list(const KnnArgs& a, uint64_t list, int64_t out_row, int64_t index_offset,
                                           int64_t pstart) {
    if (lane_id() >= K) return;
    const int64_t idx = static_cast<int32_t>(static_cast<uint32_t>(list));
    a.out_indices[out_row * K + lane_id()] = idx >= 0 ? idx + index_offset : idx;
    a.out_distances[out_row * K + lane_id()] = __uint_as_float(static_cast<uint32_t>(list >> 32));
    if (a.out_positions != nullptr) {
        const int C = a.source_cols;
        float* op = a.out_positions + (out_row * K + lane_id()) * C;
        const float* src = a.source_points + (pstart + (idx >= 0 ? idx : 0)) * C;
        for (int c = 0; c < C; ++c) op[c] = idx >= 0 ? src[c] : 0.0f;
    }
}

// kSteps: wave_steps(l.n), or 0 to look it up.
template <int D, int K, int kSteps>
__device__ __forceinline__ void wave_search(const KnnArgs& a, const QueryLoc& l, float bound) {
    WaveQuery<D, K> w;
    w.init((l.second ? a.node_aabbs2 : a.node_aabbs) + l.nstart * (2 * D),
           static_cast<const float4*>(l.second ? a.accel2 : a.accel) + l.pstart, l.n, bound);
#pragma unroll
    for (int d = 0; d < D; ++d) w.q[d] = a.queries[l.row * D + d];
    // A second time, without the bound, when it kept out points that it stands
    // for: the boxes do not bound the distance of a point with a NaN
    // coordinate, which the traversal may have reached on another way.
    while (true) {
        switch (kSteps > 0 ? kSteps : wave_steps(l.n)) {
            case 1: w.template expand<0>(0); break;
            case 2: w.template expand<1>(0); break;
            case 3: w.template expand<2>(0); break;
            default: w.template expand<3>(0); break;
        }
        if (!(bound < kFar) || static_cast<uint32_t>(w.kth) != 0xffffffffu) break;
        bound = kFar;
        w.restart(bound);
    }
    write_list<D, K>(a, w.list, l.out_row, l.index_offset, l.pstart);
}

// The plain call has a kernel for each number of steps: a lone wave's time is
// partly its cold instruction fetches (1,000 queries of 50,000 points 28 us with
// the number looked up, 24 us without).
template <int D, int K, bool kOrdered, bool kRagged, int kSteps>
__global__ __launch_bounds__(kWave) void knn_wave_kernel(KnnArgs a) {
    const QueryLoc l = locate<kOrdered, kRagged, false, false>(a, blockIdx.x);
    if (l.row < 0) return;  // a corrupt order never indexes out of range
    wave_search<D, K, kSteps>(a, l, kFar);
}

// The queries that the traversal's waves gave up (KnnArgs::tail_masks), one
// after the other per wave.  Work-group b takes lane b % 64 of every
// stride-th traversal work-group, so queries given up together, by one wave
// or by its neighbours, go to different work-groups (four lanes per work-group
// read the marks in 5 us instead of 6 at 18,400 work-groups, but the routed
// search of 357,000 queries of surface clouds went 1.7 -> 4.4 ms).
template <int K, bool kOrdered, bool kRagged, bool kRouted>
__global__ __launch_bounds__(kWave) void knn_tail_kernel(KnnArgs a, int groups) {
    const int stride = static_cast<int>(gridDim.x) / kWave;
    const int slot = static_cast<int>(blockIdx.x) % kWave;
    for (int first = static_cast<int>(blockIdx.x) / kWave; first < groups; first += stride * kWave) {
        const int g = first + lane_id() * stride;
        // The traversal wrote the marks of the work-groups that had queries;
        // this one looks at positions inside the call or, in a fallback,
        // inside their sub-list (few work-groups have any).
        const int r = g / kXcds;
        bool marked = g < groups;
        if (a.fb_list != nullptr) {
            const int sub = g % kXcds * kGridSubLists + r % kGridSubLists;
            const int64_t at = static_cast<int64_t>(r / kGridSubLists) * kKnnBlock + slot;
            marked = marked && at < a.fb_count[sub * kCountStride];
        } else {
            const int64_t tile = static_cast<int64_t>(g % kXcds) * (groups / kXcds) + r;
            marked = marked && tile * kKnnBlock + slot < a.total_q;
        }
        const uint64_t mask = marked ? a.tail_masks[g] : 0;
        uint64_t todo = __ballot((mask >> slot) & 1ull);
        while (todo != 0) {
            const int block = first + __builtin_ctzll(todo) * stride;
            todo &= todo - 1;
            // The launch position of lane `slot` of that work-group, as in
            // the traversal.
            const int xcd = block % kXcds, rest = block / kXcds;
            int64_t gid = (static_cast<int64_t>(xcd) * (groups / kXcds) + rest) * kKnnBlock + slot;
            if (a.fb_list != nullptr) {
                const int sub = xcd * kGridSubLists + rest % kGridSubLists;
                gid = a.fb_list[sub * a.fb_seg + static_cast<int64_t>(rest / kGridSubLists) * kKnnBlock + slot];
            }
            const QueryLoc l = locate<kOrdered, kRagged, kRouted, false>(a, gid);
            if (l.row >= 0) wave_search<3, K, 0>(a, l, a.tail_bounds[gid]);
        }
    }
}

template <int D, int K>
void launch_wave(const KnnArgs& a, bool ragged, hipStream_t stream) {
    const unsigned grid = static_cast<unsigned>(a.total_q);
    const bool ordered = a.order != nullptr;
    if (ragged && ordered) knn_wave_kernel<D, K, true, true, 0><<<grid, kWave, 0, stream>>>(a);
    else if (ragged) knn_wave_kernel<D, K, false, true, 0><<<grid, kWave, 0, stream>>>(a);
    else if (ordered) knn_wave_kernel<D, K, true, false, 0><<<grid, kWave, 0, stream>>>(a);
    else switch (wave_steps(a.num_leaves)) {
        case 1: knn_wave_kernel<D, K, false, false, 1><<<grid, kWave, 0, stream>>>(a); break;
        case 2: knn_wave_kernel<D, K, false, false, 2><<<grid, kWave, 0, stream>>>(a); break;
        case 3: knn_wave_kernel<D, K, false, false, 3><<<grid, kWave, 0, stream>>>(a); break;
        default: knn_wave_kernel<D, K, false, false, 4><<<grid, kWave, 0, stream>>>(a); break;
    }
}

template <int D>
hipError_t launch_wave_k(const KnnArgs& a, int K, bool ragged, hipStream_t stream) {
    switch (K) {
        case 4: launch_wave<D, 4>(a, ragged, stream); break;
        case 8: launch_wave<D, 8>(a, ragged, stream); break;
        case 16: launch_wave<D, 16>(a, ragged, stream); break;
        case 32: launch_wave<D, 32>(a, ragged, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int K>
void launch_tail(const KnnArgs& a, bool ragged, hipStream_t stream) {
    // The traversal's grid (knn.hip launch_dk); 64 work-groups per stride.
    const int64_t tiles = (a.total_q + kKnnBlock - 1) / kKnnBlock;
    const int groups = static_cast<int>((tiles + kXcds - 1) / kXcds * kXcds);
    const unsigned grid = static_cast<unsigned>(std::min((groups + kWave - 1) / kWave, 128) * kWave);
    const bool ordered = a.order != nullptr;
    if (a.routes != nullptr) knn_tail_kernel<K, true, false, true><<<grid, kWave, 0, stream>>>(a, groups);
    else if (ragged && ordered) knn_tail_kernel<K, true, true, false><<<grid, kWave, 0, stream>>>(a, groups);
    else if (ragged) knn_tail_kernel<K, false, true, false><<<grid, kWave, 0, stream>>>(a, groups);
    else if (ordered) knn_tail_kernel<K, true, false, false><<<grid, kWave, 0, stream>>>(a, groups);
    else knn_tail_kernel<K, false, false, false><<<grid, kWave, 0, stream>>>(a, groups);
}

}  // namespace

hipError_t launch_knn_tail(const KnnArgs& a, int D, int K, bool ragged, hipStream_t stream) {
    if (a.total_q == 0) return hipSuccess;
    if (D != 3) return hipErrorInvalidValue;  // tail_workspace_bytes
    switch (K) {
        case 4: launch_tail<4>(a, ragged, stream); break;
        case 8: launch_tail<8>(a, ragged, stream); break;
        case 16: launch_tail<16>(a, ragged, stream); break;
        case 32: launch_tail<32>(a, ragged, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_knn_wave(const KnnArgs& a, int D, int K, bool ragged, hipStream_t stream) {
    if (a.total_q == 0) return hipSuccess;
    return D == 3 ? launch_wave_k<3>(a, K, ragged, stream) : launch_wave_k<2>(a, K, ragged, stream);
}

}  // namespace tbvh
