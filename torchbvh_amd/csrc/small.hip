// Small clouds in one work-group each: bounds, keys and the whole stable
// key/value sort in LDS, one launch.
//
// For clouds of up to kSmallCloud rows this replaces the bounds, Morton and
// eleven sort launches of the general sequence (tile counts, scans and
// scatters of four 8-bit passes, sort.hip), whose fixed costs set the time
// of a small build: at 10,000 points those thirteen launches take ~65 us of
// kernel time for 40 kB of keys.  Everything stays in one work-group of
// kSmallThreads threads, and every pass is the same stable counting sort as
// the general scatter (wave64 ballot ranking, per-wave digit counters, LDS
// staging in digit order), so the order is identical: ties in the key keep
// ascending original index (the CUB contract the sort replaces,
// bvh_build.cu:580-594), and the bounds are the same fminf/fmaxf reductions
// from the same seeds (bvh_build.cu:453-494).
//
// The order is that of the unique pairs (key, row), so it need not be reached
// by stable passes.  First the keys are dealt to bins by their top bits, each
// bin's keys to as many sub-bins as it holds keys by the next bits (two rounds
// of LDS counters and a scan each, about a key to a sub-bin wherever the
// density is smooth at the scale of a bin), and a key's place in its sub-bin is
// counted from the pairs there.  Only when a sub-bin holds more than
// kMostInBin keys (many equal codes) do the four stable passes run, whose
// ballot ranking (about 90 instructions per key and pass) bounds them on the one
// CU.  Point ordering by passes and by bins, us: 4,000 3-D points 25 and 15,
// 10,000 53 and 27, in eight clusters 52 and 34; the bins' attempt costs a cloud of a
// few distinct points that then takes the passes 3 to 5 us (10,000 of 64: 50 and
// 55; a limit of 96 keys: 4,000 of 64 24 and 52).
#include "tbvh_internal.hpp"

namespace tbvh {
namespace {

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;

constexpr uint32_t kMostInBin = 32;

// 16-bit counters, two to an LDS word (a cloud has fewer than 2^16 rows).
__device__ __forceinline__ uint32_t count_half(uint32_t* words, uint32_t i) {
    const uint32_t shift = (i & 1u) * 16u;
    return (atomicAdd(&words[i >> 1], 1u << shift) >> shift) & 0xffffu;
}
__device__ __forceinline__ uint32_t read_half(const uint32_t* words, uint32_t i) {
    return reinterpret_cast<const uint16_t*>(words)[i];
}

// Counters (kPer per thread, in order) -> their exclusive prefix sums, with
// the total after the last one.  Starts and ends with a barrier.
template <int kPer>
__device__ __forceinline__ void scan_halves(uint32_t* words, uint32_t* scratch) {
    static_assert(kPer % 2 == 0, "whole words per thread");
    __syncthreads();
    uint32_t w[kPer / 2];
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kPer / 2; ++i) {
        w[i] = words[threadIdx.x * (kPer / 2) + i];
        sum += (w[i] & 0xffffu) + (w[i] >> 16);
    }
    uint32_t total = 0;
    uint32_t run = block_exclusive_sum<kSmallThreads>(sum, scratch, &total);
#pragma unroll
    for (int i = 0; i < kPer / 2; ++i) {
        const uint32_t second = run + (w[i] & 0xffffu);
        words[threadIdx.x * (kPer / 2) + i] = run | second << 16;
        run = second + (w[i] >> 16);
    }
    if (threadIdx.x == 0) words[kSmallThreads * (kPer / 2)] = total;
    __syncthreads();
}

// One cloud per work-group (segment blockIdx.x).  The cloud's rows are dealt
// to all the waves in contiguous ranges of `per_wave` rows (a multiple of
// 64, the fewest that cover it): row j = w * per_wave + i * 64 + l is item i
// of lane l of wave w, so ranking within a wave is ranking in row order, and
// a wave's serial ranking chain is per_wave / 64 = ceil(n / 1024) items long
// whatever kItems is (one item per 1,024 rows: 10 at 10,000 rows, not 16).
// With `bounds`, the cloud's box from (seed_lo, seed_hi) is stored into
// scene_min/max and keys the rows against it; otherwise scene_min/max are
// read.  Passes sort 8-bit digits from first_bit up; the cloud-local order
// goes to `order` (int64) and, if given, the sorted keys to `sorted_keys`.
template <int D, int kItems, int kCurve>
__global__ __launch_bounds__(kSmallThreads) void small_sort_kernel(
    const float* __restrict__ rows, const Segment* segs, int S, UniformPlan plan, float* __restrict__ scene_min,
    float* __restrict__ scene_max, bool bounds, float seed_lo, float seed_hi, int first_bit, int passes,
    int64_t* __restrict__ order, uint32_t* __restrict__ sorted_keys) {
    constexpr int kCap = kItems * kSmallThreads;
    // Bins: about one per key of a full cloud.
    constexpr int kBinBits = kItems <= 4 ? 12 : 14;
    constexpr int kBins = 1 << kBinBits;
    constexpr int kPassWords = kSmallWaves * kRadix;
    constexpr int kBinWords = kBins / 2 + 1;
    __shared__ uint32_t s_keys[kCap];
    // The passes' values; by bins, the rows (16 bits each) and the sub-bins.
    __shared__ uint32_t s_vals[kCap + 1];
    // The passes' digit counters; by bins, the bins.
    __shared__ uint32_t s_count[kPassWords > kBinWords ? kPassWords : kBinWords];
    uint32_t (*s_cnt)[kRadix] = reinterpret_cast<uint32_t (*)[kRadix]>(s_count);
    __shared__ uint32_t s_start[kRadix];
    __shared__ uint32_t s_scan[kSmallWaves];
    __shared__ float s_red[kSmallWaves][2 * D];
    __shared__ float s_box[2 * D];
    const int s = blockIdx.x;
    if (plan.table) store_uniform_table(plan.table, S, plan.n, plan.tree);
    const Segment g = plan.n > 0 ? uniform_segment(s, plan.n, plan.tree) : segs[s];
    const int n = g.n;
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    const int per_wave = (n + kSmallThreads - 1) / kSmallThreads * kWave;
    const int base = wave * per_wave + lane;
    // Item i of this lane is a row of the cloud (the first test is wave-uniform).
    auto valid = [&](int i) { return i * kWave < per_wave && base + i * kWave < n; };

    // The rows are read twice (bounds, then keys; the second read hits in
    // cache), kChunk rows per thread at a time: the loads of a chunk issue
    // together (rows past the cloud read its last row and are masked), so
    // the work-group waits kItems / kChunk round trips per sweep instead of
    // kItems, and no thread holds all its rows (which spills at 16).
    constexpr int kChunk = kItems % 8 == 0 ? 8 : 4;
    static_assert(kItems % kChunk == 0, "whole chunks of rows");
    const PointRow<D>* src = reinterpret_cast<const PointRow<D>*>(rows + g.start * D);
    float lo[D], hi[D];
    if (bounds) {
#pragma unroll
        for (int d = 0; d < D; ++d) { lo[d] = seed_lo; hi[d] = seed_hi; }
#pragma unroll
        for (int c = 0; c < kItems; c += kChunk) {
            PointRow<D> r[kChunk];
#pragma unroll
            for (int u = 0; u < kChunk; ++u) r[u] = src[min(base + (c + u) * kWave, n - 1)];
#pragma unroll
            for (int u = 0; u < kChunk; ++u) {
                if (valid(c + u)) {
#pragma unroll
                    for (int d = 0; d < D; ++d) {
                        lo[d] = fminf(lo[d], r[u].v[d]);
                        hi[d] = fmaxf(hi[d], r[u].v[d]);
                    }
                }
            }
        }
        block_box<D, kSmallThreads>(lo, hi, s_red, s_box);
        __syncthreads();
#pragma unroll
        for (int d = 0; d < D; ++d) { lo[d] = s_box[d]; hi[d] = s_box[D + d]; }
        if (threadIdx.x < D) {
            scene_min[static_cast<int64_t>(s) * D + threadIdx.x] = s_box[threadIdx.x];
            scene_max[static_cast<int64_t>(s) * D + threadIdx.x] = s_box[D + threadIdx.x];
        }
    } else {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            lo[d] = scene_min[static_cast<int64_t>(s) * D + d];
            hi[d] = scene_max[static_cast<int64_t>(s) * D + d];
        }
    }
    uint32_t key[kItems], val[kItems];
#pragma unroll
    for (int c = 0; c < kItems; c += kChunk) {
        PointRow<D> r[kChunk];
#pragma unroll
        for (int u = 0; u < kChunk; ++u) r[u] = src[min(base + (c + u) * kWave, n - 1)];
#pragma unroll
        for (int u = 0; u < kChunk; ++u) {
            const int i = c + u;
            const int j = base + i * kWave;
            // The bits below first_bit (the schedule's key holds two in 3-D) take
            // no part in the order.
            key[i] = valid(i) ? hilbert::sort_key<D, kCurve>(r[u].v, lo, hi) >> first_bit << first_bit : 0xffffffffu;
            val[i] = static_cast<uint32_t>(j);
        }
    }

    {
        constexpr int kLow = morton::key_bits<D>() - kBinBits;  // bits below a bin's
        static_assert(kLow >= 14, "a bin's sub-bins take at most log2(kSmallCloud) bits");
        uint32_t* bins = s_count;
        uint32_t* sub = s_vals;
        uint16_t* rows16 = reinterpret_cast<uint16_t*>(s_vals + kCap / 2 + 1);
        for (int i = threadIdx.x; i < kBinWords; i += kSmallThreads) bins[i] = 0u;
        for (int i = threadIdx.x; i < kCap / 2 + 1; i += kSmallThreads) sub[i] = 0u;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (valid(i)) count_half(bins, key[i] >> kLow);
        }
        scan_halves<kBins / kSmallThreads>(bins, s_scan);
        // A bin of c keys from place s has its floor-log2(c)-bit sub-bins at
        // counters s .. s + c - 1.
        uint32_t at[kItems];
        uint32_t most = 0;
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (valid(i)) {
                const uint32_t b = key[i] >> kLow;
                const uint32_t first = read_half(bins, b);
                const int m = 31 - __builtin_clz(read_half(bins, b + 1) - first);
                const uint32_t slot = first + ((key[i] >> (kLow - m)) & ((1u << m) - 1u));
                const uint32_t arrived = count_half(sub, slot);
                at[i] = slot | arrived << 16;
                most = max(most, arrived);
            }
        }
        if (!__syncthreads_or(most >= kMostInBin)) {
            scan_halves<kItems>(sub, s_scan);
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                if (valid(i)) {
                    const uint32_t place = read_half(sub, at[i] & 0xffffu) + (at[i] >> 16);
                    s_keys[place] = key[i];
                    rows16[place] = static_cast<uint16_t>(val[i]);
                }
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                if (valid(i)) {
                    const uint32_t slot = at[i] & 0xffffu;
                    const uint32_t first = read_half(sub, slot), end = read_half(sub, slot + 1);
                    uint32_t place = first;
                    for (uint32_t j = first; j < end; ++j) {
                        const uint32_t k = s_keys[j];
                        place += k < key[i] || (k == key[i] && rows16[j] < val[i]) ? 1u : 0u;
                    }
                    at[i] = place;
                }
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                if (valid(i)) {
                    s_keys[at[i]] = key[i];
                    rows16[at[i]] = static_cast<uint16_t>(val[i]);
                }
            }
            __syncthreads();
            for (int j = threadIdx.x; j < n; j += kSmallThreads) {
                order[g.start + j] = static_cast<int64_t>(rows16[j]);
                if (sorted_keys) sorted_keys[g.start + j] = s_keys[j];
            }
            return;
        }
    }

    const uint64_t below = (1ull << lane) - 1ull;
    for (int p = 0; p < passes; ++p) {
        const int shift = first_bit + p * kRadixBits;
        for (int i = threadIdx.x; i < kSmallWaves * kRadix; i += kSmallThreads) (&s_cnt[0][0])[i] = 0u;
        __syncthreads();
        // Stable rank of each key among this wave's keys of its digit.
        uint32_t rank[kItems];
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            rank[i] = 0;
            if (i * kWave >= per_wave) continue;  // the wave's rows end before this item
            const bool ok = base + i * kWave < n;
            const uint32_t digit = (key[i] >> shift) & (kRadix - 1);
            const uint64_t peers = match_digit(digit, ok);
            const uint32_t before = static_cast<uint32_t>(__popcll(peers & below));
            const uint32_t prior = ok ? s_cnt[wave][digit] : 0u;
            __builtin_amdgcn_wave_barrier();
            if (ok && before == 0) s_cnt[wave][digit] = prior + static_cast<uint32_t>(__popcll(peers));
            __builtin_amdgcn_wave_barrier();
            rank[i] = prior + before;
        }
        __syncthreads();
        // Thread d < kRadix: the digit's counts in earlier waves, and the
        // cloud's keys of smaller digits.
        const int d = threadIdx.x;
        uint32_t count = 0;
        if (d < kRadix) {
#pragma unroll
            for (int w = 0; w < kSmallWaves; ++w) {
                const uint32_t c = s_cnt[w][d];
                s_cnt[w][d] = count;
                count += c;
            }
        }
        const uint32_t start = block_exclusive_sum<kSmallThreads>(count, s_scan);
        if (d < kRadix) s_start[d] = start;
        __syncthreads();
        // A key's place: smaller digits, then its digit in earlier waves,
        // then earlier in its own wave: a bijection onto [0, n).
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (valid(i)) {
                const uint32_t digit = (key[i] >> shift) & (kRadix - 1);
                const uint32_t at = s_start[digit] + s_cnt[wave][digit] + rank[i];
                s_keys[at] = key[i];
                s_vals[at] = val[i];
            }
        }
        __syncthreads();
        if (p + 1 < passes) {
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                if (valid(i)) {
                    key[i] = s_keys[base + i * kWave];
                    val[i] = s_vals[base + i * kWave];
                }
            }
        }
    }
    for (int j = threadIdx.x; j < n; j += kSmallThreads) {
        order[g.start + j] = static_cast<int64_t>(s_vals[j]);
        if (sorted_keys) sorted_keys[g.start + j] = s_keys[j];
    }
}

template <int D, int kItems>
void launch_items(const float* rows, const Segment* segs, int64_t S, UniformPlan plan, float* scene_min,
                  float* scene_max, bool bounds, float seed_lo, float seed_hi, SortBits bits, int64_t* order,
                  uint32_t* sorted_keys, hipStream_t stream) {
    const unsigned grid = static_cast<unsigned>(S);
    const auto run = [&](auto kernel) {
        kernel<<<grid, kSmallThreads, 0, stream>>>(rows, segs, static_cast<int>(S), plan, scene_min, scene_max, bounds,
                                                   seed_lo, seed_hi, bits.first_bit, bits.passes(), order,
                                                   sorted_keys);
    };
    if (bits.curve == hilbert::kFine) run(small_sort_kernel<D, kItems, hilbert::kFine>);
    else if (bits.curve == hilbert::kSchedule) run(small_sort_kernel<D, kItems, hilbert::kSchedule>);
    else run(small_sort_kernel<D, kItems, hilbert::kMorton>);
}

template <int D>
void launch_d(const float* rows, const Segment* segs, int64_t S, UniformPlan plan, int64_t max_n, float* scene_min,
              float* scene_max, bool bounds, float seed_lo, float seed_hi, SortBits bits, int64_t* order,
              uint32_t* sorted_keys, hipStream_t stream) {
    // Up to 4 keys per thread (51 kB of LDS) to 4,096 rows, else up to 12
    // (133 kB).  At 16 keys per thread (16,384 rows) the stable passes measured
    // slower than the general sequence (full build 130.6 against 121.5 us at
    // 16,384 points), at 10,000 points faster (107.4 against 120.5 us).
    if (max_n <= 4 * kSmallThreads) {
        launch_items<D, 4>(rows, segs, S, plan, scene_min, scene_max, bounds, seed_lo, seed_hi, bits, order,
                           sorted_keys, stream);
    } else {
        launch_items<D, kSmallCloud / kSmallThreads>(rows, segs, S, plan, scene_min, scene_max, bounds, seed_lo,
                                                     seed_hi, bits, order, sorted_keys, stream);
    }
}

// The rows of one sort tile, already in order of their keys' top 16 bits, into
// order of all their bits (nearly), for a schedule, whose order changes no
// result.  Bins over the tile's key range and sub-bins as in the small sort, by
// the key's place in the range.  One read and one write of 8 bytes a row: 8 us at
// 1M rows, 18 at 4M, where two more passes of the global sort took 32 and 66.
// The rows wait in LDS: in registers they took the kernel past 64, one
// work-group per CU in place of two (24 us at 4M rows).
//
// Every call gives the same order: among points with a NaN coordinate a search's
// rows depend on which queries share a wave.  Rows of a slot in the order they
// reach it, which differs from call to call, took 6 and 13 us.  A tile with more than
// kMostInBin rows in a slot stays as it is (1M points and queries, k = 16, ordering
// and search with that limit 32 / 128 / none, us: 8 clusters 758 / 763 / 940, 500 tight ones
// 1208 / 1163 / 1290, 40 copies of each point 309 / 318 / 317).
__global__ __launch_bounds__(kSmallThreads) void refine_kernel(const Segment* __restrict__ segs, int S, int key_bits,
                                                               const uint32_t* __restrict__ keys,
                                                               const uint32_t* __restrict__ vals,
                                                               int64_t* __restrict__ order) {
    constexpr int kItems = kSortTile / kSmallThreads;
    static_assert(kItems % 2 == 0, "whole counter words per thread");
    __shared__ uint32_t bins[kSortTile / 2 + 1];
    __shared__ uint32_t sub[kSortTile / 2 + 1];
    __shared__ uint32_t s_vals[kSortTile];
    __shared__ uint32_t s_scan[kSmallWaves];
    __shared__ int s_seg;
    const int64_t t = blockIdx.x;
    const int s = block_find_segment([&](int i) { return static_cast<int64_t>(segs[i].tile_first); }, S, t, &s_seg);
    const Segment g = segs[s];
    const int lt = static_cast<int>(t - g.tile_first);
    if (lt >= g.tiles) return;  // surplus tile
    const int64_t row0 = g.start + static_cast<int64_t>(lt) * kSortTile;
    const int count = min(kSortTile, g.n - lt * kSortTile);
    uint32_t key[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const int j = i * kSmallThreads + threadIdx.x;
        key[i] = keys[row0 + (j < count ? j : 0)];
        s_vals[j] = vals[row0 + (j < count ? j : 0)];
    }
    const uint32_t low = (1u << (key_bits - 16)) - 1u;
    const uint32_t base = keys[row0] & ~low;
    const float scale = static_cast<float>(kSortTile) / (static_cast<float>((keys[row0 + count - 1] | low) - base) + 1.0f);
    for (int i = threadIdx.x; i < kSortTile / 2 + 1; i += kSmallThreads) {
        bins[i] = 0u;
        sub[i] = 0u;
    }
    __syncthreads();
    float x[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        x[i] = fminf(static_cast<float>(key[i] - base) * scale, static_cast<float>(kSortTile - 1));
        if (i * kSmallThreads + threadIdx.x < count) count_half(bins, static_cast<uint32_t>(x[i]));
    }
    scan_halves<kItems>(bins, s_scan);
    uint32_t at[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        if (i * kSmallThreads + threadIdx.x < count) {
            const uint32_t b = static_cast<uint32_t>(x[i]);
            const uint32_t first = read_half(bins, b), held = read_half(bins, b + 1) - first;
            const uint32_t slot = first + min(static_cast<uint32_t>((x[i] - static_cast<float>(b)) *
                                                                    static_cast<float>(held)), held - 1u);
            at[i] = slot | count_half(sub, slot) << 16;
        }
    }
    // Rows of one slot keep their order in the tile: their arrivals, which
    // differ from call to call, are ranked by it.
    uint32_t most = 0;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        if (i * kSmallThreads + threadIdx.x < count) most = max(most, at[i] >> 16);
    }
    uint16_t* rows16 = reinterpret_cast<uint16_t*>(bins);
    // With many rows of one key or nearly, the tile stays as it is.
    const bool sorted = !__syncthreads_or(most >= kMostInBin);
    if (sorted) {
        scan_halves<kItems>(sub, s_scan);
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int j = i * kSmallThreads + threadIdx.x;
            if (j < count) rows16[read_half(sub, at[i] & 0xffffu) + (at[i] >> 16)] = static_cast<uint16_t>(j);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int j = i * kSmallThreads + threadIdx.x;
            if (j < count) {
                const uint32_t slot = at[i] & 0xffffu;
                const uint32_t first = read_half(sub, slot), end = read_half(sub, slot + 1);
                uint32_t place = first;
                for (uint32_t o = first; o < end; ++o) place += rows16[o] < j ? 1u : 0u;
                at[i] = place;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int j = i * kSmallThreads + threadIdx.x;
            if (j < count) rows16[at[i]] = static_cast<uint16_t>(j);
        }
        __syncthreads();
    }
    for (int j = threadIdx.x; j < count; j += kSmallThreads) {
        order[row0 + j] = static_cast<int64_t>(s_vals[sorted ? rows16[j] : j]);
    }
}

}  // namespace

hipError_t launch_refine(const Segment* segs, int64_t S, int64_t tiles, int key_bits, const uint32_t* keys,
                         const uint32_t* vals, int64_t* order, hipStream_t stream) {
    refine_kernel<<<static_cast<unsigned>(tiles), kSmallThreads, 0, stream>>>(segs, static_cast<int>(S), key_bits, keys,
                                                                             vals, order);
    return hipGetLastError();
}

hipError_t launch_small_sort(const float* rows, int D, const Segment* segs, int64_t S, UniformPlan plan,
                             int64_t max_n, float* scene_min, float* scene_max, bool bounds, float seed_lo,
                             float seed_hi, SortBits bits, int64_t* order, uint32_t* sorted_keys,
                             hipStream_t stream) {
    if (max_n > kSmallCloud || S < 1) return hipErrorInvalidValue;
    if (D == 3) {
        launch_d<3>(rows, segs, S, plan, max_n, scene_min, scene_max, bounds, seed_lo, seed_hi, bits, order,
                    sorted_keys, stream);
    } else {
        launch_d<2>(rows, segs, S, plan, max_n, scene_min, scene_max, bounds, seed_lo, seed_hi, bits, order,
                    sorted_keys, stream);
    }
    return hipGetLastError();
}

}  // namespace tbvh
