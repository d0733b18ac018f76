// primitives.hip -- project-written sort, scan and compaction for gfx950.
//
// Replaces the reference's CUB/Thrust calls (cub::DeviceRadixSort SortKeys /
// SortPairs, thrust scans, copy_if; src/coarsen.cu:898-934,1017,1069-1111,
// 1336-1339,1550; src/refine_incremental.cuh:277).
//
// Radix sort: stable LSD over 8-bit digits. Per pass:
//   1. digit histogram of each 2048- or 4096-key tile (LDS counters);
//   2. exclusive scan of the digit-major [256 x tiles] histogram (global bases);
//   3. scatter: each wave ranks its keys with a 64-lane multisplit (eight
//      ballots give the lanes sharing a digit), waves are combined in LDS, the
//      tile is staged in LDS in digit order and written out so that consecutive
//      threads store consecutive addresses of one digit run.
// Inputs of at most 8192 keys (four tiles) are sorted in one launch instead:
// three or more launches per 8-bit pass cost more than comparing all pairs.
#include "internal.hpp"
#include "scan.hpp"

namespace gpart_hip {
namespace {

// A tile's shape: the threads of its workgroup and the keys of each.
template <int Threads, int Items>
struct Tile {
    static constexpr int kThreads = Threads;
    static constexpr int kItems = Items;
    static constexpr int kWaves = Threads / kWave;
    static constexpr int kKeys = Threads * Items;
    __device__ static __forceinline__ std::int64_t item(int wave, int it, int lane) {
        return static_cast<std::int64_t>(wave) * (kWave * Items) + it * kWave + lane;
    }
};
using SmallTile = Tile<256, 8>;
using LargeTile = Tile<512, 8>;
// From here on large tiles: a digit's run in a tile is twice as long and the digit-major
// histograms, stored and scanned 4 bytes apart by tiles, are half as many. A pass over
// 32 Mi keys, histogram and scatter: 84 + 174 -> 69 + 166 us, with 4-byte values
// 84 + 296 -> 69 + 265; tiles of 8,192 keys lose more in the scatter (176, 213) than the
// histogram gains (57). 4 Mi keys: 10.4 + 21.0 -> 7.5 + 20.9 us; 1 Mi keys: no difference;
// smaller sorts need the tiles to fill the chip.
constexpr std::int64_t kLargeSort = std::int64_t{1} << 21;
constexpr int kDigits = 256;
// Sorts of at most this many tiles scan the digit histograms inside each scatter
// workgroup (at most 256 x 64 loads) instead of two scan launches per pass.
constexpr std::int64_t kInlineHistogramTiles = 64;

template <typename S>
__global__ void __launch_bounds__(S::kThreads) radix_histogram_kernel(const std::uint64_t* keys, std::int64_t n, int shift,
                                                                      std::uint64_t mask, std::uint32_t* hist,
                                                                      std::int64_t tiles) {
    constexpr int kSortThreads = S::kThreads, kSortWaves = S::kWaves, kSortItems = S::kItems, kSortTile = S::kKeys;
    __shared__ std::uint32_t counts[kSortWaves][kDigits];
    for (int i = threadIdx.x; i < kSortWaves * kDigits; i += kSortThreads)
        (&counts[0][0])[i] = 0;
    __syncthreads();
    const int wave = threadIdx.x / kWave, lane = lane_id();
    const std::int64_t tile_start = static_cast<std::int64_t>(blockIdx.x) * kSortTile;
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
        const std::int64_t idx = tile_start + S::item(wave, it, lane);
        if (idx < n) {
            const int d = static_cast<int>((keys[idx] >> shift) & mask);
            atomicAdd(&counts[wave][d], 1U);
        }
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kDigits; d += kSortThreads) {
        std::uint32_t total = 0;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) total += counts[w][d];
        hist[static_cast<std::int64_t>(d) * tiles + blockIdx.x] = total;
    }
}

// offsets: the digit-major exclusive scan of the tiles' histograms, or, with
// raw_histogram, the histograms themselves, which each workgroup then scans
// for its own tile (grids of at most kInlineHistogramTiles tiles).
template <typename S, typename V, bool HasValues>
__global__ void __launch_bounds__(S::kThreads) radix_scatter_kernel(const std::uint64_t* keys_in, std::uint64_t* keys_out,
                                                                    const V* values_in, V* values_out, std::int64_t n,
                                                                    int shift, std::uint64_t mask,
                                                                    const std::uint32_t* offsets, std::int64_t tiles,
                                                                    int raw_histogram) {
    constexpr int kSortThreads = S::kThreads, kSortWaves = S::kWaves, kSortItems = S::kItems, kSortTile = S::kKeys;
    __shared__ std::uint32_t wave_counts[kSortWaves][kDigits];
    __shared__ std::uint32_t digit_start[kDigits + 1];
    __shared__ std::uint32_t global_base[kDigits];
    __shared__ std::uint64_t stage_keys[kSortTile];
    __shared__ V stage_values[HasValues ? kSortTile : 1];
    __shared__ std::uint32_t scan_waves[kSortWaves + 1];

    const int wave = threadIdx.x / kWave, lane = lane_id();
    for (int i = threadIdx.x; i < kSortWaves * kDigits; i += kSortThreads)
        (&wave_counts[0][0])[i] = 0;
    __syncthreads();
    const std::int64_t tile_start = static_cast<std::int64_t>(blockIdx.x) * kSortTile;
    const int tile_valid = static_cast<int>(n - tile_start < kSortTile ? n - tile_start : kSortTile);

    std::uint64_t key[kSortItems];
    V value[kSortItems];
    int digit[kSortItems];
    std::uint32_t rank[kSortItems];
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
        const std::int64_t idx = tile_start + S::item(wave, it, lane);
        const bool valid = idx < n;
        key[it] = valid ? keys_in[idx] : 0;
        if constexpr (HasValues) value[it] = valid ? values_in[idx] : V{};
        const int d = valid ? static_cast<int>((key[it] >> shift) & mask) : 0;
        digit[it] = valid ? d : -1;
        // the lanes of the same digit, bit by bit: ~(ballot ^ own bit), in 32-bit halves
        const std::uint64_t in_tile = __ballot(valid);
        unsigned low = static_cast<unsigned>(in_tile), high = static_cast<unsigned>(in_tile >> 32);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int own = (d << (31 - b)) >> 31;  // all ones where bit b is set
            const std::uint64_t set = __ballot(own != 0);
            low &= ~(static_cast<unsigned>(set) ^ static_cast<unsigned>(own));
            high &= ~(static_cast<unsigned>(set >> 32) ^ static_cast<unsigned>(own));
        }
        std::uint32_t before = 0;
        if (valid) before = wave_counts[wave][d];
        const std::uint32_t mine = __builtin_amdgcn_mbcnt_hi(high, __builtin_amdgcn_mbcnt_lo(low, 0U));
        rank[it] = before + mine;
        // the lowest peer publishes the new running count
        if (valid && mine == 0) wave_counts[wave][d] = before + __popc(low) + __popc(high);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // per digit: wave offsets within the tile, digit totals
    std::uint32_t digit_total = 0;
    std::uint32_t all_tiles = 0, tiles_before = 0;  // raw_histogram: the digit over all tiles, and before this one
    if (threadIdx.x < kDigits) {
        const int d = threadIdx.x;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
            const std::uint32_t c = wave_counts[w][d];
            wave_counts[w][d] = digit_total;
            digit_total += c;
        }
        if (raw_histogram) {
            const std::uint32_t* row = offsets + static_cast<std::int64_t>(d) * tiles;
            for (std::int64_t b = 0; b < tiles; ++b) {
                const std::uint32_t c = row[b];
                all_tiles += c;
                tiles_before += b < static_cast<std::int64_t>(blockIdx.x) ? c : 0;
            }
        } else {
            global_base[d] = offsets[static_cast<std::int64_t>(d) * tiles + blockIdx.x];
        }
    }
    if (raw_histogram) {  // the same branch in every thread
        std::uint32_t everything;
        const std::uint32_t digit_first = block_exclusive_scan(all_tiles, SumOp<std::uint32_t>{}, &everything,
                                                               scan_waves);
        if (threadIdx.x < kDigits) global_base[threadIdx.x] = digit_first + tiles_before;
    }
    std::uint32_t total;
    const std::uint32_t start = block_exclusive_scan(digit_total, SumOp<std::uint32_t>{}, &total, scan_waves);
    if (threadIdx.x < kDigits) digit_start[threadIdx.x] = start;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
        if (digit[it] < 0) continue;
        const int d = digit[it];
        const std::uint32_t pos = digit_start[d] + wave_counts[wave][d] + rank[it];
        stage_keys[pos] = key[it];
        if constexpr (HasValues) stage_values[pos] = value[it];
    }
    __syncthreads();
    for (int j = threadIdx.x; j < tile_valid; j += kSortThreads) {
        const std::uint64_t k = stage_keys[j];
        const int d = static_cast<int>((k >> shift) & mask);
        const std::int64_t out = static_cast<std::int64_t>(global_base[d]) + (j - static_cast<int>(digit_start[d]));
        keys_out[out] = k;
        if constexpr (HasValues) values_out[out] = stage_values[j];
    }
}

// Stable sort of at most kRankSortMax keys by their bits [shift, shift + width) in one
// launch: an entry's place is the number of entries that come before it, counted against
// all keys. A workgroup has kRankEntries entries, their digits in scalar registers; its
// waves take every 16th run of 64 keys, a key per lane, so that one vector compare and
// one population count serve 64 pairs. The n^2 / 64 compares are spread over all CUs,
// without barriers or dependent passes. 64-bit digits of 1,000, 2,000, 4,096 and 8,192
// keys: 5.6, 6.4, 9.8 and 21 us (a bitonic network in one workgroup: 17, 25, 46 and 96);
// of 16,384 keys 61 us and of 32,768 keys 210 us, where the passes of 8 bits below take
// 160 and 170 us, 90 us for 31 bits and 45 us for 16: the line is drawn at 8,192.
constexpr int kRankSortMax = 8192;
constexpr int kRankEntries = 16;
constexpr int kRankWaves = 16;

template <typename D>
__device__ __forceinline__ D uniform(D v) {
    if constexpr (sizeof(D) == 4)
        return read_lane(v, 0);
    else
        return static_cast<D>(read_lane(static_cast<unsigned long long>(v), 0));
}

template <typename V, bool HasValues, typename D>
__global__ void __launch_bounds__(kRankWaves* kWave) rank_sort_kernel(const std::uint64_t* keys_in,
                                                                      std::uint64_t* keys_out, const V* values_in,
                                                                      V* values_out, int n, int shift,
                                                                      std::uint64_t mask) {
    static_assert(kWave % kRankEntries == 0, "a workgroup's entries lie in one run of keys");
    __shared__ int before[kRankWaves][kRankEntries];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int base = blockIdx.x * kRankEntries, own_run = base / kWave, runs = (n + kWave - 1) / kWave;
    auto digit = [&](int i) { return static_cast<D>((keys_in[i] >> shift) & mask); };
    D mine[kRankEntries];
    int count[kRankEntries];
#pragma unroll
    for (int e = 0; e < kRankEntries; ++e) {
        mine[e] = uniform(digit(min(base + e, n - 1)));
        count[e] = 0;
    }
    // keys of an earlier run come before an equal entry, of a later run after it
    auto add = [&](int run, D other) {
        if (run < own_run) {
#pragma unroll
            for (int e = 0; e < kRankEntries; ++e) count[e] += __popcll(__ballot(other <= mine[e]));
        } else if (run > own_run) {
#pragma unroll
            for (int e = 0; e < kRankEntries; ++e) count[e] += __popcll(__ballot(other < mine[e]));
        } else {
#pragma unroll
            for (int e = 0; e < kRankEntries; ++e)
                count[e] += __popcll(
                    __ballot((other < mine[e]) | ((other == mine[e]) & (run * kWave + lane < base + e))));
        }
    };
    constexpr int kAtOnce = 8;
    for (int run = wave; run < runs; run += kAtOnce * kRankWaves) {
        D other[kAtOnce];
#pragma unroll
        for (int r = 0; r < kAtOnce; ++r) {
            const int i = (run + r * kRankWaves) * kWave + lane;
            other[r] = i < n ? digit(i) : static_cast<D>(~D(0));  // past the end: before none
        }
#pragma unroll
        for (int r = 0; r < kAtOnce; ++r)
            if (run + r * kRankWaves < runs) add(run + r * kRankWaves, other[r]);
    }
    int c = 0;
#pragma unroll
    for (int e = 0; e < kRankEntries; ++e) c = lane == e ? count[e] : c;
    if (lane < kRankEntries) before[wave][lane] = c;
    __syncthreads();
    const int i = base + static_cast<int>(threadIdx.x);
    if (threadIdx.x < kRankEntries && i < n) {
        int rank = 0;
#pragma unroll
        for (int w = 0; w < kRankWaves; ++w) rank += before[w][threadIdx.x];
        keys_out[rank] = keys_in[i];
        if constexpr (HasValues) values_out[rank] = values_in[i];
    }
}

template <typename S, typename V, bool HasValues>
bool radix_passes(gpart_ctx* ctx, std::uint64_t* keys, std::uint64_t* keys_alt, V* values, V* values_alt,
                  std::int64_t n, int begin_bit, int end_bit) {
    const std::int64_t tiles = (n + S::kKeys - 1) / S::kKeys;
    Scratch<std::uint32_t> hist(ctx, tiles * kDigits);
    std::uint64_t* src_k = keys;
    std::uint64_t* dst_k = keys_alt;
    V* src_v = values;
    V* dst_v = values_alt;
    bool in_alt = false;
    for (int shift = begin_bit; shift < end_bit; shift += 8) {
        const int bits = end_bit - shift < 8 ? end_bit - shift : 8;
        const std::uint64_t mask = (1ULL << bits) - 1;
        hipLaunchKernelGGL(radix_histogram_kernel<S>, dim3(static_cast<unsigned>(tiles)), dim3(S::kThreads), 0,
                           ctx->stream, src_k, n, shift, mask, hist.get(), tiles);
        GPART_LAUNCH_CHECK();
        const bool raw = tiles <= kInlineHistogramTiles;
        if (!raw)
            device_scan<std::uint32_t, SumOp<std::uint32_t>>(ctx, ArrayLoad<std::uint32_t>{hist.get()},
                                                             ExclusiveStore<std::uint32_t>{hist.get()},
                                                             tiles * kDigits, SumOp<std::uint32_t>{});
        hipLaunchKernelGGL((radix_scatter_kernel<S, V, HasValues>), dim3(static_cast<unsigned>(tiles)), dim3(S::kThreads),
                           0, ctx->stream, src_k, dst_k, src_v, dst_v, n, shift, mask, hist.get(), tiles, raw ? 1 : 0);
        GPART_LAUNCH_CHECK();
        std::swap(src_k, dst_k);
        std::swap(src_v, dst_v);
        in_alt = !in_alt;
    }
    return in_alt;
}

template <typename V, bool HasValues>
bool radix_sort_impl(gpart_ctx* ctx, std::uint64_t* keys, std::uint64_t* keys_alt, V* values, V* values_alt,
                     std::int64_t n, int begin_bit, int end_bit) {
    if (n <= 1 || end_bit <= begin_bit) return false;
    if (n > (std::int64_t{1} << 32) - SmallTile::kKeys)
        throw Error(GPART_ERR_INVALID_ARGUMENT, "radix sort supports fewer than 2^32 keys per call");
    if (n <= kRankSortMax) {
        const int width = end_bit - begin_bit;
        const std::uint64_t mask = width >= 64 ? ~0ULL : ((1ULL << width) - 1);
        const dim3 grid(static_cast<unsigned>((n + kRankEntries - 1) / kRankEntries)), block(kRankWaves * kWave);
        if (width <= 32)
            hipLaunchKernelGGL((rank_sort_kernel<V, HasValues, unsigned>), grid, block, 0, ctx->stream, keys, keys_alt,
                               values, values_alt, static_cast<int>(n), begin_bit, mask);
        else
            hipLaunchKernelGGL((rank_sort_kernel<V, HasValues, std::uint64_t>), grid, block, 0, ctx->stream, keys,
                               keys_alt, values, values_alt, static_cast<int>(n), begin_bit, mask);
        GPART_LAUNCH_CHECK();
        return true;
    }
    if (n < kLargeSort)
        return radix_passes<SmallTile, V, HasValues>(ctx, keys, keys_alt, values, values_alt, n, begin_bit, end_bit);
    return radix_passes<LargeTile, V, HasValues>(ctx, keys, keys_alt, values, values_alt, n, begin_bit, end_bit);
}

struct FlagLoad {
    const std::int32_t* flags;
    __device__ __forceinline__ std::int64_t operator()(std::int64_t i) const { return flags[i] != 0 ? 1 : 0; }
};

struct CompactStore {
    std::int32_t* out;
    std::int64_t n;
    std::int64_t* count;
    __device__ __forceinline__ void operator()(std::int64_t i, std::int64_t prefix, std::int64_t item) const {
        if (item) out[prefix] = static_cast<std::int32_t>(i);
        if (i == n - 1) *count = prefix + item;
    }
};

}  // namespace

template <typename V>
bool radix_sort_pairs(gpart_ctx* ctx, std::uint64_t* keys, std::uint64_t* keys_alt, V* values, V* values_alt,
                      std::int64_t n, int begin_bit, int end_bit) {
    return radix_sort_impl<V, true>(ctx, keys, keys_alt, values, values_alt, n, begin_bit, end_bit);
}
template bool radix_sort_pairs<std::uint32_t>(gpart_ctx*, std::uint64_t*, std::uint64_t*, std::uint32_t*,
                                              std::uint32_t*, std::int64_t, int, int);
template bool radix_sort_pairs<std::uint64_t>(gpart_ctx*, std::uint64_t*, std::uint64_t*, std::uint64_t*,
                                              std::uint64_t*, std::int64_t, int, int);

bool radix_sort_keys(gpart_ctx* ctx, std::uint64_t* keys, std::uint64_t* keys_alt, std::int64_t n, int begin_bit,
                     int end_bit) {
    return radix_sort_impl<std::uint32_t, false>(ctx, keys, keys_alt, nullptr, nullptr, n, begin_bit, end_bit);
}

template <typename T>
void exclusive_scan(gpart_ctx* ctx, const T* in, T* out, std::int64_t n, T* total_device) {
    device_scan<T, SumOp<T>>(ctx, ArrayLoad<T>{in}, ExclusiveStore<T>{out}, n, SumOp<T>{});
    (void)total_device;
}
template <typename T>
void inclusive_scan(gpart_ctx* ctx, const T* in, T* out, std::int64_t n) {
    device_scan<T, SumOp<T>>(ctx, ArrayLoad<T>{in}, InclusiveStore<T>{out}, n, SumOp<T>{});
}
template void exclusive_scan<std::uint64_t>(gpart_ctx*, const std::uint64_t*, std::uint64_t*, std::int64_t,
                                            std::uint64_t*);
template void exclusive_scan<std::int64_t>(gpart_ctx*, const std::int64_t*, std::int64_t*, std::int64_t,
                                           std::int64_t*);
template void exclusive_scan<std::uint32_t>(gpart_ctx*, const std::uint32_t*, std::uint32_t*, std::int64_t,
                                            std::uint32_t*);
template void inclusive_scan<std::uint64_t>(gpart_ctx*, const std::uint64_t*, std::uint64_t*, std::int64_t);

void compact_indices(gpart_ctx* ctx, const std::int32_t* flags, std::int64_t n, std::int32_t* out,
                     std::int64_t* d_count) {
    if (n <= 0) {
        fill_bytes(ctx, d_count, 0, sizeof(std::int64_t));
        return;
    }
    device_scan<std::int64_t, SumOp<std::int64_t>>(ctx, FlagLoad{flags}, CompactStore{out, n, d_count}, n,
                                                   SumOp<std::int64_t>{});
}

}  // namespace gpart_hip

using namespace gpart_hip;

extern "C" {

int gpart_sort_pairs_u64(gpart_ctx* ctx, uint64_t* keys, void* values, int value_bytes, int64_t n,
                         int begin_bit, int end_bit) {
    return guarded([&] {
        if (begin_bit < 0 || end_bit > 64 || begin_bit > end_bit)
            throw Error(GPART_ERR_INVALID_ARGUMENT, "invalid radix sort bit range");
        if (n <= 1) return;
        Scratch<std::uint64_t> keys_alt(ctx, n);
        bool alt = false;
        if (!values) {
            alt = radix_sort_keys(ctx, keys, keys_alt.get(), n, begin_bit, end_bit);
            if (alt) copy_device(ctx, keys, keys_alt.get(), n * 8);
        } else if (value_bytes == 4) {
            Scratch<std::uint32_t> values_alt(ctx, n);
            alt = radix_sort_pairs(ctx, keys, keys_alt.get(), static_cast<std::uint32_t*>(values), values_alt.get(), n,
                                   begin_bit, end_bit);
            if (alt) {
                copy_device(ctx, keys, keys_alt.get(), n * 8);
                copy_device(ctx, values, values_alt.get(), n * 4);
            }
        } else if (value_bytes == 8) {
            Scratch<std::uint64_t> values_alt(ctx, n);
            alt = radix_sort_pairs(ctx, keys, keys_alt.get(), static_cast<std::uint64_t*>(values), values_alt.get(), n,
                                   begin_bit, end_bit);
            if (alt) {
                copy_device(ctx, keys, keys_alt.get(), n * 8);
                copy_device(ctx, values, values_alt.get(), n * 8);
            }
        } else {
            throw Error(GPART_ERR_INVALID_ARGUMENT, "value_bytes must be 4 or 8");
        }
    });
}

int gpart_exclusive_scan_u64(gpart_ctx* ctx, const uint64_t* in, uint64_t* out, int64_t n) {
    return guarded([&] { exclusive_scan<std::uint64_t>(ctx, in, out, n); });
}

int gpart_compact_flags(gpart_ctx* ctx, const int32_t* flags, int64_t n, int32_t* out, int64_t* count) {
    return guarded([&] {
        Scratch<std::int64_t> d_count(ctx, 1);
        compact_indices(ctx, flags, n, out, d_count.get());
        *count = read_scalar(ctx, d_count.get());
    });
}

}  // extern "C"
