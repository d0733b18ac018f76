// refine.hip -- incremental bucketed refinement for gfx950
// (src/refine.cu and src/refine_incremental.cuh of the reference).
//
// Per-vertex edge loops use the level's degree classes: 8 lanes for degree <= 8,
// a wave for <= 256 and a workgroup above. Row scans of the n x k connectivity
// cache use 1, 2 or 4 lanes per row, each owning 8 consecutive parts, so a wave
// has 16-64 rows in flight per pass.
//
// The reference ranks vertices inside a rebalance bucket by the return value of
// atomicAdd (src/refine_incremental.cuh:185,216): any order is legal. Here the
// rank is the weight of the bucket's lower-id members, so refinement is
// reproducible run to run.
//
// A round (LP or rebalance) keeps its counts on the device: kernels after a
// compaction read the length from a RoundState and loop grid-stride, and the
// host reads one RoundState back at the end of the round.
#include "internal.hpp"
#include "reduce.hpp"
#include "scan.hpp"
#include "tiles.hpp"
#include "hubs.hpp"
#include "refine_device.hpp"
#include "refine_rows.hpp"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <list>
#include <unordered_set>

namespace gpart_hip {
namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(std::int64_t threads) { return static_cast<unsigned>((threads + kBlock - 1) / kBlock); }

// ---------------------------------------------------------------- round state

// Device record of one round, read back once at its end.
struct RoundState {
    long long light;       // movers with degree <= kHeavyDegree
    long long heavy;       // movers above
    long long delta;       // exact cut decrease
    long long candidates;  // rebalance: vertices of overloaded parts
    unsigned long long max_weight;
    long long edges;       // CSR entries of all movers (light + heavy)
    unsigned long long cut_directed;  // rebuild rounds: directed cut weight after the round
    unsigned long long arrivals;  // workgroups of the round's last launch that have finished
    unsigned long long refused;   // rebalance: more vertices leave than one workgroup selects among
    unsigned long long pw[32];
};

constexpr int kHeavyDegree = 64;
// Levels whose largest degree is at most this update their heavy movers' cache rows
// a wave per mover (one launch); above it the movers' entries are flattened into
// tiles first (a scan and a tile map, three more launches) so that hubs spread
// over many workgroups.
constexpr int kWaveHeavyMaxDegree = 4096;
constexpr int kRoundBlocks = 1024;  // cap of grid-stride launches whose count lives on the device
constexpr int kCacheBlocks = 4096;  // cap of the cache build launches (grid-stride)


// ---------------------------------------------------------------- cut / weights

constexpr int kCutBlocks = 1024;  // of a cut's pass over the edge tiles at most, a partial each

// Directed cut weight over edge tiles (grid-stride over tiles); one partial per
// workgroup in directed[blockIdx.x]. A lane loads its run's neighbours and
// weights up front, then gathers their labels, so 16 loads are in flight per lane.
template <typename O, typename W>
__global__ void __launch_bounds__(kTileLanes) cut_kernel(std::int64_t n, std::int64_t m, std::int64_t tiles,
                                                         const O* offsets, const std::int32_t* tile_row,
                                                         const std::int32_t* neighbors, const W* weights,
                                                         const std::int32_t* labels, unsigned long long* directed) {
    __shared__ unsigned long long waves[kTileLanes / kWave];
    unsigned long long local = 0;
    for (std::int64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        std::int64_t e, stop;
        std::int32_t r;
        if (!tile_run(offsets, tile_row, tiles, n, m, t, &e, &stop, &r)) continue;
        std::int32_t other[kTileRun];
        W w[kTileRun];
#pragma unroll
        for (int j = 0; j < kTileRun; ++j) {
            const bool in = e + j < stop;
            other[j] = in ? neighbors[e + j] : 0;
            w[j] = in ? weights[e + j] : W{0};
        }
#pragma unroll
        for (int j = 0; j < kTileRun; ++j) other[j] = labels[other[j]];
        std::int64_t next = static_cast<std::int64_t>(offsets[r + 1]);
        std::int32_t p = labels[r];
#pragma unroll
        for (int j = 0; j < kTileRun; ++j) {
            if (e + j < stop) {
                if (e + j >= next) {
                    do next = static_cast<std::int64_t>(offsets[++r + 1]);
                    while (e + j >= next);
                    p = labels[r];
                }
                if (other[j] != p) local += static_cast<unsigned long long>(w[j]);
            }
        }
    }
    local = group_sum_u64<kWave>(local);
    if (lane_id() == 0) waves[threadIdx.x / kWave] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long total = 0;
        for (int w = 0; w < kTileLanes / kWave; ++w) total += waves[w];
        directed[blockIdx.x] = total;
    }
}

template <typename W>
__global__ void part_weights_kernel(std::int64_t n, const std::int32_t* labels, const W* vertex_weights, int k,
                                    unsigned long long* out) {
    __shared__ unsigned long long local[32];
    if (threadIdx.x < 32) local[threadIdx.x] = 0;
    __syncthreads();
    for (std::int64_t v = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < n;
         v += static_cast<std::int64_t>(gridDim.x) * blockDim.x)
        atomicAdd(&local[labels[v]], static_cast<unsigned long long>(vertex_weights[v]));
    __syncthreads();
    if (threadIdx.x < k && local[threadIdx.x]) atomicAdd(out + threadIdx.x, local[threadIdx.x]);
}

__global__ void project_kernel(std::int64_t n, const std::int32_t* map, const std::int32_t* coarse,
                               std::int32_t* fine) {
    const std::int64_t v = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (v < n) fine[v] = coarse[map[v]];
}

// ---------------------------------------------------------------- cache

// Adds the workgroup's sum of v to *out with one atomic. Called by every thread
// of a kBlock-thread workgroup; waves holds kBlock / kWave entries.
__device__ __forceinline__ void block_add_u64(unsigned long long v, unsigned long long* waves,
                                              unsigned long long* out) {
    v = group_sum_u64<kWave>(v);
    if (lane_id() == 0) waves[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long total = 0;
        for (int w = 0; w < kBlock / kWave; ++w) total += waves[w];
        if (total) atomicAdd(out, total);
    }
}

template <typename O, typename W, int G, typename C>
__global__ void __launch_bounds__(kBlock) build_cache_kernel(std::int64_t count, const std::int32_t* list,
                                                             const O* offsets, const std::int32_t* neighbors,
                                                             const W* weights, const std::int32_t* labels, int k,
                                                             C* cache, const long long* gate, long long above,
                                                             unsigned long long* cut) {
    // gate: a rebuild inside a round runs only when the round's mover entries exceed
    // `above`; grid-stride over groups so that a gated-off launch is a small grid.
    // cut (optional) receives the directed cut weight of `labels`.
    if (gate && *gate <= above) return;
    constexpr int kGroups = kBlock / G;
    __shared__ unsigned long long rows[kGroups][32];
    __shared__ unsigned long long wave_cut[kBlock / kWave];
    const int local_group = threadIdx.x / G;
    const int sub = threadIdx.x & (G - 1);
    unsigned long long cut_local = 0;
    for (std::int64_t first = static_cast<std::int64_t>(blockIdx.x) * kGroups; first < count;
         first += static_cast<std::int64_t>(gridDim.x) * kGroups) {
        const std::int64_t group = first + local_group;
        for (int p = sub; p < 32; p += G) rows[local_group][p] = 0;
        __syncthreads();
        std::int32_t v = 0;
        bool own = group < count;
        if (own) {
            v = list ? list[group] : static_cast<std::int32_t>(group);
            // rows above kHubChunk entries are hubs, built by build_cache_hub_kernel
            own = G < kBlock || offsets[v + 1] - offsets[v] <= kHubChunk;
            if (own) {
                const std::int32_t lv = labels[v];
                for (std::int64_t e = static_cast<std::int64_t>(offsets[v]) + sub; e < offsets[v + 1]; e += G) {
                    const std::int32_t u = neighbors[e];
                    if (u == v) continue;
                    const std::int32_t lu = labels[u];
                    const auto w = static_cast<unsigned long long>(weights[e]);
                    atomicAdd(&rows[local_group][lu], w);
                    if (lu != lv) cut_local += w;
                }
            }
        }
        __syncthreads();
        if (own)
            for (int p = sub; p < k; p += G)
                cache[static_cast<std::int64_t>(v) * k + p] = static_cast<C>(rows[local_group][p]);
        __syncthreads();
    }
    if (cut) block_add_u64(cut_local, wave_cut, cut);
}

template <typename C>
__global__ void hub_rows_zero_kernel(std::int64_t count, const std::int64_t* chunk_start, const std::int32_t* list,
                                     int k, C* cache, const long long* gate, long long above) {
    if (gate && *gate <= above) return;
    const std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= count || chunk_start[i] == chunk_start[i + 1]) return;
    C* row = cache + static_cast<std::int64_t>(list[i]) * k;
    for (int p = 0; p < k; ++p) row[p] = 0;
}

// Hub rows (degree > kHubChunk), one chunk per workgroup pass: the chunk's part
// sums gather in LDS and reach the zeroed cache row as k atomic adds.
template <typename O, typename W, typename C>
__global__ void __launch_bounds__(kBlock) build_cache_hub_kernel(const std::int64_t* chunk_total,
                                                                 const std::int64_t* chunk_start,
                                                                 const std::int32_t* chunk_hub,
                                                                 const std::int32_t* list, const O* offsets,
                                                                 const std::int32_t* neighbors, const W* weights,
                                                                 const std::int32_t* labels, int k, C* cache,
                                                                 const long long* gate, long long above,
                                                                 unsigned long long* cut) {
    __shared__ unsigned long long row[32];
    __shared__ unsigned long long wave_cut[kBlock / kWave];
    if (gate && *gate <= above) return;
    unsigned long long cut_local = 0;
    const std::int64_t chunks = *chunk_total;
    for (std::int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        if (threadIdx.x < 32) row[threadIdx.x] = 0;
        __syncthreads();
        std::int32_t i, v;
        std::int64_t begin, end;
        hub_chunk_range(offsets, list, chunk_start, chunk_hub, c, &i, &v, &begin, &end);
        const std::int32_t lv = labels[v];
        for (std::int64_t e = begin + threadIdx.x; e < end; e += kBlock) {
            const std::int32_t u = neighbors[e];
            if (u == v) continue;
            const std::int32_t lu = labels[u];
            const auto w = static_cast<unsigned long long>(weights[e]);
            atomicAdd(&row[lu], w);
            if (lu != lv) cut_local += w;
        }
        __syncthreads();
        if (threadIdx.x < k && row[threadIdx.x])
            atomicAdd(cache + static_cast<std::int64_t>(v) * k + threadIdx.x, static_cast<C>(row[threadIdx.x]));
        __syncthreads();
    }
    if (cut) block_add_u64(cut_local, wave_cut, cut);
}

// incremental_lp_proposals (:27-46): argmax over p != source of cache > 0,
// lowest index on ties; accepted if best >= current or within the filter.
template <int G, typename C>
__global__ void __launch_bounds__(kBlock) lp_proposals_kernel(std::int64_t n, const C* cache,
                                                              const std::int32_t* labels, int k, double filter,
                                                              std::int32_t* locks, std::int32_t* targets,
                                                              long long* gains, unsigned char* state,
                                                              RoundState* st) {
    // the round's state starts at zero (the filter appends the movers to it)
    if (blockIdx.x == 0 && threadIdx.x < sizeof(RoundState) / 8)
        reinterpret_cast<unsigned long long*>(st)[threadIdx.x] = 0;
    const std::int64_t v = (static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / G;
    const int j = threadIdx.x & (G - 1);
    if (v >= n) return;  // uniform per group
    const std::int32_t source = labels[v];
    const C* row = cache + v * k;
    unsigned long long best = 0, current = 0;
    int best_p = 0x7fffffff;
    unsigned long long span[kRowSpan];
    load_span(row, j, k, span);
#pragma unroll
    for (int e = 0; e < kRowSpan; ++e) {
        const int p = j * kRowSpan + e;
        const unsigned long long value = span[e];
        if (p == source) current = value;
        else if (value > best) {  // strict: the lowest index keeps a tie
            best = value;
            best_p = p;
        }
    }
#pragma unroll
    for (int m = G / 2; m > 0; m /= 2) {
        const auto ob = shfl_xor_u64(best, m, G);
        const int op = static_cast<int>(lane_xor(static_cast<unsigned>(best_p), m, G));
        const auto oc = shfl_xor_u64(current, m, G);
        if (ob > best || (ob == best && op < best_p)) {
            best = ob;
            best_p = op;
        }
        current = oc > current ? oc : current;  // only the source's lane holds it
    }
    if (j != 0) return;
    if (state) state[v] = static_cast<unsigned char>(source);  // refine_rows.hpp
    if (locks[v] != 0) {
        locks[v] = 0;
        targets[v] = -1;
        gains[v] = static_cast<long long>(0x8000000000000000ULL);
        return;
    }
    std::int32_t target = -1;
    long long gain = static_cast<long long>(0x8000000000000000ULL);
    if (best > 0 &&
        (best >= current ||
         current - best < static_cast<unsigned long long>(filter * static_cast<double>(current)))) {
        target = best_p;
        gain = best >= current ? static_cast<long long>(best - current) : -static_cast<long long>(current - best);
    }
    targets[v] = target;
    gains[v] = gain;
}

// Appends the taking threads' vertices to the light/heavy mover lists (one
// global atomic per list per workgroup pass). Called by every thread of the
// workgroup.
template <int Threads, typename O>
__device__ void append_movers(bool take, std::int32_t v, const O* offsets, std::int32_t* light,
                              std::int32_t* heavy, RoundState* st, unsigned* counts, unsigned long long* base) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const long long degree = take ? static_cast<long long>(offsets[v + 1] - offsets[v]) : 0;
    const bool is_heavy = degree > kHeavyDegree;
    const long long edges = group_sum_i64<kWave>(degree);
    if (lane == 0 && edges) atomicAdd(reinterpret_cast<unsigned long long*>(&st->edges),
                                      static_cast<unsigned long long>(edges));
    const bool is_light = take && !is_heavy;
    const unsigned long long bl = __ballot(is_light), bh = __ballot(is_heavy);
    if (lane == 0) {
        counts[wave] = static_cast<unsigned>(__popcll(bl));
        counts[Threads / kWave + wave] = static_cast<unsigned>(__popcll(bh));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned tl = 0, th = 0;
        for (int q = 0; q < Threads / kWave; ++q) {
            tl += counts[q];
            th += counts[Threads / kWave + q];
        }
        base[0] = tl ? atomicAdd(reinterpret_cast<unsigned long long*>(&st->light), tl) : 0;
        base[1] = th ? atomicAdd(reinterpret_cast<unsigned long long*>(&st->heavy), th) : 0;
    }
    __syncthreads();
    if (take) {
        unsigned before = 0;
        const unsigned* row = is_heavy ? counts + Threads / kWave : counts;
        for (int q = 0; q < wave; ++q) before += row[q];
        const unsigned long long mask = is_heavy ? bh : bl;
        before += static_cast<unsigned>(__popcll(mask & lanemask_lt()));
        (is_heavy ? heavy : light)[(is_heavy ? base[1] : base[0]) + before] = v;
    }
    __syncthreads();
}

// incremental_priority_filter (:48-67) over one class list with G lanes per row,
// by the workgroups numbered `block` of the list's range. Called by every thread
// of the workgroup; true on the one lane of a row whose vertex (*vertex) moves.
template <typename O, typename W, int G>
__device__ __forceinline__ bool priority_filter_rows(std::int64_t count, const std::int32_t* list, long long block,
                                                     const O* offsets, const std::int32_t* neighbors,
                                                     const W* weights, const std::int32_t* labels,
                                                     const std::int32_t* targets, const long long* gains,
                                                     std::int32_t* flags, unsigned char* state,
                                                     long long* block_sum, std::int32_t* vertex) {
    const std::int64_t group = (block * blockDim.x + threadIdx.x) / G;
    const int sub = threadIdx.x & (G - 1);
    const bool active = group < count;
    const std::int32_t v = active ? (list ? list[group] : static_cast<std::int32_t>(group)) : 0;
    const std::int32_t target = active ? targets[v] : -1;
    // rows above kHubChunk entries are hubs, done in chunks by priority_filter_hub_kernel
    bool take = false;
    if (G == kBlock && active && offsets[v + 1] - offsets[v] > kHubChunk) return false;  // uniform per block
    long long correction = 0;
    if (active && target >= 0)
        correction = filter_correction(v, target, labels[v], gains[v], static_cast<std::int64_t>(offsets[v]) + sub,
                                       static_cast<std::int64_t>(offsets[v + 1]), G, neighbors, weights, labels,
                                       targets, gains);
    if constexpr (G <= kWave) {
        correction = group_sum_i64<G>(correction);
        if (active && sub == 0) {
            take = target >= 0 && gains[v] + correction >= 0;
            flags[v] = take ? labels[v] + 1 : 0;
            if (take) mark_mover(state, v, target);
        }
    } else {
        correction = group_sum_i64<kWave>(correction);
        if (lane_id() == 0) block_sum[threadIdx.x / kWave] = correction;
        __syncthreads();
        if (threadIdx.x == 0 && active) {
            long long total = 0;
            for (int w = 0; w < kBlock / kWave; ++w) total += block_sum[w];
            take = target >= 0 && gains[v] + total >= 0;
            flags[v] = take ? labels[v] + 1 : 0;
            if (take) mark_mover(state, v, target);
        }
    }
    *vertex = v;
    return take;
}

// The three degree classes in one launch: workgroups [0, low_blocks) take the low
// rows (8 lanes each), the next medium_blocks the medium rows (a wave each), the
// rest the high rows (a workgroup each). Append: the workgroups also append their
// movers to the round's lists (three counter atomics per workgroup that has any,
// so only for small levels; the lists' order does not matter).
template <typename O, typename W, bool Append>
__global__ void __launch_bounds__(kBlock) priority_filter_kernel(
    std::int64_t low_count, const std::int32_t* low, unsigned low_blocks, std::int64_t medium_count,
    const std::int32_t* medium, unsigned medium_blocks, std::int64_t high_count, const std::int32_t* high,
    const O* offsets, const std::int32_t* neighbors, const W* weights, const std::int32_t* labels,
    const std::int32_t* targets, const long long* gains, std::int32_t* flags, unsigned char* state,
    std::int32_t* light, std::int32_t* heavy, RoundState* st) {
    __shared__ long long block_sum[kBlock / kWave];
    const long long b = blockIdx.x;
    bool take;
    std::int32_t v = 0;
    if (b < low_blocks)
        take = priority_filter_rows<O, W, 8>(low_count, low, b, offsets, neighbors, weights, labels, targets, gains,
                                             flags, state, block_sum, &v);
    else if (b < low_blocks + medium_blocks)
        take = priority_filter_rows<O, W, 64>(medium_count, medium, b - low_blocks, offsets, neighbors, weights,
                                              labels, targets, gains, flags, state, block_sum, &v);
    else
        take = priority_filter_rows<O, W, kBlock>(high_count, high, b - low_blocks - medium_blocks, offsets,
                                                  neighbors, weights, labels, targets, gains, flags, state, block_sum,
                                                  &v);
    if constexpr (Append) {
        __shared__ unsigned counts[2 * (kBlock / kWave)];
        __shared__ unsigned long long base[2];
        if (__syncthreads_or(take)) append_movers<kBlock>(take, v, offsets, light, heavy, st, counts, base);
    }
}

// Hub rows (degree > kHubChunk): each chunk adds its share of the correction to
// sums[i]; priority_filter_hub_finish_kernel then sets the hub's flag.
template <typename O, typename W>
__global__ void __launch_bounds__(kBlock) priority_filter_hub_kernel(const std::int64_t* chunk_total,
                                                                     const std::int64_t* chunk_start,
                                                                     const std::int32_t* chunk_hub,
                                                                     const std::int32_t* list, const O* offsets,
                                                                     const std::int32_t* neighbors, const W* weights,
                                                                     const std::int32_t* labels,
                                                                     const std::int32_t* targets,
                                                                     const long long* gains, long long* sums) {
    __shared__ long long block_sum[kBlock / kWave];
    const std::int64_t chunks = *chunk_total;
    for (std::int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        std::int32_t i, v;
        std::int64_t begin, end;
        hub_chunk_range(offsets, list, chunk_start, chunk_hub, c, &i, &v, &begin, &end);
        const std::int32_t target = targets[v];
        long long correction = 0;
        if (target >= 0)
            correction = filter_correction(v, target, labels[v], gains[v], begin + threadIdx.x, end, kBlock,
                                           neighbors, weights, labels, targets, gains);
        correction = group_sum_i64<kWave>(correction);
        if (lane_id() == 0) block_sum[threadIdx.x / kWave] = correction;
        __syncthreads();
        if (threadIdx.x == 0) {
            long long total = 0;
            for (int w = 0; w < kBlock / kWave; ++w) total += block_sum[w];
            if (total) atomicAdd(reinterpret_cast<unsigned long long*>(sums + i), static_cast<unsigned long long>(total));
        }
        __syncthreads();
    }
}

__global__ void priority_filter_hub_finish_kernel(std::int64_t count, const std::int64_t* chunk_start,
                                                  const std::int32_t* list, const std::int32_t* labels,
                                                  const std::int32_t* targets, const long long* gains,
                                                  long long* sums, std::int32_t* flags, unsigned char* state) {
    const std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= count || chunk_start[i] == chunk_start[i + 1]) return;
    const std::int32_t v = list[i];
    const bool take = targets[v] >= 0 && gains[v] + sums[i] >= 0;
    flags[v] = take ? labels[v] + 1 : 0;
    if (take) mark_mover(state, v, targets[v]);
    sums[i] = 0;
}

// The round's status into the host-visible words (word 0: seq, stored last, after
// a system-scope fence). Called by one wave; weight(p) and delta are the part
// weights and the cut decrease as the round left them. Lane p < k holds part p's
// weight; every lane writes one status word.
template <typename Weight>
__device__ void publish_status(const RoundState* st, Weight weight, long long delta, int k,
                               unsigned long long* status, unsigned long long* counter) {
    constexpr int kHead = static_cast<int>(offsetof(RoundState, pw) / 8);  // words before pw
    constexpr int kDelta = static_cast<int>(offsetof(RoundState, delta) / 8);
    constexpr int kMax = static_cast<int>(offsetof(RoundState, max_weight) / 8);
    const int lane = lane_id();
    const unsigned long long w = lane < k ? weight(lane) : 0;
    unsigned long long maximum = w;
    for (int m = kWave / 2; m > 0; m /= 2) {
        const unsigned long long o = shfl_xor_u64(maximum, m, kWave);
        maximum = o > maximum ? o : maximum;
    }
    if (lane < kHead) {
        const auto* words = reinterpret_cast<const unsigned long long*>(st);
        status[1 + lane] = lane == kMax ? maximum : lane == kDelta ? static_cast<unsigned long long>(delta) : words[lane];
    }
    if (lane < k) status[1 + kHead + lane] = w;
    __threadfence_system();
    if (lane == 0) {
        const unsigned long long seq = *counter + 1;
        *counter = seq;
        __hip_atomic_store(status, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
static_assert(sizeof(RoundState) % 8 == 0 && sizeof(RoundState) / 8 + 1 <= kStatusWords, "status words");

__global__ void __launch_bounds__(kWave) round_status_kernel(const RoundState* st,
                                                             const unsigned long long* part_weights, int k,
                                                             unsigned long long* status,
                                                             unsigned long long* counter) {
    publish_status(st, [&](int p) { return part_weights[p]; }, st->delta, k, status, counter);
}

// The part weight moves of a workgroup's committed movers, in LDS.
struct PartMoves {
    unsigned long long gained[32], lost[32];
    __device__ __forceinline__ void clear() {
        if (threadIdx.x < 32) gained[threadIdx.x] = lost[threadIdx.x] = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void flush(int k, unsigned long long* part_weights) const {
        if (threadIdx.x < static_cast<unsigned>(k)) {
            const unsigned long long change = gained[threadIdx.x] - lost[threadIdx.x];
            if (change) atomicAdd(part_weights + threadIdx.x, change);
        }
    }
};

// incremental_commit (:97-109) of one mover: its label, its lock after an LP round,
// its weight. Its old part is in flags, so nobody reads a mover's label any more.
template <typename W>
__device__ __forceinline__ void commit_mover(std::int32_t v, std::int32_t source, std::int32_t target,
                                             const W* vertex_weights, std::int32_t* labels, std::int32_t* locks,
                                             PartMoves& moves) {
    const auto w = static_cast<unsigned long long>(vertex_weights[v]);
    atomicAdd(&moves.lost[source], w);
    atomicAdd(&moves.gained[target], w);
    labels[v] = target;
    if (locks) locks[v] = 1;
}

// incremental_update_cache_and_cut (:69-95) and incremental_commit (:97-109) over a
// mover list whose length is on the device, G lanes per mover, by the workgroups
// [0, blocks) numbered `block`; returns the lane's gain. update: false in rebuild
// rounds, which only commit. flags holds a mover's old part + 1, so labels may
// change meanwhile: a neighbour's label is read only when it does not move.
template <typename O, typename W, int G, typename C>
__device__ __forceinline__ long long update_cache_movers(long long count, const std::int32_t* movers,
                                                         const O* offsets, const std::int32_t* neighbors,
                                                         const W* weights, const W* vertex_weights,
                                                         std::int32_t* labels, const std::int32_t* targets,
                                                         const std::int32_t* flags, std::int32_t* locks, int k,
                                                         C* cache, bool update, long long block, long long blocks,
                                                         PartMoves& moves) {
    const int sub = threadIdx.x & (G - 1);
    const long long groups = blocks * (kBlock / G);
    long long gain = 0;
    for (long long group = (block * blockDim.x + threadIdx.x) / G; group < count; group += groups) {
        const std::int32_t v = movers[group];
        const std::int32_t source = flags[v] - 1;
        const std::int32_t target = targets[v];
        if (sub == 0) commit_mover(v, source, target, vertex_weights, labels, locks, moves);
        if (!update) continue;
        for (std::int64_t e = static_cast<std::int64_t>(offsets[v]) + sub; e < offsets[v + 1]; e += G) {
            const std::int32_t u = neighbors[e];
            if (u == v) continue;
            const auto w = static_cast<unsigned long long>(weights[e]);
            // modular arithmetic: entries fit C at every point of the round
            atomicAdd(cache + static_cast<std::int64_t>(u) * k + source, static_cast<C>(0ULL - w));
            atomicAdd(cache + static_cast<std::int64_t>(u) * k + target, static_cast<C>(w));
            const std::int32_t fu = flags[u];
            if (!fu || u > v) {
                const std::int32_t lu = fu ? fu - 1 : labels[u];
                const std::int32_t nu = fu ? targets[u] : lu;
                gain += static_cast<long long>(w) * ((source != lu) - (target != nu));
            }
        }
    }
    return gain;
}

// Adds the workgroup's sum of v to *out with one atomic. Called by every thread
// of a kBlock-thread workgroup; block_sum holds kBlock / kWave entries.
__device__ __forceinline__ void block_add_i64(long long v, long long* block_sum, long long* out) {
    v = group_sum_i64<kWave>(v);
    if (lane_id() == 0) block_sum[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long total = 0;
        for (int w = 0; w < kBlock / kWave; ++w) total += block_sum[w];
        if (total) atomicAdd(reinterpret_cast<unsigned long long*>(out), static_cast<unsigned long long>(total));
    }
}

// Cache updates and commits of a round. Workgroups [0, light_blocks) take the light
// movers (8 lanes each); the rest of the grid the heavy movers (a wave each). With
// no such rest (wave_heavy_blocks == 0) the light workgroups commit the heavy movers,
// whose entries update_cache_tiles_kernel walks next.
//
// status (optional): the last workgroup to finish publishes the round's status, so
// that the round ends with this launch (commit and status as launches of their own
// cost 3.8 and 3.6 us per round on the 128^3 mesh). Only workgroups with movers of
// their own take part (the others return at once), so the arrival counter sees as
// many atomics as there is work. What the last workgroup reads of the others --
// part weights and the cut decrease -- was written by device-scope atomics, which
// have left the workgroup when it arrives (s_waitcnt before its barrier) and are
// performed past the XCDs' caches; it reads them with device-scope atomic loads. No
// cache write-back is needed: the labels are read by later launches, or after the entry
// point's wait for this one's end (complete_outputs).
template <typename O, typename W, typename C>
__global__ void __launch_bounds__(kBlock) update_cache_kernel(
    RoundState* st, const std::int32_t* light, const std::int32_t* heavy, unsigned light_blocks,
    unsigned wave_heavy_blocks, const O* offsets, const std::int32_t* neighbors, const W* weights,
    const W* vertex_weights, std::int32_t* labels, const std::int32_t* targets, const std::int32_t* flags,
    std::int32_t* locks, int k, C* cache, unsigned long long* part_weights, long long rebuild_above,
    unsigned long long* status, unsigned long long* counter) {
    __shared__ long long block_sum[kBlock / kWave];
    __shared__ PartMoves moves;
    __shared__ int last;
    // a rebuild round recomputes cache and cut from the CSR after the commit
    const bool update = rebuild_above < 0 || st->edges <= rebuild_above;
    const long long lights = st->light, heavies = st->heavy;
    // the workgroups with movers: the first `pl` light ones, the first `ph` heavy ones
    auto blocks_of = [](long long count, long long per, unsigned blocks) {
        const long long want = (count + per - 1) / per;
        return static_cast<unsigned>(want < blocks ? want : blocks);
    };
    const unsigned pl = blocks_of(wave_heavy_blocks || heavies < lights ? lights : max(lights, heavies),
                                  kBlock / 8, light_blocks);
    const unsigned ph = blocks_of(heavies, kBlock / kWave, wave_heavy_blocks);
    const bool is_light = blockIdx.x < light_blocks;
    const bool none = pl + ph == 0;
    if (is_light ? blockIdx.x >= pl && !(none && blockIdx.x == 0) : blockIdx.x - light_blocks >= ph) return;
    moves.clear();
    long long gain;
    if (is_light) {
        gain = update_cache_movers<O, W, 8, C>(lights, light, offsets, neighbors, weights, vertex_weights, labels,
                                               targets, flags, locks, k, cache, update, blockIdx.x, max(pl, 1U),
                                               moves);
        if (!wave_heavy_blocks)
            for (long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i < heavies;
                 i += static_cast<long long>(max(pl, 1U)) * kBlock) {
                const std::int32_t v = heavy[i];
                commit_mover(v, flags[v] - 1, targets[v], vertex_weights, labels, locks, moves);
            }
    } else {
        gain = update_cache_movers<O, W, kWave, C>(heavies, heavy, offsets, neighbors, weights, vertex_weights,
                                                   labels, targets, flags, locks, k, cache, update,
                                                   blockIdx.x - light_blocks, ph, moves);
    }
    block_add_i64(gain, block_sum, &st->delta);  // its barrier also completes the LDS sums
    moves.flush(k, part_weights);
    if (!status) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long before = __hip_atomic_fetch_add(&st->arrivals, 1ULL, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT);
        last = before + 1 == (none ? 1 : pl + ph);
    }
    __syncthreads();
    if (last && threadIdx.x < kWave) {
        auto load = [](const unsigned long long* p) {
            return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        const auto delta = static_cast<long long>(load(reinterpret_cast<const unsigned long long*>(&st->delta)));
        publish_status(st, [&](int p) { return load(part_weights + p); }, delta, k, status, counter);
    }
}

// The end of a round without an incremental cache (refine_rows.hpp): commits, part
// weights, the cut change and the status (as update_cache_kernel publishes it), in one
// launch. A workgroup takes every gridDim-th heavy mover and spreads their entries over
// its waves in segments of kGainSegment: the cut change is a plain sum, so a long row
// need not stay with one wave. The light movers take 8 lanes each. Hub rows of the
// cache are cleared on the way.
constexpr int kGainSegment = 4 * kWave;
template <typename O, typename W, int Form>
__global__ void __launch_bounds__(kRowsThreads) gain_commit_kernel(
    RoundState* st, const std::int32_t* light, const std::int32_t* heavy, RowLists lists, const unsigned char* states,
    std::int64_t n, const O* offsets, const std::int32_t* neighbors, const W* weights, const W* vertex_weights,
    std::int32_t* labels, const std::int32_t* targets, const std::int32_t* flags, std::int32_t* locks, int k,
    unsigned* cache, unsigned long long* part_weights, unsigned long long* status, unsigned long long* counter) {
    extern __shared__ __align__(16) unsigned lds[];  // the states, stored 16 bytes at once
    __shared__ long long wave_gain[kRowsWaves];
    __shared__ PartMoves moves;
    __shared__ int last;
    __shared__ unsigned wave_segments[kRowsWaves];
    __shared__ unsigned first_segment[kRowsThreads];  // of a pass's movers
    __shared__ std::int32_t mover[kRowsThreads];
    stage_states<Form>(states, n, lds);
    moves.clear();  // its barrier also completes the states
    const States<Form> state{lds, states};
    const int t = threadIdx.x, lane = lane_id(), wave_in = t / kWave;
    const std::int64_t groups = gridDim.x, heavies = st->heavy, lights = st->light;
    long long gain = 0;
    for (std::int64_t base = blockIdx.x; base < heavies; base += groups * kRowsThreads) {
        const std::int64_t i = base + t * groups;
        unsigned segments = 0;
        std::int32_t v = 0;
        if (i < heavies) {
            v = heavy[i];
            segments = static_cast<unsigned>((offsets[v + 1] - offsets[v] + kGainSegment - 1) / kGainSegment);
            commit_mover(v, flags[v] - 1, targets[v], vertex_weights, labels, locks, moves);
        }
        const unsigned inclusive = wave_scan(segments);
        if (lane == kWave - 1) wave_segments[wave_in] = inclusive;
        __syncthreads();
        unsigned before = 0, all = 0;
        for (int w = 0; w < kRowsWaves; ++w) {
            if (w == wave_in) before = all;
            all += wave_segments[w];
        }
        first_segment[t] = before + inclusive - segments;
        mover[t] = v;
        __syncthreads();
        // the last mover whose first segment is not behind s owns segment s
        for (unsigned s = static_cast<unsigned>(wave_in); s < all; s += kRowsWaves) {
            int lo = 0;
#pragma unroll
            for (int step = kRowsThreads / 2; step > 0; step /= 2)
                if (first_segment[lo + step] <= s) lo += step;
            const std::int32_t x = mover[lo];
            const std::int64_t begin = static_cast<std::int64_t>(offsets[x]) +
                                       static_cast<std::int64_t>(s - first_segment[lo]) * kGainSegment;
            const auto row_end = static_cast<std::int64_t>(offsets[x + 1]);
            const std::int64_t end = begin + kGainSegment < row_end ? begin + kGainSegment : row_end;
            gain += mover_gain<kWave, kGainSegment / kWave>(x, flags[x] - 1, state.part(x), begin, end, lane, neighbors,
                                                            weights, state, flags);
        }
        __syncthreads();
    }
    for (std::int64_t i = blockIdx.x + (t / 8) * groups; i < lights; i += groups * (kRowsThreads / 8)) {
        const std::int32_t v = light[i], source = flags[v] - 1, target = targets[v];
        if ((t & 7) == 0) commit_mover(v, source, target, vertex_weights, labels, locks, moves);
        gain += mover_gain<8, 4>(v, source, target, static_cast<std::int64_t>(offsets[v]),
                                 static_cast<std::int64_t>(offsets[v + 1]), t & 7, neighbors, weights, state, flags);
    }
    if (lists.chunk_total) {
        const std::int64_t chunks = *lists.chunk_total;
        for (std::int64_t c = static_cast<std::int64_t>(blockIdx.x) * kRowsWaves + wave_in; c < chunks;
             c += groups * kRowsWaves) {
            const std::int32_t i = lists.chunk_hub[c];
            if (c == lists.chunk_start[i] && lane < k) cache[static_cast<std::int64_t>(lists.high[i]) * k + lane] = 0;
        }
    }
    gain = group_sum_i64<kWave>(gain);
    if (lane == 0) wave_gain[wave_in] = gain;
    __syncthreads();  // also completes the LDS sums of the part weights
    if (t == 0) {
        long long total = 0;
        for (int w = 0; w < kRowsWaves; ++w) total += wave_gain[w];
        if (total) atomicAdd(reinterpret_cast<unsigned long long*>(&st->delta), static_cast<unsigned long long>(total));
    }
    moves.flush(k, part_weights);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t == 0) {
        const unsigned long long arrived = __hip_atomic_fetch_add(&st->arrivals, 1ULL, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT);
        last = arrived + 1 == gridDim.x;
    }
    __syncthreads();
    if (last && t < kWave) {
        auto load = [](const unsigned long long* p) {
            return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        const auto delta = static_cast<long long>(load(reinterpret_cast<const unsigned long long*>(&st->delta)));
        publish_status(st, [&](int p) { return load(part_weights + p); }, delta, k, status, counter);
    }
}

// Heavy movers (degree > kHeavyDegree) as one flattened entry range: heavy_start
// holds the exclusive prefix of their degrees (count + 1 entries, the last one
// the total), tiled as in tiles.hpp with the movers as rows.
template <typename O>
struct HeavyDegreeLoad {
    const RoundState* st;
    const std::int32_t* heavy;
    const O* offsets;
    __device__ __forceinline__ long long operator()(std::int64_t i) const {
        if (i >= st->heavy) return 0;
        const std::int32_t v = heavy[i];
        return static_cast<long long>(offsets[v + 1] - offsets[v]);
    }
};

__global__ void heavy_tiles_kernel(const RoundState* st, const long long* heavy_start, std::int32_t* tile_mover) {
    const long long count = st->heavy;
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
         i += static_cast<long long>(gridDim.x) * blockDim.x) {
        const long long lo = heavy_start[i], hi = heavy_start[i + 1];
        for (long long t = (lo + kTileEdges - 1) / kTileEdges; t * kTileEdges < hi; ++t)
            tile_mover[t] = static_cast<std::int32_t>(i);
    }
}

// incremental_update_cache_and_cut over the heavy movers' entries, kTileRun per lane
// (update_cache_kernel has committed them; flags holds their old parts).
template <typename O, typename W, typename C>
__global__ void __launch_bounds__(kTileLanes) update_cache_tiles_kernel(
    const RoundState* st, const long long* heavy_start, const std::int32_t* tile_mover, const std::int32_t* movers,
    const O* offsets, const std::int32_t* neighbors, const W* weights, const std::int32_t* labels,
    const std::int32_t* targets, const std::int32_t* flags, int k, C* cache, long long* delta,
    long long rebuild_above) {
    __shared__ long long block_sum[kTileLanes / kWave];
    if (rebuild_above >= 0 && st->edges > rebuild_above) return;  // a rebuild round
    const long long count = st->heavy;
    const long long total = heavy_start[count];
    const long long tiles = tile_count(total);
    long long gain = 0;
    for (long long t = blockIdx.x; t < tiles; t += gridDim.x) {
        std::int64_t x, stop;
        std::int32_t i;
        if (!tile_run(heavy_start, tile_mover, tiles, count, total, t, &x, &stop, &i)) continue;
        std::int32_t v = movers[i];
        std::int32_t source = flags[v] - 1, target = targets[v];
        long long next = heavy_start[i + 1];
        std::int64_t base = static_cast<std::int64_t>(offsets[v]) - heavy_start[i];
        for (; x < stop; ++x) {
            while (x >= next) {
                ++i;
                v = movers[i];
                source = flags[v] - 1;
                target = targets[v];
                base = static_cast<std::int64_t>(offsets[v]) - heavy_start[i];
                next = heavy_start[i + 1];
            }
            const std::int64_t e = base + x;
            const std::int32_t u = neighbors[e];
            if (u == v) continue;
            const auto w = static_cast<unsigned long long>(weights[e]);
            atomicAdd(cache + static_cast<std::int64_t>(u) * k + source, static_cast<C>(0ULL - w));
            atomicAdd(cache + static_cast<std::int64_t>(u) * k + target, static_cast<C>(w));
            const std::int32_t fu = flags[u];
            if (!fu || u > v) {
                const std::int32_t lu = fu ? fu - 1 : labels[u];
                const std::int32_t nu = fu ? targets[u] : lu;
                gain += static_cast<long long>(w) * ((source != lu) - (target != nu));
            }
        }
    }
    static_assert(kTileLanes == kBlock, "block_add_i64 sums a kBlock-thread workgroup");
    block_add_i64(gain, block_sum, delta);
}

// Movers are split by degree so the cache update can give heavy rows a workgroup.
struct MoverPair {
    long long light, heavy, edges;
};
struct MoverPairOp {
    __device__ __forceinline__ MoverPair identity() const { return MoverPair{0, 0, 0}; }
    __device__ __forceinline__ MoverPair operator()(const MoverPair& a, const MoverPair& b) const {
        return MoverPair{a.light + b.light, a.heavy + b.heavy, a.edges + b.edges};
    }
};
template <typename O>
struct MoverLoad {
    const std::int32_t* flags;
    const O* offsets;
    __device__ __forceinline__ MoverPair operator()(std::int64_t v) const {
        if (!flags[v]) return MoverPair{0, 0, 0};
        const long long degree = static_cast<long long>(offsets[v + 1] - offsets[v]);
        const bool heavy = degree > kHeavyDegree;
        return MoverPair{heavy ? 0 : 1, heavy ? 1 : 0, degree};
    }
};
struct MoverStore {
    std::int32_t* light;
    std::int32_t* heavy;
    std::int64_t n;
    RoundState* st;
    __device__ __forceinline__ void operator()(std::int64_t v, const MoverPair& prefix, const MoverPair& item) const {
        if (item.light) light[prefix.light] = static_cast<std::int32_t>(v);
        if (item.heavy) heavy[prefix.heavy] = static_cast<std::int32_t>(v);
        if (v == n - 1) {
            st->light = prefix.light + item.light;
            st->heavy = prefix.heavy + item.heavy;
            st->edges = prefix.edges + item.edges;
        }
    }
};

// ---------------------------------------------------------------- rebalance
//
// One iteration of the reference's two-sided bucketed rebalance:
//   proposals   every vertex of an overloaded part picks a destination and lands
//               in a source bucket (part, gain class, section);
//   sources     a vertex leaves when the weight ranked before it in its part's
//               bucket order is below the part's overload;
//   destinations it is admitted when the weight ranked before it plus its own
//               fits the destination's slack.
// Buckets are visited in a fixed order, so within one part every bucket is
// either wholly taken, wholly refused, or the single boundary bucket that
// straddles the part's threshold. Only boundary members need a rank; they get
// the weight of the lower-id members of their bucket (a blocked multisplit),
// one legal outcome of the reference's atomicAdd ranking.

// The overloaded parts as a bit mask. Called by whole waves.
__device__ __forceinline__ unsigned overloaded_parts(const unsigned long long* part_weights, int k,
                                                     std::uint64_t capacity) {
    const int lane = lane_id();
    return static_cast<unsigned>(__ballot(lane < k && part_weights[lane < k ? lane : 0] > capacity));
}

// Candidates: vertices of overloaded parts, in id order, by a count per tile of
// kBlock * Items vertices and a pass that lists them behind the counts below its tile.
// A thread's vertices are kBlock apart (coalesced), a tile's order is (item, wave,
// lane). The generic scan, with its gather of a part weight per vertex and pass, took
// 5.3 + 8.6 us on the 128^3 mesh's levels on average.
constexpr int kTileWaves = kBlock / kWave;
constexpr std::int64_t kCandidateTiles = 1024;  // every workgroup sums the counts below its own

template <int Items>
__global__ void __launch_bounds__(kBlock) candidate_count_kernel(std::int64_t n, const std::int32_t* labels,
                                                                 const unsigned long long* part_weights, int k,
                                                                 std::uint64_t capacity, std::int32_t* tile_counts) {
    __shared__ int wave_counts[kTileWaves];
    const unsigned over = overloaded_parts(part_weights, k, capacity);
    const std::int64_t base = static_cast<std::int64_t>(blockIdx.x) * kBlock * Items + threadIdx.x;
    std::int32_t label[Items];
#pragma unroll
    for (int i = 0; i < Items; ++i) label[i] = base + i * kBlock < n ? labels[base + i * kBlock] : -1;
    int count = 0;
#pragma unroll
    for (int i = 0; i < Items; ++i) count += __popcll(__ballot(label[i] >= 0 && (over >> label[i] & 1U)));
    if (lane_id() == 0) wave_counts[threadIdx.x / kWave] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
        for (int w = 0; w < kTileWaves; ++w) total += wave_counts[w];
        tile_counts[blockIdx.x] = total;
    }
}

// Every flag is cleared on the way (movers are flagged later in the iteration), and
// the states of refine_rows.hpp, where the level has them, are rewritten.
template <int Items>
__global__ void __launch_bounds__(kBlock) candidate_list_kernel(RoundState* st, std::int64_t n,
                                                                const std::int32_t* labels,
                                                                const unsigned long long* part_weights, int k,
                                                                std::uint64_t capacity,
                                                                const std::int32_t* tile_counts,
                                                                std::int32_t* candidates, std::int32_t* flags,
                                                                unsigned char* state) {
    static_assert(Items * kTileWaves <= 2 * kWave, "one wave scans the counts, two per lane");
    __shared__ int at[Items * kTileWaves];
    __shared__ int below[kTileWaves];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const unsigned over = overloaded_parts(part_weights, k, capacity);
    const std::int64_t base = static_cast<std::int64_t>(blockIdx.x) * kBlock * Items + threadIdx.x;
    std::int32_t label[Items];
#pragma unroll
    for (int i = 0; i < Items; ++i) label[i] = base + i * kBlock < n ? labels[base + i * kBlock] : -1;
    int carry = 0;
    for (int t = threadIdx.x; t < static_cast<int>(blockIdx.x); t += kBlock) carry += tile_counts[t];
    carry = wave_scan(carry);
    if (lane == kWave - 1) below[wave] = carry;
#pragma unroll
    for (int i = 0; i < Items; ++i) {
        const unsigned long long in = __ballot(label[i] >= 0 && (over >> label[i] & 1U));
        if (lane == 0) at[i * kTileWaves + wave] = __popcll(in);
    }
    __syncthreads();
    if (wave == 0) {
        int first = 0;
        for (int w = 0; w < kTileWaves; ++w) first += below[w];
        constexpr int kPer = (Items * kTileWaves + kWave - 1) / kWave;
        int counts[kPer], sum = 0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            counts[i] = lane * kPer + i < Items * kTileWaves ? at[lane * kPer + i] : 0;
            sum += counts[i];
        }
        const int inclusive = wave_scan(sum);
        int running = first + inclusive - sum;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (lane * kPer + i < Items * kTileWaves) at[lane * kPer + i] = running;
            running += counts[i];
        }
        if (lane == kWave - 1 && blockIdx.x == gridDim.x - 1) st->candidates = running;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Items; ++i) {
        const bool is = label[i] >= 0 && (over >> label[i] & 1U);
        const unsigned long long in = __ballot(is);
        const std::int64_t v = base + i * kBlock;
        if (is) candidates[at[i * kTileWaves + wave] + __popcll(in & lanemask_lt())] = static_cast<std::int32_t>(v);
        if (label[i] >= 0) {
            flags[v] = 0;
            if (state) state[v] = static_cast<unsigned char>(label[i]);
        }
    }
}

// The same for levels of more tiles, through the generic scan.
struct OverloadedLoad {
    const std::int32_t* labels;
    const unsigned long long* part_weights;
    std::uint64_t capacity;
    // 32-bit counts: vertex ids, and so candidate counts, stay below 2^31
    __device__ __forceinline__ int operator()(std::int64_t v) const {
        return part_weights[labels[v]] > capacity ? 1 : 0;
    }
};
struct CandidateStore {
    std::int32_t* candidates;
    std::int32_t* flags;
    const std::int32_t* labels;
    unsigned char* state;  // refine_rows.hpp, or null
    std::int64_t n;
    RoundState* st;
    __device__ __forceinline__ void operator()(std::int64_t v, int prefix, int item) const {
        flags[v] = 0;
        if (state) state[v] = static_cast<unsigned char>(labels[v]);
        if (item) candidates[prefix] = static_cast<std::int32_t>(v);
        if (v == n - 1) st->candidates = prefix + item;
    }
};

// The choice of incremental_rebalance_proposals (:111-157) for one vertex of an
// overloaded part, by a group of G lanes, lane j owning parts [8j, 8j + 8) of its
// cache row: the destination (-1: none) and the source bucket (-1: none). Every lane
// returns both. U: the type of connectivities and slacks. 32 bits hold them, and every
// sum of slacks, when cache entries have 4 bytes and k parts of the capacity fit; the
// 64-bit form spent most of the finest mesh level's 62 us per launch in arithmetic.
struct BalanceChoice {
    int target;
    int bucket;
};
// The parts' slacks (0: no part, or full) and the bucket thresholds, in LDS.
template <typename U>
struct BalanceTables {
    U slack[4 * kRowSpan];
    double powers[48];
    __device__ __forceinline__ void load(const unsigned long long* part_weights, int k, std::uint64_t capacity,
                                         const PowerTable& table) {
        const int t = threadIdx.x;
        if (t < 4 * kRowSpan) {
            const unsigned long long w = t < k ? part_weights[t] : capacity;
            slack[t] = static_cast<U>(w < capacity ? capacity - w : 0);
        }
        if (t >= kWave && t < kWave + 48) powers[t - kWave] = table.value[t - kWave];
    }
};
template <typename U>
__device__ __forceinline__ U group_xor(U v, int mask, int width) {
    if constexpr (sizeof(U) == 4) return lane_xor(v, mask, width);
    else return shfl_xor_u64(v, mask, width);
}
template <typename U>
__device__ __forceinline__ U saturated(U a, U b) {
    if constexpr (sizeof(U) == 4) return a + b;  // every sum of slacks fits
    else return ~U{0} - a < b ? ~U{0} : a + b;
}
template <int G, typename U, typename C>
__device__ __forceinline__ BalanceChoice balance_choice(std::int64_t v, std::int32_t source, std::uint64_t weight,
                                                        const C* cache, int j, int k, const BalanceTables<U>& tables) {
    const C* row = cache + v * k;
    const U w = sizeof(U) == 4 && weight > 0xffffffffULL ? static_cast<U>(~U{0}) : static_cast<U>(weight);
    U slack[kRowSpan];
    U conn = 0, best_slack = 0, current = 0;
    int bp = 0x7fffffff;
    U span[kRowSpan];
    load_span(row, j, k, span);
    // lane-local best by (conn, slack), lowest index on ties (ascending p)
#pragma unroll
    for (int e = 0; e < kRowSpan; ++e) {
        const int p = j * kRowSpan + e;
        const U value = span[e];
        if (p == source) current = value;
        const U room = tables.slack[p];
        const bool ok = p != source && room > 0 && w <= room;
        slack[e] = ok ? room : 0;
        if (ok && (bp == 0x7fffffff || value > conn || (value == conn && room > best_slack))) {
            conn = value;
            best_slack = room;
            bp = p;
        }
    }
#pragma unroll
    for (int m = G / 2; m > 0; m /= 2) {
        const U oc = group_xor(conn, m, G);
        const U os = group_xor(best_slack, m, G);
        const int op = static_cast<int>(lane_xor(static_cast<unsigned>(bp), m, G));
        const U ocur = group_xor(current, m, G);
        const bool ob = op != 0x7fffffff;
        const bool mine = bp != 0x7fffffff;
        if (ob && (!mine || oc > conn || (oc == conn && (os > best_slack || (os == best_slack && op < bp))))) {
            conn = oc;
            best_slack = os;
            bp = op;
        }
        current = ocur > current ? ocur : current;  // only the source's lane holds it
    }
    int best = bp == 0x7fffffff ? -1 : bp;
    if (best >= 0 && conn == 0) {
        // No affinity anywhere: a ticket mix32(v) mod total slack walks the
        // eligible parts in index order. Saturating sums of non-negative terms do
        // not depend on the order of addition, so the running total before part p
        // is the lane's running prefix plus the saturated total of lower lanes;
        // the walk stops at the first part whose running total exceeds the ticket.
        U running[kRowSpan];
        U lane_total = 0;
#pragma unroll
        for (int e = 0; e < kRowSpan; ++e) {
            lane_total = saturated(lane_total, slack[e]);
            running[e] = lane_total;
        }
        // the totals of the group's lanes: up to four, exchanged by xor
        U lower = 0, total = lane_total;
#pragma unroll
        for (int m = 1; m < G; m <<= 1) {
            const U other = group_xor(total, m, G);
            if (j & m) lower = saturated(lower, other);
            total = saturated(total, other);
        }
        const std::uint32_t hash = mix32(static_cast<std::uint32_t>(v));
        const U ticket = sizeof(U) == 8 && total > 0xffffffffULL ? hash : hash % static_cast<std::uint32_t>(total);
        int hit = 0x7fffffff;
#pragma unroll
        for (int e = kRowSpan - 1; e >= 0; --e)
            if (saturated(lower, running[e]) > ticket) hit = j * kRowSpan + e;
#pragma unroll
        for (int m = G / 2; m > 0; m /= 2) {
            const int other = static_cast<int>(lane_xor(static_cast<unsigned>(hit), m, G));
            hit = other < hit ? other : hit;
        }
        best = hit;
    }
    int bucket = -1;
    if (best >= 0) {
        const double gain =
            conn >= current ? static_cast<double>(conn - current) : -static_cast<double>(current - conn);
        const double per_weight = gain / static_cast<double>(weight);
        bucket = source * kBalanceWidth + gain_bucket(per_weight, tables.powers) * kBalanceSections +
                 static_cast<int>(mix32(static_cast<std::uint32_t>(v)) % kBalanceSections);
    }
    return BalanceChoice{best, bucket};
}

// incremental_rebalance_proposals (:111-157) + balance_source_histogram (:174-186).
// One group of G lanes per candidate, lane j owning parts [8j, 8j + 8).
template <typename W, int G, typename U, typename C>
__global__ void __launch_bounds__(kBlock) balance_proposals_kernel(RoundState* st, const std::int32_t* cand,
                                                                   const C* cache,
                                                                   const std::int32_t* labels, const W* vertex_weights,
                                                                   int k, const unsigned long long* part_weights,
                                                                   std::uint64_t capacity, PowerTable powers,
                                                                   std::int32_t* targets, std::int32_t* cbucket,
                                                                   unsigned long long* replicas) {
    __shared__ BalanceTables<U> tables;
    __shared__ BucketTable table;
    // the round state past the candidate count starts at zero
    constexpr unsigned kCandidateWord = offsetof(RoundState, candidates) / 8;
    if (blockIdx.x == 0 && threadIdx.x < sizeof(RoundState) / 8 && threadIdx.x != kCandidateWord)
        reinterpret_cast<unsigned long long*>(st)[threadIdx.x] = 0;
    tables.load(part_weights, k, capacity, powers);
    table_clear(table);
    __syncthreads();
    unsigned long long* counts = replicas + static_cast<long long>(blockIdx.x % kReplicas) * k * kBalanceWidth;
    const long long count = st->candidates;
    const int j = threadIdx.x & (G - 1);
    const long long groups = static_cast<long long>(gridDim.x) * (kBlock / G);
    for (long long index = (static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x) / G; index < count;
         index += groups) {
        const std::int64_t v = cand[index];
        const std::int32_t source = labels[v];
        const std::uint64_t weight = static_cast<std::uint64_t>(vertex_weights[v]);
        const BalanceChoice choice = balance_choice<G, U>(v, source, weight, cache, j, k, tables);
        if (j == 0) {
            if (choice.bucket >= 0) table_add(table, static_cast<unsigned>(choice.bucket), weight, counts);
            targets[v] = choice.target;
            cbucket[index] = choice.bucket;
        }
    }
    __syncthreads();
    table_flush(table, counts);
}

// ---------------------------------------------------------------- small levels
//
// A rebalance iteration of a level of at most kSelectVertices vertices takes three
// launches: the proposals of every vertex (no candidate list: a vertex of a part
// within capacity is skipped), both selections in one workgroup, and the update.
// Such a level is bound by its chain of launches, each 3-5 us whatever it does: the
// ten launches these two replace (candidate scan, proposals, two bucket scans, two
// times two selections, commit, status) took 46-65 us per iteration with the host's
// wait, on levels of 669 to 12,220 vertices.

// balance_choice for every vertex of an overloaded part. choices[v]: the bucket
// within a part in bits 0-9, the source part in bits 10-14, the destination in bits
// 15-19; -1 for a vertex without a destination, -2 for one of no overloaded part.
// Flags and the round state are cleared on the way.
constexpr int kNoCandidate = -2;
constexpr int kBucketBits = 10, kSourceShift = 10, kTargetShift = 15;
static_assert(kBalanceWidth <= 1 << kBucketBits, "a part's buckets fit their field");
template <typename W, int G, typename U, typename C>
__global__ void __launch_bounds__(kBlock) balance_vertices_kernel(RoundState* st, std::int64_t n, const C* cache,
                                                                  const std::int32_t* labels, const W* vertex_weights,
                                                                  int k, const unsigned long long* part_weights,
                                                                  std::uint64_t capacity, PowerTable powers,
                                                                  std::int32_t* targets, std::int32_t* choices,
                                                                  std::int32_t* flags, unsigned char* state) {
    __shared__ BalanceTables<U> tables;
    if (blockIdx.x == 0 && threadIdx.x < sizeof(RoundState) / 8)
        reinterpret_cast<unsigned long long*>(st)[threadIdx.x] = 0;
    tables.load(part_weights, k, capacity, powers);
    const unsigned over = overloaded_parts(part_weights, k, capacity);
    __syncthreads();
    const std::int64_t v = (static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / G;
    if (v >= n) return;  // uniform per group
    const int j = threadIdx.x & (G - 1);
    const std::int32_t source = labels[v];
    BalanceChoice choice{-1, kNoCandidate};
    if (over >> source & 1U)  // uniform per group
        choice = balance_choice<G, U>(v, source, static_cast<std::uint64_t>(vertex_weights[v]), cache, j, k, tables);
    if (j == 0) {
        targets[v] = choice.target;
        choices[v] = choice.bucket < 0 ? choice.bucket
                                       : choice.bucket - source * kBalanceWidth + (source << kSourceShift) +
                                             (choice.target << kTargetShift);
        flags[v] = 0;
        if (state) state[v] = static_cast<unsigned char>(source);  // refine_rows.hpp
    }
}

constexpr int kSelectThreads = 1024;
constexpr int kSelectWaves = kSelectThreads / kWave;

// What part p's members may weigh: its overload (sources) or its slack (destinations).
__device__ __forceinline__ unsigned long long part_limit(unsigned long long w, std::uint64_t capacity,
                                                         bool destinations) {
    return destinations ? (w < capacity ? capacity - w : 0) : (w > capacity ? w - capacity : 0);
}

// For parts [base, base + parts), whose buckets' weights are in LDS (narrow, or wide):
// the boundary bucket, the first at which the running weight reaches the limit, and the
// weight before it. Members of lower buckets are all taken, those of higher ones refused
// (source_side and destination_side state the same tests). A wave per part, 13 buckets
// per lane; called by a workgroup of kSelectThreads threads.
__device__ void part_boundaries(const unsigned* narrow, const unsigned long long* wide, int base, int parts,
                                bool destinations, const unsigned long long* pw, std::uint64_t capacity,
                                int* boundary, unsigned long long* before) {
    constexpr int kPer = (kBalanceWidth + kWave - 1) / kWave;
    const int lane = lane_id();
    for (int q = threadIdx.x / kWave; q < parts; q += kSelectWaves) {
        const unsigned long long limit = part_limit(pw[base + q], capacity, destinations);
        if (!destinations && limit == 0) continue;  // not overloaded: no members
        unsigned long long count[kPer], sum = 0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int b = lane * kPer + i;
            count[i] = b >= kBalanceWidth ? 0 : narrow ? narrow[q * kBalanceWidth + b] : wide[q * kBalanceWidth + b];
            sum += count[i];
        }
        unsigned long long running = wave_scan(sum) - sum, at = 0;
        int found = kBalanceWidth;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const bool reached = destinations ? running + count[i] > limit : running + count[i] >= limit;
            if (reached && found == kBalanceWidth && lane * kPer + i < kBalanceWidth) {
                found = lane * kPer + i;
                at = running;
            }
            running += count[i];
        }
        const unsigned long long lanes = __ballot(found < kBalanceWidth);
        const int owner = lanes ? __ffsll(static_cast<unsigned long long>(lanes)) - 1 : 0;
        if (lane == owner) {
            boundary[base + q] = found;
            before[base + q] = at;
        }
    }
}

// Both selections of an iteration in one workgroup. A wave owns 64 * Items
// consecutive vertices, lane l's item i the one at 64 * i + l (every load of a wave
// is one run; Items consecutive vertices per lane took 41 instead of 27 us at 12,220
// vertices); the choices stay in registers. The bucket histogram of the
// sources, then of the destinations, is summed in LDS: 32 parts x 800 buckets of 32
// bits when the part weights' total fits, else 16 parts x 800 of 64 bits per window.
// Within a part the members before the first bucket that reaches its threshold are
// taken, those behind it refused (source_side and destination_side state the same
// tests). That bucket's own members of all parts are gathered in id order into the
// histogram's space and ranked together, kSelectThreads at a time.
constexpr int kSelectMaxItems = 16;
constexpr std::int64_t kSelectVertices = kSelectThreads * kSelectMaxItems;
struct SelectShared {
    union {
        unsigned narrow[32 * kBalanceWidth];
        unsigned long long wide[16 * kBalanceWidth];
        struct {
            std::int32_t vertex[kSelectVertices];
            unsigned char part[kSelectVertices];   // its part
            unsigned char taken[kSelectVertices];  // the outcome
        } pending;
    } u;
    unsigned long long pw[32];
    unsigned long long running[32];  // weight before the boundary bucket, then before the next member
    int boundary[32];                // the boundary bucket, kBalanceWidth: every bucket is taken
    unsigned long long waves[2][kSelectWaves];
    unsigned long long wave_total[kSelectWaves][32];
};

// Exclusive prefix of one value per thread over the kSelectThreads threads, and
// their total: one barrier (the wave totals are scanned by every wave itself);
// successive calls alternate `slot`, so that a call's totals are not overwritten
// before every wave has read them.
__device__ __forceinline__ unsigned long long select_scan(unsigned long long value, unsigned long long* total,
                                                          SelectShared& sh, int slot) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const unsigned long long inclusive = wave_scan(value);
    if (lane == kWave - 1) sh.waves[slot][wave] = inclusive;
    __syncthreads();
    const unsigned long long sums = wave_scan(lane < kSelectWaves ? sh.waves[slot][lane] : 0ULL);
    *total = read_lane(sums, kSelectWaves - 1);
    const auto below = read_lane(sums, __builtin_amdgcn_readfirstlane(wave > 0 ? wave - 1 : 0));
    return (wave > 0 ? below : 0) + inclusive - value;
}

template <typename O, typename W, int Items>
__global__ void __launch_bounds__(kSelectThreads) balance_select_kernel(
    RoundState* st, std::int64_t n, const std::int32_t* choices, const W* vertex_weights, const O* offsets, int k,
    const unsigned long long* part_weights, std::uint64_t capacity, std::int32_t* light, std::int32_t* heavy,
    std::int32_t* flags, unsigned char* state) {
    __shared__ SelectShared sh;
    const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
    const int first = wave * kWave * Items + lane;
    const int count_n = static_cast<int>(n);
    int item[Items];
    W weight[Items];
#pragma unroll
    for (int i = 0; i < Items; ++i) item[i] = first + i * kWave < count_n ? choices[first + i * kWave] : kNoCandidate;
#pragma unroll
    for (int i = 0; i < Items; ++i) weight[i] = first + i * kWave < count_n ? vertex_weights[first + i * kWave] : W{0};
    if (t < 32) sh.pw[t] = t < k ? part_weights[t] : 0;
    __syncthreads();
    unsigned long long total = 0;
    for (int p = 0; p < k; ++p) total += sh.pw[p];
    const bool narrow = total <= 0xffffffffULL;
    const int window = narrow ? 32 : 16;
    unsigned long long candidates = 0;
    unsigned in = 0;  // the items that take part in the selection
#pragma unroll
    for (int i = 0; i < Items; ++i) {
        candidates += item[i] != kNoCandidate;
        in |= static_cast<unsigned>(item[i] >= 0) << i;
    }

    // Selects among the items in `in`, by the part at `shift`: the mask of the taken.
    auto select = [&](int shift, bool destinations) -> unsigned {
        for (int base = 0; base < k; base += window) {
            const int parts = min(window, k - base);
            if (narrow) {
                for (int b = t; b < parts * kBalanceWidth; b += kSelectThreads) sh.u.narrow[b] = 0;
            } else {
                for (int b = t; b < parts * kBalanceWidth; b += kSelectThreads) sh.u.wide[b] = 0;
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < Items; ++i) {
                const int q = (item[i] >> shift & 31) - base;
                if (!(in >> i & 1U) || q < 0 || q >= parts) continue;
                const int b = q * kBalanceWidth + (item[i] & ((1 << kBucketBits) - 1));
                if (narrow) atomicAdd(&sh.u.narrow[b], static_cast<unsigned>(weight[i]));
                else atomicAdd(&sh.u.wide[b], static_cast<unsigned long long>(weight[i]));
            }
            __syncthreads();
            part_boundaries(narrow ? sh.u.narrow : nullptr, sh.u.wide, base, parts, destinations, sh.pw, capacity,
                            sh.boundary, sh.running);
            __syncthreads();
        }
        unsigned taken = 0, pending = 0;
#pragma unroll
        for (int i = 0; i < Items; ++i) {
            if (!(in >> i & 1U)) continue;
            const int b = item[i] & ((1 << kBucketBits) - 1), boundary = sh.boundary[item[i] >> shift & 31];
            if (b < boundary) taken |= 1U << i;
            else if (b == boundary) pending |= 1U << i;
        }
        // the wave's pending items in id order, from the waves' totals
        int in_wave = 0;
#pragma unroll
        for (int i = 0; i < Items; ++i) in_wave += __popcll(__ballot(pending >> i & 1U));
        unsigned long long members;
        const auto at = static_cast<int>(
            select_scan(lane == 0 ? static_cast<unsigned long long>(in_wave) : 0ULL, &members, sh, destinations ? 1 : 0));
        const int wave_at = static_cast<int>(read_lane(static_cast<unsigned>(at), 0));
        int slot = wave_at;
#pragma unroll
        for (int i = 0; i < Items; ++i) {
            const unsigned long long lanes = __ballot(pending >> i & 1U);
            if (pending >> i & 1U) {
                const int x = slot + __popcll(lanes & lanemask_lt());
                sh.u.pending.vertex[x] = first + i * kWave;
                sh.u.pending.part[x] = static_cast<unsigned char>(item[i] >> shift & 31);
            }
            slot += __popcll(lanes);
        }
        __syncthreads();
        for (int base = 0; base < static_cast<int>(members); base += kSelectThreads) {
            const int x = base + t;
            const bool member = x < static_cast<int>(members);
            const int p = member ? sh.u.pending.part[x] : 0;
            const unsigned long long w =
                member ? static_cast<unsigned long long>(vertex_weights[sh.u.pending.vertex[x]]) : 0;
            const unsigned long long rank = block_key_prefix<kSelectThreads>(member, p, w, sh.wave_total, sh.running);
            const unsigned long long limit = part_limit(sh.pw[p], capacity, destinations);
            if (member) sh.u.pending.taken[x] = destinations ? rank + w <= limit : rank < limit;
        }
        __syncthreads();
        slot = wave_at;
#pragma unroll
        for (int i = 0; i < Items; ++i) {
            const unsigned long long lanes = __ballot(pending >> i & 1U);
            if (pending >> i & 1U && sh.u.pending.taken[slot + __popcll(lanes & lanemask_lt())]) taken |= 1U << i;
            slot += __popcll(lanes);
        }
        __syncthreads();
        return taken;
    };

    in = select(kSourceShift, false);
    const unsigned moving = select(kTargetShift, true);

    // the mover lists (their order does not matter)
    unsigned long long counts = 0, edges = 0;
    unsigned is_heavy = 0;
#pragma unroll
    for (int i = 0; i < Items; ++i) {
        if (!(moving >> i & 1U)) continue;
        const int v = first + i * kWave;
        const auto degree = static_cast<unsigned long long>(offsets[v + 1] - offsets[v]);
        edges += degree;
        if (degree > kHeavyDegree) is_heavy |= 1U << i;
        counts += degree > kHeavyDegree ? 1ULL << 20 : 1ULL;
    }
    // light movers, heavy movers and candidates in 20 bits each (at most 2^14)
    unsigned long long listed, all_edges;
    unsigned long long at = select_scan(counts | candidates << 40, &listed, sh, 0) & 0xffffffffffULL;
    (void)select_scan(edges, &all_edges, sh, 1);
#pragma unroll
    for (int i = 0; i < Items; ++i) {
        if (!(moving >> i & 1U)) continue;
        const int v = first + i * kWave;
        if (is_heavy >> i & 1U) {
            heavy[at >> 20] = v;
            at += 1ULL << 20;
        } else {
            light[at & 0xfffffU] = v;
            at += 1;
        }
        flags[v] = (item[i] >> kSourceShift & 31) + 1;
        mark_mover(state, v, item[i] >> kTargetShift & 31);
    }
    if (t == 0) {
        st->light = static_cast<long long>(listed & 0xfffffU);
        st->heavy = static_cast<long long>(listed >> 20 & 0xfffffU);
        st->edges = static_cast<long long>(all_edges);
        st->candidates = static_cast<long long>(listed >> 40);
    }
}

// ---------------------------------------------------------------- large levels
//
// Larger levels list their candidates, histogram the source buckets while they choose,
// and then take four launches for the two selections: the sources' boundary buckets, a
// pass that decides every candidate outside them, a pass that ranks the boundary
// members and gathers the leaving vertices, and one workgroup that selects among
// those. Mostly the leaving vertices are few (their weight is about the overload:
// hundreds to thousands where the candidates are 10^4 to 10^6), so the destinations'
// histogram, scan, ranks and mover lists take one workgroup 12 us; as launches over
// the candidates they were four (six above 256 workgroups) of 4.4-6.2 us each. Where
// the part weights of the last round say that more than ctx->few_leaving vertices leave, the
// destinations too are selected by passes over the slices (R-MAT levels move up to a
// tenth of their vertices at once). An iteration by one workgroup and by passes, in us,
// on grids of 250,000 vertices, k = 8: 60 and 68 for 172 leaving vertices, 68 and 72 for
// 2,226, 79 and 77 for 3,951, 92 and 82 for 6,618, 124 and 89 for 13,943; of 4 M: 108 and
// 120 for 386, 128 and 127 for 5,336, 273 and 155 for 26,998. The line is 4,096.
// That guess counts vertices of average weight, and the last round may have been another
// level's. So the workgroup that finds more than kRefusedShare times as many refuses: the
// iteration moves nothing and runs again with the passes. Its launches up to there are
// spent, 60 to 110 us of the above, which is what one workgroup takes longer for 30,000.
constexpr std::int64_t kRefusedShare = 8;

// balance_scan_buckets (:188-202): the boundary bucket of every overloaded part
// (sources) or of every part (destinations) and the weight before it, from the
// kReplicas copies of the counters, which are zeroed for the next round. One workgroup
// per part, a thread per bucket: its 16 replica loads are independent and all in
// flight at once.
constexpr int kBucketScanThreads = 1024;
static_assert(kBucketScanThreads >= kBalanceWidth, "a thread per bucket");
template <bool Destinations>
__global__ void __launch_bounds__(kBucketScanThreads) bucket_boundaries_kernel(unsigned long long* replicas, int k,
                                                                               const unsigned long long* part_weights,
                                                                               std::uint64_t capacity, int* boundary,
                                                                               unsigned long long* before) {
    __shared__ unsigned long long waves[kBucketScanThreads / kWave + 1];
    const unsigned long long limit = part_limit(part_weights[blockIdx.x], capacity, Destinations);
    if (!Destinations && limit == 0) return;  // not overloaded: no members, its counters are zero
    const long long width = static_cast<long long>(k) * kBalanceWidth;
    const int b = threadIdx.x;
    unsigned long long count = 0;
    if (b < kBalanceWidth) {
        unsigned long long* mine = replicas + static_cast<long long>(blockIdx.x) * kBalanceWidth + b;
#pragma unroll
        for (int r = 0; r < kReplicas; ++r) count += mine[r * width];
#pragma unroll
        for (int r = 0; r < kReplicas; ++r) mine[r * width] = 0;
    }
    unsigned long long total;
    const unsigned long long prefix = block_exclusive_scan(count, SumOp<unsigned long long>{}, &total, waves);
    // the first bucket that reaches the limit; kBalanceWidth when none does
    auto reached = [&](unsigned long long w) { return Destinations ? w > limit : w >= limit; };
    if (b < kBalanceWidth && reached(prefix + count) && (b == 0 || !reached(prefix))) {
        boundary[blockIdx.x] = b;
        before[blockIdx.x] = prefix;
    }
    if (b == 0 && !reached(total)) {
        boundary[blockIdx.x] = kBalanceWidth;
        before[blockIdx.x] = 0;
    }
}

// The selection passes over the candidates: at most kSliceBlocks workgroups, each with
// one contiguous slice.
constexpr int kSliceThreads = 1024;
constexpr int kSliceBlocks = 256;

// balance_select_sources (:204-217) outside the boundary buckets: leaving[i] is the
// candidate's destination code (bucket | part << kBucketBits), kSourcePending for a
// boundary member, whose weights are summed per part and workgroup, or kNoBucket.
template <typename W>
__global__ void __launch_bounds__(kSliceThreads) balance_sources_kernel(const RoundState* st, const std::int32_t* cand,
                                                                        const std::int32_t* cbucket,
                                                                        std::int32_t* leaving,
                                                                        const std::int32_t* targets,
                                                                        const W* vertex_weights, const int* boundary,
                                                                        unsigned long long* block_sums) {
    __shared__ unsigned long long sums[32];
    __shared__ int bounds[32];
    if (threadIdx.x < 32) {
        sums[threadIdx.x] = 0;
        bounds[threadIdx.x] = boundary[threadIdx.x];  // set for overloaded parts, which all members belong to
    }
    __syncthreads();
    long long begin, end;
    block_slice(st->candidates, begin, end);
    for (long long i = begin + threadIdx.x; i < end; i += kSliceThreads) {
        const int b = cbucket[i];
        int code = kNoBucket;
        if (b >= 0) {
            const int part = b / kBalanceWidth, bucket = b % kBalanceWidth;
            if (bucket < bounds[part]) {
                code = bucket | targets[cand[i]] << kBucketBits;
            } else if (bucket == bounds[part]) {
                code = kSourcePending;
                atomicAdd(&sums[part], static_cast<unsigned long long>(vertex_weights[cand[i]]));
            }
        }
        leaving[i] = code;
    }
    __syncthreads();
    if (threadIdx.x < 32) block_sums[static_cast<long long>(blockIdx.x) * 32 + threadIdx.x] = sums[threadIdx.x];
}

// The boundary weights of the workgroups below this one, per part, on top of the weight
// before the boundary bucket where the part has a limit. Called by the workgroup.
constexpr int kSliceRows = kSliceThreads / 32;
__device__ __forceinline__ void slice_running(const unsigned long long* block_sums, const unsigned long long* before,
                                              const unsigned long long* part_weights, int k, std::uint64_t capacity,
                                              bool destinations, unsigned long long (*rows)[32],
                                              unsigned long long* running, unsigned long long* limits) {
    const int part = threadIdx.x & 31, row = threadIdx.x >> 5;
    unsigned long long sum = 0;
    for (int b = row; b < static_cast<int>(blockIdx.x); b += kSliceRows)
        sum += block_sums[static_cast<long long>(b) * 32 + part];
    rows[row][part] = sum;
    __syncthreads();
    if (threadIdx.x < 32) {
        const bool is = threadIdx.x < static_cast<unsigned>(k);
        const unsigned long long limit =
            is ? part_limit(part_weights[threadIdx.x], capacity, destinations) : 0;
        limits[threadIdx.x] = limit;
        unsigned long long total = is && (destinations || limit) ? before[threadIdx.x] : 0;
        for (int r = 0; r < kSliceRows; ++r) total += rows[r][threadIdx.x];
        running[threadIdx.x] = total;
    }
    __syncthreads();
}

// Source boundary members: they leave while the weight before the bucket plus their
// rank is below the overload. The slice's leaving vertices are gathered, in id order,
// at the front of its range of left_vertex and left_code. Table: their weights are also
// added to the destination buckets' counters.
template <typename W, bool Table>
__global__ void __launch_bounds__(kSliceThreads) balance_source_ranks_kernel(
    const RoundState* st, const std::int32_t* cand, const std::int32_t* cbucket, const std::int32_t* leaving,
    const std::int32_t* targets, const W* vertex_weights, const unsigned long long* part_weights, int k,
    std::uint64_t capacity, const unsigned long long* before, const unsigned long long* block_sums,
    std::int32_t* left_vertex, std::int32_t* left_code, std::int32_t* left_count, unsigned long long* replicas) {
    constexpr int kWaves = kSliceThreads / kWave;
    __shared__ unsigned long long wave_total[kWaves][32];
    __shared__ unsigned long long running[32], limits[32];
    __shared__ unsigned long long rows[kSliceRows][32];
    __shared__ int wave_left[2][kWaves];
    __shared__ std::conditional_t<Table, BucketTable, int> table;
    unsigned long long* counts = replicas + static_cast<long long>(blockIdx.x % kReplicas) * k * kBalanceWidth;
    if constexpr (Table) table_clear(table);
    slice_running(block_sums, before, part_weights, k, capacity, false, rows, running, limits);
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    long long begin, end;
    block_slice(st->candidates, begin, end);
    int left = 0, turn = 0;
    for (long long base = begin; base < end; base += kSliceThreads) {
        const long long i = base + threadIdx.x;
        int code = i < end ? leaving[i] : kNoBucket;
        const bool pending = code == kSourcePending;
        if (!__syncthreads_or(code != kNoBucket)) continue;
        if (__syncthreads_or(pending)) {
            const int b = pending ? cbucket[i] : 0, part = b / kBalanceWidth;
            const std::int32_t v = pending ? cand[i] : 0;
            const unsigned long long w = pending ? static_cast<unsigned long long>(vertex_weights[v]) : 0;
            const unsigned long long rank = block_key_prefix<kSliceThreads>(pending, part, w, wave_total, running);
            if (pending) code = rank < limits[part] ? b % kBalanceWidth | targets[v] << kBucketBits : kNoBucket;
        }
        const unsigned long long lanes = __ballot(code >= 0);
        if (lane == 0) wave_left[turn][wave] = __popcll(lanes);
        __syncthreads();
        int at = left;
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave) at += wave_left[turn][w];
            left += wave_left[turn][w];
        }
        turn ^= 1;
        if (code >= 0) {
            at += __popcll(lanes & lanemask_lt());
            const std::int32_t v = cand[i];
            left_vertex[begin + at] = v;
            left_code[begin + at] = code;
            if constexpr (Table)
                table_add(table,
                          static_cast<unsigned>((code >> kBucketBits) * kBalanceWidth + (code & ((1 << kBucketBits) - 1))),
                          static_cast<unsigned long long>(vertex_weights[v]), counts);
        }
    }
    if (threadIdx.x == 0) left_count[blockIdx.x] = left;
    if constexpr (Table) {
        __syncthreads();
        table_flush(table, counts);
    }
}

// balance_select_destinations (:219-232) over the slices' leaving vertices, in two
// passes. Ranks == false: those of buckets below the boundary move, the boundary
// members' weights are summed per part and workgroup. Ranks == true: boundary members
// move while the weight before the bucket, their rank and their own weight fit.
template <typename O, typename W, bool Ranks>
__global__ void __launch_bounds__(kSliceThreads) balance_slices_kernel(
    RoundState* st, const std::int32_t* left_vertex, const std::int32_t* left_code, const std::int32_t* left_count,
    const std::int32_t* labels, const W* vertex_weights, const O* offsets, int k,
    const unsigned long long* part_weights, std::uint64_t capacity, const int* boundary,
    const unsigned long long* before, unsigned long long* block_sums, std::int32_t* light, std::int32_t* heavy,
    std::int32_t* flags, unsigned char* state) {
    constexpr int kWaves = kSliceThreads / kWave;
    __shared__ unsigned long long wave_total[kWaves][32];
    __shared__ unsigned long long running[32], limits[32];
    __shared__ unsigned long long rows[kSliceRows][32];
    __shared__ int bounds[32];
    __shared__ unsigned counts[2 * kWaves];
    __shared__ unsigned long long bases[2];
    if (threadIdx.x < 32) bounds[threadIdx.x] = threadIdx.x < static_cast<unsigned>(k) ? boundary[threadIdx.x] : 0;
    if constexpr (Ranks) {
        slice_running(block_sums, before, part_weights, k, capacity, true, rows, running, limits);
    } else {
        if (threadIdx.x < 32) running[threadIdx.x] = 0;  // the workgroup's sums
        __syncthreads();
    }
    long long begin, end;
    block_slice(st->candidates, begin, end);
    end = begin + left_count[blockIdx.x];
    for (long long base = begin; base < end; base += kSliceThreads) {
        const long long i = base + threadIdx.x;
        std::int32_t v = 0;
        int part = 0;
        bool take = false, pending = false;
        if (i < end) {
            const int code = left_code[i], bucket = code & ((1 << kBucketBits) - 1);
            part = code >> kBucketBits;
            pending = bucket == bounds[part];
            take = !Ranks && bucket < bounds[part];
            if (take || pending) v = left_vertex[i];
        }
        const unsigned long long w = pending ? static_cast<unsigned long long>(vertex_weights[v]) : 0;
        if constexpr (Ranks) {
            if (!__syncthreads_or(pending)) continue;
            const unsigned long long rank = block_key_prefix<kSliceThreads>(pending, part, w, wave_total, running);
            take = pending && rank + w <= limits[part];
        } else if (pending) {
            atomicAdd(&running[part], w);
        }
        if (take) {
            flags[v] = labels[v] + 1;
            mark_mover(state, v, part);
        }
        append_movers<kSliceThreads>(take, v, offsets, light, heavy, st, counts, bases);
    }
    if constexpr (!Ranks) {
        __syncthreads();
        if (threadIdx.x < 32) block_sums[static_cast<long long>(blockIdx.x) * 32 + threadIdx.x] = running[threadIdx.x];
    }
}

// balance_select_destinations (:219-232) over all leaving vertices, by one workgroup: the
// destination buckets' weights in LDS (as in balance_select_kernel), their boundary
// buckets, then the vertices in id order, kSelectThreads at a time: those of lower
// buckets move, boundary members while the weight before the bucket, their rank and
// their own weight fit the slack.
struct DestinationShared {
    union {
        unsigned narrow[32 * kBalanceWidth];
        unsigned long long wide[16 * kBalanceWidth];
    } u;
    unsigned long long pw[32];
    unsigned long long running[32];
    int boundary[32];
    unsigned long long wave_total[kSelectWaves][32];
    int first[kSliceBlocks];  // of each slice's vertices in the order of all
    int waves[kSelectWaves];
    unsigned light, heavy;
    unsigned long long edges;
};
template <typename O, typename W>
__global__ void __launch_bounds__(kSelectThreads) balance_destinations_kernel(
    RoundState* st, int slices, const std::int32_t* left_vertex, const std::int32_t* left_code,
    const std::int32_t* left_count, const std::int32_t* labels, const W* vertex_weights, const O* offsets, int k,
    const unsigned long long* part_weights, std::uint64_t capacity, std::int64_t most, std::int32_t* light,
    std::int32_t* heavy, std::int32_t* flags, unsigned char* state) {
    __shared__ DestinationShared sh;
    const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
    const long long candidates = st->candidates, per = (candidates + slices - 1) / slices;
    const int mine = t < slices ? left_count[t] : 0;
    if (t < 32) sh.pw[t] = t < k ? part_weights[t] : 0;
    if (t == 0) {
        sh.light = sh.heavy = 0;
        sh.edges = 0;
    }
    const int inclusive = wave_scan(mine);
    if (lane == kWave - 1) sh.waves[wave] = inclusive;
    __syncthreads();
    int below = 0, count = 0;
    for (int w = 0; w < kSelectWaves; ++w) {
        if (w == wave) below = count;
        count += sh.waves[w];
    }
    if (count > most) {  // uniform
        if (t == 0) st->refused = 1;
        return;
    }
    if (t < kSliceBlocks) sh.first[t] = below + inclusive - mine;
    unsigned long long total = 0;
    for (int p = 0; p < k; ++p) total += sh.pw[p];
    const bool narrow = total <= 0xffffffffULL;
    const int window = narrow ? 32 : 16;
    __syncthreads();
    // the x-th leaving vertex: in the last slice that starts at or before it
    auto locate = [&](int x) -> long long {
        int lo = 0;
#pragma unroll
        for (int step = kSliceBlocks / 2; step > 0; step /= 2)
            if (sh.first[lo + step] <= x) lo += step;
        return lo * per + (x - sh.first[lo]);
    };
    for (int base = 0; base < k; base += window) {
        const int parts = min(window, k - base);
        if (narrow) {
            for (int b = t; b < parts * kBalanceWidth; b += kSelectThreads) sh.u.narrow[b] = 0;
        } else {
            for (int b = t; b < parts * kBalanceWidth; b += kSelectThreads) sh.u.wide[b] = 0;
        }
        __syncthreads();
        for (int x = t; x < count; x += kSelectThreads) {
            const long long i = locate(x);
            const int code = left_code[i], q = (code >> kBucketBits) - base;
            if (q < 0 || q >= parts) continue;
            const auto w = static_cast<unsigned long long>(vertex_weights[left_vertex[i]]);
            const int b = q * kBalanceWidth + (code & ((1 << kBucketBits) - 1));
            if (narrow) atomicAdd(&sh.u.narrow[b], static_cast<unsigned>(w));
            else atomicAdd(&sh.u.wide[b], w);
        }
        __syncthreads();
        part_boundaries(narrow ? sh.u.narrow : nullptr, sh.u.wide, base, parts, true, sh.pw, capacity, sh.boundary,
                        sh.running);
        __syncthreads();
    }
    unsigned long long edges = 0;
    for (int start = 0; start < count; start += kSelectThreads) {
        const int x = start + t;
        int part = 0, v = 0;
        bool take = false, pending = false;
        if (x < count) {
            const long long i = locate(x);
            const int code = left_code[i], bucket = code & ((1 << kBucketBits) - 1);
            v = left_vertex[i];
            part = code >> kBucketBits;
            take = bucket < sh.boundary[part];
            pending = bucket == sh.boundary[part];
        }
        if (__syncthreads_or(pending)) {
            const unsigned long long w = pending ? static_cast<unsigned long long>(vertex_weights[v]) : 0;
            const unsigned long long rank = block_key_prefix<kSelectThreads>(pending, part, w, sh.wave_total, sh.running);
            if (pending) take = rank + w <= part_limit(sh.pw[part], capacity, true);
        }
        const unsigned long long degree =
            take ? static_cast<unsigned long long>(offsets[v + 1] - offsets[v]) : 0;
        const unsigned long long bh = __ballot(take && degree > kHeavyDegree);
        const unsigned long long bl = __ballot(take && degree <= kHeavyDegree);
        unsigned at_light = 0, at_heavy = 0;
        if (lane == 0) {
            if (bl) at_light = atomicAdd(&sh.light, static_cast<unsigned>(__popcll(bl)));
            if (bh) at_heavy = atomicAdd(&sh.heavy, static_cast<unsigned>(__popcll(bh)));
        }
        at_light = read_lane(at_light, 0);
        at_heavy = read_lane(at_heavy, 0);
        edges += degree;
        if (take) {
            if (degree > kHeavyDegree) heavy[at_heavy + __popcll(bh & lanemask_lt())] = v;
            else light[at_light + __popcll(bl & lanemask_lt())] = v;
            flags[v] = labels[v] + 1;
            mark_mover(state, v, part);
        }
    }
    edges = group_sum_u64<kWave>(edges);
    if (lane == 0 && edges) atomicAdd(&sh.edges, edges);
    __syncthreads();
    if (t == 0) {
        st->light = sh.light;
        st->heavy = sh.heavy;
        st->edges = static_cast<long long>(sh.edges);
    }
}

// ---------------------------------------------------------------- round graphs
//
// A refinement round (an LP round or a rebalance iteration) is a fixed sequence
// of launches for a given level and set of arrays, repeated tens of times per
// level, each followed by a host wait for its status. The first call of a
// sequence captures its launches into hipGraphs; later calls with the same key
// (every pointer, size and setting the launches depend on) replay them, which
// submits a round at once instead of launch by launch (on MI355X 2.0-2.6 us per
// kernel instead of 2.8-4.3 us with a host wait every 20 kernels). The round's
// scratch comes from its plan, whose blocks keep their addresses from call to
// call. A family timed with events runs outside the graphs (events recorded in a
// capture carry no timing), which splits the sequence into segments.
constexpr std::size_t kMaxRoundPlans = 64;
constexpr std::int64_t kMaxGraphVertices = std::int64_t{1} << 23;  // larger levels are not launch-bound

BlockCache* plan_cache(gpart_ctx* ctx) {
    if (!ctx->plan_cache) {
        SegmentSource source;
        source.allocate = [](std::size_t bytes) -> void* {
            void* q = nullptr;
            const hipError_t e = hipMalloc(&q, bytes);
            if (e == hipErrorOutOfMemory) {
                (void)hipGetLastError();
                return nullptr;
            }
            GPART_HIP_CHECK(e);
            return q;
        };
        source.release = [](void* q) { GPART_HIP_CHECK(hipFree(q)); };
        source.drain = [ctx] { GPART_HIP_CHECK(hipStreamSynchronize(ctx->stream)); };
        ctx->plan_cache = std::make_unique<BlockCache>(std::move(source));
    }
    return ctx->plan_cache.get();
}

struct RoundPlan final : ScratchRecorder {
    explicit RoundPlan(gpart_ctx* c, std::vector<std::uint64_t> k) : ctx(c), key(std::move(k)) {}
    ~RoundPlan() override {
        for (auto g : segments) (void)hipGraphExecDestroy(g);
        for (auto& list : blocks)
            for (auto& b : list) ctx->plan_cache->free(b.first);
    }
    void* take(gpart_ctx*, std::size_t bytes) override {
        if (blocks.size() <= static_cast<std::size_t>(phase)) {
            blocks.resize(phase + 1);
            cursor.resize(phase + 1, 0);
        }
        auto& list = blocks[phase];
        std::size_t& at = cursor[phase];
        if (!recorded) {
            void* p = nullptr;
            try {
                p = plan_cache(ctx)->allocate(bytes);
            } catch (const std::runtime_error& e) {
                if (dynamic_cast<const Error*>(&e)) throw;
                throw Error(GPART_ERR_RUNTIME, e.what());
            }
            list.emplace_back(p, bytes);
            owned.insert(p);
            ++at;
            return p;
        }
        if (at >= list.size() || list[at].second != bytes)
            throw Error(GPART_ERR_RUNTIME, "a recorded refinement round asked for different scratch");
        return list[at++].first;
    }
    bool owns(const void* p) const override { return owned.count(p) != 0; }

    gpart_ctx* ctx;
    std::vector<std::uint64_t> key;
    std::vector<std::vector<std::pair<void*, std::size_t>>> blocks;  // per phase; 0: the round's body
    std::vector<std::size_t> cursor;
    std::unordered_set<const void*> owned;
    std::vector<hipGraphExec_t> segments;
    bool recorded = false;  // a first call has captured the segments
    bool broken = false;    // a capture failed: the plan is dropped
    int phase = 0;
    long long calls = 0, captures = 0, replays = 0;
};

struct RoundPlans {
    gpart_ctx* ctx = nullptr;
    std::list<std::unique_ptr<RoundPlan>> plans;  // most recently used first
    long long captures = 0, replays = 0;
    ~RoundPlans() {
        if (ctx && !plans.empty()) (void)hipStreamSynchronize(ctx->stream);
    }
};

RoundPlans& round_plans(gpart_ctx* ctx) {
    if (!ctx->round_plans) {
        auto* set = new RoundPlans;
        set->ctx = ctx;
        ctx->round_plans = std::shared_ptr<void>(set, [](void* q) { delete static_cast<RoundPlans*>(q); });
    }
    return *static_cast<RoundPlans*>(ctx->round_plans.get());
}

// The plan of a round with this key, or nullptr (launch directly) when the
// context does not use round graphs, the level is large, or the key is new: a
// round is recorded on its second call, so a sequence that runs once never pays
// for a capture.
RoundPlan* round_plan(gpart_ctx* ctx, std::int64_t n, std::vector<std::uint64_t> key) {
    if (!ctx->round_graphs || n > kMaxGraphVertices) return nullptr;
    for (int f = 0; f < GPART_PROFILE_FAMILIES; ++f) key.push_back(ctx->profile[f].enabled ? 1 : 0);
    auto& set = round_plans(ctx);
    for (auto it = set.plans.begin(); it != set.plans.end(); ++it) {
        if ((*it)->key != key) continue;
        if ((*it)->broken) {
            set.plans.erase(it);
            break;
        }
        set.plans.splice(set.plans.begin(), set.plans, it);
        RoundPlan* plan = set.plans.front().get();
        return ++plan->calls >= 2 ? plan : nullptr;
    }
    if (set.plans.size() >= kMaxRoundPlans) {
        GPART_HIP_CHECK(hipStreamSynchronize(ctx->stream));  // its graphs may still run
        set.plans.pop_back();
    }
    set.plans.push_front(std::make_unique<RoundPlan>(ctx, std::move(key)));
    set.plans.front()->calls = 1;
    return nullptr;
}

// One call of a round: phases run their launches into the plan's graphs (first
// call) or replay them (later calls). Scratch of the round's body is taken
// before, between or after phases in the same order every call.
class RoundRun {
public:
    RoundRun(gpart_ctx* ctx, RoundPlan* plan) : ctx_(ctx), plan_(plan) {
        if (!plan_) return;
        ctx_->recorder = plan_;
        plan_->phase = 0;
        std::fill(plan_->cursor.begin(), plan_->cursor.end(), 0);
        if (plan_->recorded) {
            ++plan_->replays;
            ++round_plans(ctx_).replays;
        } else {
            ++plan_->captures;
            ++round_plans(ctx_).captures;
        }
    }
    ~RoundRun() {
        if (!plan_) return;
        if (capturing_) {  // an exception left a capture open
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(ctx_->stream, &g);
            if (g) (void)hipGraphDestroy(g);
            plan_->broken = true;
        }
        ctx_->recorder = nullptr;
    }
    RoundRun(const RoundRun&) = delete;
    RoundRun& operator=(const RoundRun&) = delete;

    // The launches of one phase; family >= 0: the profile family they report to
    // (run outside the graphs while that family is timed).
    template <typename F>
    void phase(int family, F&& launches) {
        if (!plan_) {
            launches();
            return;
        }
        plan_->phase = ++phases_;
        if (plan_->cursor.size() > static_cast<std::size_t>(phases_)) plan_->cursor[phases_] = 0;
        const bool direct = family >= 0 && ctx_->profile[family].enabled;
        if (direct) {
            close_segment();
            in_segment_ = false;
            launches();
        } else if (!plan_->recorded) {
            if (!capturing_) {
                GPART_HIP_CHECK(hipStreamBeginCapture(ctx_->stream, hipStreamCaptureModeRelaxed));
                capturing_ = true;
            }
            launches();
        } else if (!in_segment_) {
            if (segment_ >= plan_->segments.size())
                throw Error(GPART_ERR_RUNTIME, "a recorded refinement round has fewer segments than its calls");
            GPART_HIP_CHECK(hipGraphLaunch(plan_->segments[segment_++], ctx_->stream));
            in_segment_ = true;
        }
        plan_->phase = 0;
    }
    // After the last phase.
    void end() {
        if (!plan_) return;
        close_segment();
        plan_->recorded = true;
    }

private:
    // First call: the open capture becomes a segment and runs now.
    void close_segment() {
        if (!capturing_) return;
        hipGraph_t graph = nullptr;
        capturing_ = false;
        GPART_HIP_CHECK(hipStreamEndCapture(ctx_->stream, &graph));
        hipGraphExec_t exec = nullptr;
        const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (e != hipSuccess) {
            plan_->broken = true;
            GPART_HIP_CHECK(e);
        }
        plan_->segments.push_back(exec);
        GPART_HIP_CHECK(hipGraphLaunch(exec, ctx_->stream));
    }

    gpart_ctx* ctx_;
    RoundPlan* plan_;
    int phases_ = 0;
    bool capturing_ = false;
    bool in_segment_ = false;
    std::size_t segment_ = 0;
};

inline std::uint64_t key_of(const void* p) { return reinterpret_cast<std::uintptr_t>(p); }
inline std::uint64_t key_of(double v) {
    std::uint64_t b;
    std::memcpy(&b, &v, sizeof b);
    return b;
}

// ---------------------------------------------------------------- drivers

template <typename O, typename W, typename C = unsigned long long>
struct Ops {
    static void cut(gpart_ctx* ctx, const gpart_csr_view* g, const std::int32_t* labels, std::uint64_t* out) {
        const std::int64_t tiles = g->n > 0 && g->m > 0 ? tile_count(g->m) : 0;
        Scratch<std::int32_t> tile_row(ctx, tiles);
        Scratch<unsigned long long> partials(ctx, std::min<std::int64_t>(tiles, kCutBlocks));
        cut_with(ctx, g, labels, tile_row.get(), partials.get(), out);
    }

    // The cut over caller-provided device scratch: tile_row (tile_count(m) entries) and
    // partials (min(tiles, kCutBlocks) words, folded by one workgroup).
    static void cut_with(gpart_ctx* ctx, const gpart_csr_view* g, const std::int32_t* labels,
                         std::int32_t* tile_row, unsigned long long* partials, std::uint64_t* out) {
        unsigned long long directed = 0;
        const auto* off = static_cast<const O*>(g->offsets);
        const auto* w = static_cast<const W*>(g->edge_weights);
        if (g->n > 0 && g->m > 0) {
            // edge tiles, capped grid
            const std::int64_t tiles = tile_count(g->m);
            hipLaunchKernelGGL(tile_rows_kernel<O>, dim3(grid_for(g->n)), dim3(kBlock), 0, ctx->stream, g->n, off,
                               tile_row);
            const int blocks = static_cast<int>(std::min<std::int64_t>(tiles, kCutBlocks));
            hipLaunchKernelGGL((cut_kernel<O, W>), dim3(blocks), dim3(kTileLanes), 0, ctx->stream, g->n, g->m, tiles,
                               off, tile_row, g->neighbors, w, labels, partials);
            GPART_LAUNCH_CHECK();
            static_assert(kCutBlocks <= kReduceThreads * kReduceLoads, "one workgroup: no scratch");
            reduce_read<SumU64>(ctx, WidenLoad<unsigned long long>{partials}, blocks, &directed);
        }
        if (directed & 1ULL) throw Error(GPART_ERR_RUNTIME, "refinement cut is not symmetric");
        *out = directed / 2;
    }

    // Writes every row of the cache. With a gate, the kernels run only when
    // *gate > above (decided on the device, inside a round); cut, when given,
    // receives the directed cut weight of `labels`.
    static void build_cache(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                            const std::int32_t* labels, int k, C* cache, const long long* gate = nullptr,
                            long long above = 0, unsigned long long* cut = nullptr) {
        const auto* off = static_cast<const O*>(g->offsets);
        const auto* w = static_cast<const W*>(g->edge_weights);
        if (!gate) profile_begin(ctx, GPART_PROFILE_REFINE_CACHE);
        auto grid = [](std::int64_t threads) {
            return static_cast<unsigned>(std::min<std::int64_t>(grid_for(threads), kCacheBlocks));
        };
        if (c->low_count)
            hipLaunchKernelGGL((build_cache_kernel<O, W, 8, C>), dim3(grid(c->low_count * 8)), dim3(kBlock), 0,
                               ctx->stream, c->low_count, c->low, off, g->neighbors, w, labels, k, cache, gate, above,
                               cut);
        if (c->medium_count)
            hipLaunchKernelGGL((build_cache_kernel<O, W, 64, C>), dim3(grid(c->medium_count * 64)), dim3(kBlock), 0,
                               ctx->stream, c->medium_count, c->medium, off, g->neighbors, w, labels, k, cache, gate,
                               above, cut);
        if (c->high_count)
            hipLaunchKernelGGL((build_cache_kernel<O, W, kBlock, C>), dim3(grid(c->high_count * kBlock)),
                               dim3(kBlock), 0, ctx->stream, c->high_count, c->high, off, g->neighbors, w, labels, k,
                               cache, gate, above, cut);
        if (c->max_degree > kHubChunk) {
            HubChunks chunks;
            build_hub_chunks(ctx, off, c->high, c->high_count, c->high_edges, kHubChunk, chunks);
            hipLaunchKernelGGL(hub_rows_zero_kernel<C>, dim3(grid_for(c->high_count)), dim3(kBlock), 0, ctx->stream,
                               c->high_count, chunks.start.get(), c->high, k, cache, gate, above);
            hipLaunchKernelGGL((build_cache_hub_kernel<O, W, C>), dim3(chunks.grid()), dim3(kBlock), 0, ctx->stream,
                               chunks.total(), chunks.start.get(), chunks.hub.get(), c->high, off, g->neighbors, w,
                               labels, k, cache, gate, above, cut);
        }
        GPART_LAUNCH_CHECK();
        if (gate) return;
        const double n = static_cast<double>(g->n), m = static_cast<double>(g->m);
        profile_end(ctx, GPART_PROFILE_REFINE_CACHE,
                    (n + 1) * sizeof(O) + m * (4 + sizeof(W)) + 4 * m + static_cast<double>(sizeof(C)) * n * k);
    }

    // append: the movers also go to the round's lists (levels without hub rows only).
    static void filter_movers(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                              const std::int32_t* labels, const std::int32_t* targets, const long long* gains,
                              std::int32_t* flags, bool append, std::int32_t* light, std::int32_t* heavy,
                              RoundState* st, const gpart_refine_rows* rows) {
        const auto* off = static_cast<const O*>(g->offsets);
        const auto* w = static_cast<const W*>(g->edge_weights);
        profile_begin(ctx, GPART_PROFILE_REFINE_FILTER);
        const unsigned low_blocks = grid_for(c->low_count * 8), medium_blocks = grid_for(c->medium_count * 64);
        const auto high_blocks = static_cast<unsigned>(c->high_count);
        const unsigned blocks = low_blocks + medium_blocks + high_blocks;
        unsigned char* state = rows ? rows->states.get() : nullptr;
        if (blocks > 0 && append)
            hipLaunchKernelGGL((priority_filter_kernel<O, W, true>), dim3(blocks), dim3(kBlock), 0, ctx->stream,
                               c->low_count, c->low, low_blocks, c->medium_count, c->medium, medium_blocks,
                               c->high_count, c->high, off, g->neighbors, w, labels, targets, gains, flags, state, light,
                               heavy, st);
        else if (blocks > 0)
            hipLaunchKernelGGL((priority_filter_kernel<O, W, false>), dim3(blocks), dim3(kBlock), 0, ctx->stream,
                               c->low_count, c->low, low_blocks, c->medium_count, c->medium, medium_blocks,
                               c->high_count, c->high, off, g->neighbors, w, labels, targets, gains, flags, state, light,
                               heavy, st);
        if (c->max_degree > kHubChunk) {
            HubChunks own;
            if (!rows) build_hub_chunks(ctx, off, c->high, c->high_count, c->high_edges, kHubChunk, own);
            const HubChunks& chunks = rows ? rows->chunks : own;
            Scratch<long long> sums(ctx, c->high_count);
            fill_bytes(ctx, sums.get(), 0, static_cast<std::size_t>(c->high_count) * 8);
            hipLaunchKernelGGL((priority_filter_hub_kernel<O, W>), dim3(chunks.grid()), dim3(kBlock), 0, ctx->stream,
                               chunks.total(), chunks.start.get(), chunks.hub.get(), c->high, off, g->neighbors, w,
                               labels, targets, gains, sums.get());
            hipLaunchKernelGGL(priority_filter_hub_finish_kernel, dim3(grid_for(c->high_count)), dim3(kBlock), 0,
                               ctx->stream, c->high_count, chunks.start.get(), c->high, labels, targets, gains,
                               sums.get(), flags, state);
        }
        GPART_LAUNCH_CHECK();
        const double nd = static_cast<double>(g->n), m = static_cast<double>(g->m);
        profile_end(ctx, GPART_PROFILE_REFINE_FILTER, (nd + 1) * sizeof(O) + m * (4 + sizeof(W)) + 16 * m + 20 * nd);
    }

    static RowLists row_lists(const gpart_degree_classes* c, const gpart_refine_rows* r) {
        RowLists l{};
        l.low = c->low;
        l.medium = c->medium;
        l.high = c->high;
        l.low_count = c->low_count;
        l.medium_count = c->medium_count;
        l.high_count = c->high_count;
        if (r->hubs) {
            l.chunk_total = r->chunks.total();
            l.chunk_start = r->chunks.start.get();
            l.chunk_hub = r->chunks.hub.get();
        }
        return l;
    }
    // Workgroups of a pass over about `entries` entries: 256 entries a wave, at least
    // a few workgroups so that a small level's rows spread over some CUs.
    static unsigned rows_groups(std::int64_t entries, std::size_t lds) {
        const std::int64_t per = std::int64_t{256} * kRowsWaves;
        return static_cast<unsigned>(std::clamp<std::int64_t>((entries + per - 1) / per, 16,
                                                              lds <= kRowsPairLds ? 2 * kRowsGroups : kRowsGroups));
    }

    // Before a round; the round that completes leaves the handle ready.
    static void prepare_rows(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                             gpart_refine_rows* r, const std::int32_t* labels, int k, C* cache) {
        if (!r->ready) launch_prepare(ctx, g, c, r, labels, r->states.get(), k, cache);
        r->ready = false;
    }
    static void launch_prepare(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                               const gpart_refine_rows* r, const std::int32_t* labels, unsigned char* states, int k,
                               C* cache) {
        if constexpr (sizeof(C) == 4) {
            hipLaunchKernelGGL(rows_prepare_kernel, dim3(std::min<unsigned>(grid_for(g->n), kRoundBlocks)), dim3(256), 0,
                               ctx->stream, row_lists(c, r), g->n, labels, states, k, cache);
            GPART_LAUNCH_CHECK();
        }
    }

    // The entries in which the rows that the next round will sum, from the states and over
    // the hub rows as the last one left them, differ from the expected ones.
    static std::int64_t check_rows(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                                   const gpart_refine_rows* r, const std::int32_t* labels, int k, C* cache,
                                   const unsigned long long* part_weights, std::uint64_t capacity,
                                   const unsigned* expected) {
        unsigned long long differing = 0;
        if constexpr (sizeof(C) == 4) {
            rows(ctx, g, c, r, k, cache, part_weights, capacity);
            reduce_read<SumU64>(ctx, RowsDiffer{cache, expected, labels, part_weights, capacity, k}, g->n * k,
                                &differing);
            launch_prepare(ctx, g, c, r, labels, nullptr, k, cache);
        }
        return static_cast<std::int64_t>(differing);
    }

    // The rows of every vertex, or (part_weights) of the parts above capacity.
    static void rows(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                     const gpart_refine_rows* r, int k, C* cache, const unsigned long long* part_weights,
                     std::uint64_t capacity) {
        if constexpr (sizeof(C) == 4) {
            profile_begin(ctx, GPART_PROFILE_REFINE_CACHE);
            const std::size_t lds = kRowsWaveBytes + state_lds_bytes(g->n, r->form);
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(rows_groups(g->m, lds)), dim3(kRowsThreads), lds, ctx->stream,
                                   row_lists(c, r), r->states.get(), g->n, static_cast<const O*>(g->offsets),
                                   g->neighbors, static_cast<const W*>(g->edge_weights), k, cache, part_weights,
                                   capacity);
            };
            if (r->form == kByteState) launch(rows_kernel<O, W, kByteState>);
            else if (r->form == kNibbleState) launch(rows_kernel<O, W, kNibbleState>);
            else launch(rows_kernel<O, W, kMemoryState>);
            GPART_LAUNCH_CHECK();
            const double n = static_cast<double>(g->n), m = static_cast<double>(g->m);
            profile_end(ctx, GPART_PROFILE_REFINE_CACHE,
                        part_weights ? 0.0 : (n + 1) * sizeof(O) + m * (4 + sizeof(W)) + n + 4 * n * k);
        }
    }

    // gain_commit_kernel over the round's movers.
    static void apply_rows(gpart_ctx* ctx, RoundRun& run, const gpart_csr_view* g, const gpart_degree_classes* c,
                           const gpart_refine_rows* r, RoundState* st, const std::int32_t* light,
                           const std::int32_t* heavy, std::int32_t* labels, const std::int32_t* targets,
                           const std::int32_t* flags, int k, C* cache, unsigned long long* part_weights,
                           std::int32_t* locks) {
        if constexpr (sizeof(C) == 4) {
            run.phase(GPART_PROFILE_CACHE_UPDATE, [&] {
                profile_begin(ctx, GPART_PROFILE_CACHE_UPDATE);
                const std::size_t lds = state_lds_bytes(g->n, r->form);
                auto launch = [&](auto kernel) {
                    // a tenth of the entries move in a round of a dense level
                    hipLaunchKernelGGL(kernel, dim3(rows_groups(g->m / 8, lds)), dim3(kRowsThreads), lds, ctx->stream,
                                       st, light, heavy, row_lists(c, r), r->states.get(), g->n, static_cast<const O*>(g->offsets), g->neighbors,
                                       static_cast<const W*>(g->edge_weights),
                                       static_cast<const W*>(g->vertex_weights), labels, targets, flags, locks, k,
                                       cache, part_weights, reinterpret_cast<unsigned long long*>(ctx->status_device),
                                       ctx->status_counter);
                };
                if (r->form == kByteState) launch(gain_commit_kernel<O, W, kByteState>);
                else if (r->form == kNibbleState) launch(gain_commit_kernel<O, W, kNibbleState>);
                else launch(gain_commit_kernel<O, W, kMemoryState>);
                GPART_LAUNCH_CHECK();
                profile_end(ctx, GPART_PROFILE_CACHE_UPDATE, 0.0);
            });
        }
    }

    // incremental_update_cache_and_cut + incremental_commit over the round's movers.
    // On levels of at least ctx->rebuild_min_entries entries the device chooses,
    // from the round's mover entries, between atomic updates (two per mover entry)
    // and a full rebuild of the cache after the commit (one gather per entry, no
    // atomics, same cache); the cut delta is summed from the movers' entries
    // either way. Ends with the round's status: published by the update launch where
    // that is the round's last, else by a launch of its own.
    static void apply(gpart_ctx* ctx, RoundRun& run, const gpart_csr_view* g, const gpart_degree_classes* c,
                      RoundState* st, const std::int32_t* light, const std::int32_t* heavy, std::int32_t* labels,
                      const std::int32_t* targets, const std::int32_t* flags, int k, C* cache,
                      unsigned long long* part_weights, std::int32_t* locks) {
        const std::int64_t n = g->n;
        const auto* off = static_cast<const O*>(g->offsets);
        const auto* w = static_cast<const W*>(g->edge_weights);
        const auto* vw = static_cast<const W*>(g->vertex_weights);
        const long long rebuild_above = rebuild_threshold(ctx, g);
        // levels whose degrees stay at most kWaveHeavyMaxDegree update their heavy
        // movers a wave each, in the same launch
        const bool wave_heavy = c->max_degree > kHeavyDegree && c->max_degree <= kWaveHeavyMaxDegree;
        const bool tiles = c->max_degree > kWaveHeavyMaxDegree;
        const bool ends_round = !tiles && rebuild_above < 0;
        auto* status = reinterpret_cast<unsigned long long*>(ctx->status_device);
        const std::int64_t heavy_bound = c->medium_count + c->high_count;
        // a launch that ends the round keeps the arrivals at its counter few
        const std::int64_t cap = ends_round ? kRoundBlocks : 4 * kRoundBlocks;
        const auto light_blocks = static_cast<unsigned>(std::min<std::int64_t>(grid_for(n * 8), cap));
        const unsigned heavy_blocks =
            wave_heavy ? static_cast<unsigned>(
                             std::max<std::int64_t>(1, std::min<std::int64_t>(grid_for(heavy_bound * kWave), cap)))
                       : 0;
        run.phase(GPART_PROFILE_CACHE_UPDATE, [&] {
        profile_begin(ctx, GPART_PROFILE_CACHE_UPDATE);
        hipLaunchKernelGGL((update_cache_kernel<O, W, C>), dim3(light_blocks + heavy_blocks), dim3(kBlock), 0,
                           ctx->stream, st, light, heavy, light_blocks, heavy_blocks, off, g->neighbors, w, vw,
                           labels, targets, flags, locks, k, cache, part_weights, rebuild_above,
                           ends_round ? status : nullptr, ctx->status_counter);
        if (tiles) {
            Scratch<long long> heavy_start(ctx, heavy_bound + 1);
            Scratch<std::int32_t> tile_mover(ctx, tile_count(g->m) + 1);
            device_scan<long long, SumOp<long long>>(ctx, HeavyDegreeLoad<O>{st, heavy, off},
                                                     ExclusiveStore<long long>{heavy_start.get()}, heavy_bound + 1,
                                                     SumOp<long long>{});
            hipLaunchKernelGGL(heavy_tiles_kernel,
                               dim3(static_cast<unsigned>(std::min<std::int64_t>(grid_for(heavy_bound), kRoundBlocks))),
                               dim3(kBlock), 0, ctx->stream, st, heavy_start.get(), tile_mover.get());
            const auto blocks = static_cast<unsigned>(std::max<std::int64_t>(
                1, std::min<std::int64_t>(tile_count(g->m), 2 * kRoundBlocks)));
            hipLaunchKernelGGL((update_cache_tiles_kernel<O, W, C>), dim3(blocks), dim3(kTileLanes), 0, ctx->stream,
                               st, heavy_start.get(), tile_mover.get(), heavy, off, g->neighbors, w, labels, targets,
                               flags, k, cache, &st->delta, rebuild_above);
        }
        GPART_LAUNCH_CHECK();
        profile_end(ctx, GPART_PROFILE_CACHE_UPDATE, 0.0);
        });
        if (ends_round) return;
        run.phase(-1, [&] {
            if (rebuild_above >= 0)
                build_cache(ctx, g, c, labels, k, cache, &st->edges, rebuild_above, &st->cut_directed);
            hipLaunchKernelGGL(round_status_kernel, dim3(1), dim3(kWave), 0, ctx->stream, st, part_weights, k, status,
                               ctx->status_counter);
            GPART_LAUNCH_CHECK();
        });
    }

    // Mover entries above which a round rebuilds the cache; -1: never.
    static long long rebuild_threshold(const gpart_ctx* ctx, const gpart_csr_view* g) {
        return ctx->rebuild_share > 0 && g->m >= ctx->rebuild_min_entries ? g->m / ctx->rebuild_share : -1;
    }

    // The host's wait for the status that apply's last launch publishes, and its
    // reading.
    // False: a rebalance iteration refused (kRefusedShare) and left everything as it was.
    static bool finish(gpart_ctx* ctx, RoundRun& run, const gpart_csr_view* g, int k, bool rows_form,
                       gpart_refine_status* out) {
        run.end();
        const std::uint64_t seq = ++ctx->status_seq;
        wait_status(ctx, seq);
        RoundState h{};
        std::memcpy(&h, ctx->status_host + 1, offsetof(RoundState, pw) + 8 * static_cast<std::size_t>(k));
        out->movers = h.light + h.heavy;
        out->cut_delta = h.delta;
        out->candidates = h.candidates;
        out->max_part_weight = h.max_weight;
        for (int p = 0; p < 32; ++p) ctx->round_part_weights[p] = out->part_weights[p] = p < k ? h.pw[p] : 0;
        out->mover_entries = h.edges;
        const long long rebuild_above = rows_form ? -1 : rebuild_threshold(ctx, g);
        out->rebuilt = rebuild_above >= 0 && h.edges > rebuild_above ? 1 : 0;
        out->cut_after = 0;
        if (rows_form) {
            // the movers' rows and ids, per entry a neighbour, a weight and the label,
            // target and flag gathers
            profile_add_bytes(ctx, GPART_PROFILE_CACHE_UPDATE,
                              static_cast<double>(out->movers) * (2.0 * sizeof(O) + 16.0) +
                                  static_cast<double>(h.edges) * (4.0 + sizeof(W) + 12.0));
        } else if (!out->rebuilt) {
            // the movers' rows and ids, per entry a neighbour, a weight, two cache
            // atomics (read and write each) and the label, target and flag gathers
            const double movers = static_cast<double>(out->movers), entries = static_cast<double>(h.edges);
            profile_add_bytes(ctx, GPART_PROFILE_CACHE_UPDATE,
                              movers * (2.0 * sizeof(O) + 16.0) + entries * (4.0 + sizeof(W) + 4.0 * sizeof(C) + 12.0));
            profile_add_units(ctx, GPART_PROFILE_CACHE_UPDATE, 2.0 * entries);
        }
        if (out->rebuilt) {
            if (h.cut_directed & 1ULL) throw Error(GPART_ERR_RUNTIME, "refinement cut is not symmetric");
            out->cut_after = h.cut_directed / 2;
            out->cut_delta = 0;
        }
        return h.refused == 0;
    }

    // One LP round: proposals, priority filter, movers, apply; one synchronisation.
    static void lp_round(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                         C* cache, std::int32_t* labels, int k, double filter,
                         std::int32_t* locks, std::int32_t* targets, long long* gains, std::int32_t* flags,
                         unsigned long long* part_weights, const gpart_refine_rows* r, gpart_refine_status* out) {
        const std::int64_t n = g->n;
        const auto* off = static_cast<const O*>(g->offsets);
        RoundRun run(ctx, round_plan(ctx, n, round_key(ctx, g, c, cache, labels, k, targets, flags, part_weights, r,
                                                       {0, key_of(filter), key_of(locks), key_of(gains)})));
        // the proposals kernel zeroes the round state
        Scratch<RoundState> st(ctx, 1);
        Scratch<std::int32_t> light(ctx, n), heavy(ctx, n);
        const int G = group_for_k(k);
        unsigned char* state = r ? r->states.get() : nullptr;
        if (r) run.phase(GPART_PROFILE_REFINE_CACHE, [&] { rows(ctx, g, c, r, k, cache, nullptr, 0); });
        run.phase(GPART_PROFILE_REFINE_PROPOSALS, [&] {
            profile_begin(ctx, GPART_PROFILE_REFINE_PROPOSALS);
            const unsigned blocks = std::max<unsigned>(1, grid_for(n * G));
            switch (G) {
                case 1: hipLaunchKernelGGL((lp_proposals_kernel<1, C>), dim3(blocks), dim3(kBlock), 0, ctx->stream, n, cache, labels, k, filter, locks, targets, gains, state, st.get()); break;
                case 2: hipLaunchKernelGGL((lp_proposals_kernel<2, C>), dim3(blocks), dim3(kBlock), 0, ctx->stream, n, cache, labels, k, filter, locks, targets, gains, state, st.get()); break;
                default: hipLaunchKernelGGL((lp_proposals_kernel<4, C>), dim3(blocks), dim3(kBlock), 0, ctx->stream, n, cache, labels, k, filter, locks, targets, gains, state, st.get()); break;
            }
            GPART_LAUNCH_CHECK();
            profile_end(ctx, GPART_PROFILE_REFINE_PROPOSALS, static_cast<double>(n) * (20.0 + sizeof(C) * k));
        });
        // Small levels list their movers in the filter launch; on large ones its
        // thousands of workgroups would contend for the list counters (128^3 mesh
        // uncoarsening 43 -> 49 ms), so their movers come from a scan of the flags.
        const bool append = n <= kSelectVertices && c->max_degree <= kHubChunk;
        run.phase(GPART_PROFILE_REFINE_FILTER, [&] {
            filter_movers(ctx, g, c, labels, targets, gains, flags, append, light.get(), heavy.get(), st.get(), r);
        });
        if (!append)
            run.phase(-1, [&] {
                device_scan<MoverPair, MoverPairOp>(ctx, MoverLoad<O>{flags, off},
                                                    MoverStore{light.get(), heavy.get(), n, st.get()}, n,
                                                    MoverPairOp{});
            });
        if (r)
            apply_rows(ctx, run, g, c, r, st.get(), light.get(), heavy.get(), labels, targets, flags, k, cache,
                       part_weights, locks);
        else
            apply(ctx, run, g, c, st.get(), light.get(), heavy.get(), labels, targets, flags, k, cache, part_weights,
                  locks);
        finish(ctx, run, g, k, r != nullptr, out);
    }

    // Everything a round's launches depend on besides its own scratch.
    static std::vector<std::uint64_t> round_key(const gpart_ctx* ctx, const gpart_csr_view* g,
                                                const gpart_degree_classes* c, const C* cache,
                                                const std::int32_t* labels, int k, const std::int32_t* targets,
                                                const std::int32_t* flags, const unsigned long long* part_weights,
                                                const gpart_refine_rows* r,
                                                std::initializer_list<std::uint64_t> extra) {
        std::vector<std::uint64_t> key{sizeof(O), sizeof(C), static_cast<std::uint64_t>(g->n),
                                       static_cast<std::uint64_t>(g->m), key_of(g->offsets), key_of(g->neighbors),
                                       key_of(g->edge_weights), key_of(g->vertex_weights), key_of(c->low),
                                       key_of(c->medium), key_of(c->high), static_cast<std::uint64_t>(c->low_count),
                                       static_cast<std::uint64_t>(c->medium_count),
                                       static_cast<std::uint64_t>(c->high_count),
                                       static_cast<std::uint64_t>(c->high_edges),
                                       static_cast<std::uint64_t>(c->max_degree), key_of(cache), key_of(labels),
                                       static_cast<std::uint64_t>(k), key_of(targets), key_of(flags),
                                       key_of(part_weights), static_cast<std::uint64_t>(rebuild_threshold(ctx, g)),
                                       key_of(ctx->status_device), key_of(ctx->status_counter),
                                       r ? key_of(r->states.get()) : 0, r ? static_cast<std::uint64_t>(r->form) : 0,
                                       r && r->hubs ? key_of(r->chunks.start.get()) : 0,
                                       r && r->hubs ? key_of(r->chunks.hub.get()) : 0};
        key.insert(key.end(), extra.begin(), extra.end());
        return key;
    }

    // Calls launch(lanes per row, a value of balance_choice's U): 32 bits when 4-byte
    // cache entries and k parts of the capacity fit them.
    template <typename Launch>
    static void choose(int k, std::uint64_t capacity, Launch&& launch) {
        auto with = [&](auto slack) {
            switch (group_for_k(k)) {
                case 1: launch(std::integral_constant<int, 1>{}, slack); break;
                case 2: launch(std::integral_constant<int, 2>{}, slack); break;
                default: launch(std::integral_constant<int, 4>{}, slack); break;
            }
        };
        if constexpr (sizeof(C) == 4) {
            if (capacity <= 0xffffffffULL / static_cast<unsigned>(k)) return with(unsigned{0});
        }
        with(0ULL);
    }

    // About how many vertices leave their parts in the next rebalance iteration, from the
    // part weights of the context's last round (a wrong guess costs time only).
    static std::int64_t expected_leaving(const gpart_ctx* ctx, std::int64_t n, int k, std::uint64_t capacity) {
        double overload = 0, total = 0;
        for (int p = 0; p < k; ++p) {
            const auto w = ctx->round_part_weights[p];
            total += static_cast<double>(w);
            if (w > capacity) overload += static_cast<double>(w - capacity);
        }
        return total > 0 ? static_cast<std::int64_t>(overload / total * static_cast<double>(n)) : 0;
    }

    // A rebalance iteration of a small level (balance_vertices_kernel,
    // balance_select_kernel, update).
    static void rebalance_round_small(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                                      C* cache, std::int32_t* labels, int k, unsigned long long* part_weights,
                                      std::uint64_t capacity, std::int32_t* targets, std::int32_t* flags,
                                      const PowerTable& powers, const gpart_refine_rows* r,
                                      gpart_refine_status* out) {
        const std::int64_t n = g->n;
        const auto* off = static_cast<const O*>(g->offsets);
        const auto* vw = static_cast<const W*>(g->vertex_weights);
        RoundRun run(ctx, round_plan(ctx, n, round_key(ctx, g, c, cache, labels, k, targets, flags, part_weights, r,
                                                       {2, capacity})));
        Scratch<RoundState> st(ctx, 1);
        Scratch<std::int32_t> choices(ctx, n), light(ctx, n), heavy(ctx, n);
        unsigned char* state = r ? r->states.get() : nullptr;
        if (r)
            run.phase(GPART_PROFILE_REFINE_CACHE,
                      [&] { rows(ctx, g, c, r, k, cache, part_weights, capacity); });
        run.phase(GPART_PROFILE_REBALANCE, [&] {
            profile_begin(ctx, GPART_PROFILE_REBALANCE);
            choose(k, capacity, [&](auto group, auto slack) {
                constexpr int kG = decltype(group)::value;
                using U = decltype(slack);
                hipLaunchKernelGGL((balance_vertices_kernel<W, kG, U, C>), dim3(grid_for(n * kG)), dim3(kBlock), 0,
                                   ctx->stream, st.get(), n, cache, labels, vw, k, part_weights, capacity, powers, targets,
                                   choices.get(), flags, state);
            });
            GPART_LAUNCH_CHECK();
            profile_end(ctx, GPART_PROFILE_REBALANCE, 0.0);
        });
        run.phase(-1, [&] {
#define GPART_BALANCE_SELECT(ITEMS)                                                                              \
    hipLaunchKernelGGL((balance_select_kernel<O, W, ITEMS>), dim3(1), dim3(kSelectThreads), 0, ctx->stream,      \
                       st.get(), n, choices.get(), vw, off, k, part_weights, capacity, light.get(), heavy.get(), \
                       flags, state)
            if (n <= kSelectThreads) GPART_BALANCE_SELECT(1);
            else if (n <= 4 * kSelectThreads) GPART_BALANCE_SELECT(4);
            else GPART_BALANCE_SELECT(kSelectMaxItems);
#undef GPART_BALANCE_SELECT
            GPART_LAUNCH_CHECK();
        });
        if (r)
            apply_rows(ctx, run, g, c, r, st.get(), light.get(), heavy.get(), labels, targets, flags, k, cache,
                       part_weights, nullptr);
        else
            apply(ctx, run, g, c, st.get(), light.get(), heavy.get(), labels, targets, flags, k, cache, part_weights,
                  nullptr);
        finish(ctx, run, g, k, r != nullptr, out);
    }

    // One rebalance iteration: proposals, source and destination bucket quotas,
    // apply; one synchronisation.
    static void rebalance_round(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                                C* cache, std::int32_t* labels, int k,
                                unsigned long long* part_weights, std::uint64_t capacity, std::int32_t* targets,
                                std::int32_t* flags, const gpart_refine_rows* r, gpart_refine_status* out) {
        static const PowerTable powers = make_power_table();
        if (g->n <= kSelectVertices)
            rebalance_round_small(ctx, g, c, cache, labels, k, part_weights, capacity, targets, flags, powers, r,
                                  out);
        else {
            const bool few = expected_leaving(ctx, g->n, k, capacity) <= ctx->few_leaving;
            ++(few ? ctx->single_selections : ctx->slice_selections);
            if (!rebalance_round_large(ctx, g, c, cache, labels, k, part_weights, capacity, targets, flags, powers,
                                       r, few, out)) {
                ++ctx->refused_selections;
                rebalance_round_large(ctx, g, c, cache, labels, k, part_weights, capacity, targets, flags, powers, r,
                                      false, out);
            }
        }
        // per candidate: id, label, weight, cache row, target and bucket writes
        profile_add_bytes(ctx, GPART_PROFILE_REBALANCE,
                          static_cast<double>(out->candidates) * (16.0 + sizeof(W) + sizeof(C) * k));
        // one bucket-histogram add per candidate (balance_source_histogram, :173-186)
        profile_add_units(ctx, GPART_PROFILE_REBALANCE, static_cast<double>(out->candidates));
    }

    // few: one workgroup selects the destinations, or refuses (returns false).
    static bool rebalance_round_large(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* c,
                                      C* cache, std::int32_t* labels, int k, unsigned long long* part_weights,
                                      std::uint64_t capacity, std::int32_t* targets, std::int32_t* flags,
                                      const PowerTable& powers, const gpart_refine_rows* r, bool few,
                                      gpart_refine_status* out) {
        const std::int64_t n = g->n;
        const auto* off = static_cast<const O*>(g->offsets);
        const auto* vw = static_cast<const W*>(g->vertex_weights);
        const std::int64_t width = static_cast<std::int64_t>(k) * kBalanceWidth;
        // Both replica arrays live in the context between rounds and are zero at rest (the
        // boundary search clears what it reads); the proposals kernel zeroes the round
        // state after the candidate count.
        const std::size_t counter_bytes = static_cast<std::size_t>(2 * kReplicas * width) * 8;
        if (ctx->rebalance_counter_bytes < counter_bytes) {
            if (ctx->rebalance_counters) ctx_free(ctx, ctx->rebalance_counters);
            ctx->rebalance_counters = nullptr;
            ctx->rebalance_counter_bytes = 0;
            ctx->rebalance_counters = ctx_alloc(ctx, counter_bytes);
            ctx->rebalance_counter_bytes = counter_bytes;
            ctx->rebalance_counters_zero = false;
        }
        if (!ctx->rebalance_counters_zero) fill_bytes(ctx, ctx->rebalance_counters, 0, ctx->rebalance_counter_bytes);
        ctx->rebalance_counters_zero = false;  // until this round completes
        const std::int64_t most = kRefusedShare * ctx->few_leaving;
        RoundRun run(ctx, round_plan(ctx, n, round_key(ctx, g, c, cache, labels, k, targets, flags, part_weights, r,
                                                       {1, capacity, few, static_cast<std::uint64_t>(most),
                                                        key_of(ctx->rebalance_counters)})));
        Scratch<RoundState> st(ctx, 1);
        auto* st_ptr = st.get();
        auto* replicas = static_cast<unsigned long long*>(ctx->rebalance_counters);
        unsigned long long* destination_replicas = replicas + kReplicas * width;
        Scratch<std::int32_t> cand(ctx, n), cbucket(ctx, n), leaving(ctx, n), left_vertex(ctx, n), left_code(ctx, n),
            light(ctx, n), heavy(ctx, n), left_count(ctx, kSliceBlocks), tile_counts(ctx, kCandidateTiles);
        const int slices =
            static_cast<int>(std::min<std::int64_t>((n + kSliceThreads - 1) / kSliceThreads, kSliceBlocks));
        Scratch<unsigned long long> sums(ctx, std::int64_t{kSliceBlocks} * 32), before(ctx, 32);
        Scratch<int> boundary(ctx, 32);
        unsigned char* state = r ? r->states.get() : nullptr;

        run.phase(-1, [&] {
            auto listed = [&](auto items) {
                constexpr int kItems = decltype(items)::value;
                const auto tiles = static_cast<unsigned>((n + kBlock * kItems - 1) / (kBlock * kItems));
                hipLaunchKernelGGL(candidate_count_kernel<kItems>, dim3(tiles), dim3(kBlock), 0, ctx->stream, n, labels,
                                   part_weights, k, capacity, tile_counts.get());
                hipLaunchKernelGGL(candidate_list_kernel<kItems>, dim3(tiles), dim3(kBlock), 0, ctx->stream, st_ptr, n,
                                   labels, part_weights, k, capacity, tile_counts.get(), cand.get(), flags, state);
                GPART_LAUNCH_CHECK();
            };
            if (n <= kCandidateTiles * kBlock * 8)
                listed(std::integral_constant<int, 8>{});
            else if (n <= kCandidateTiles * kBlock * 32)
                listed(std::integral_constant<int, 32>{});
            else
                device_scan<int, SumOp<int>>(ctx, OverloadedLoad{labels, part_weights, capacity},
                                             CandidateStore{cand.get(), flags, labels, state, n, st_ptr}, n,
                                             SumOp<int>{});
        });
        const auto blocks = static_cast<unsigned>(std::min<std::int64_t>(grid_for(n * group_for_k(k)), ctx->balance_blocks));
        if (r)
            run.phase(GPART_PROFILE_REFINE_CACHE,
                      [&] { rows(ctx, g, c, r, k, cache, part_weights, capacity); });
        run.phase(GPART_PROFILE_REBALANCE, [&] {
            profile_begin(ctx, GPART_PROFILE_REBALANCE);
            choose(k, capacity, [&](auto group, auto slack) {
                constexpr int kG = decltype(group)::value;
                using U = decltype(slack);
                hipLaunchKernelGGL((balance_proposals_kernel<W, kG, U, C>), dim3(blocks), dim3(kBlock), 0, ctx->stream,
                                   st_ptr, cand.get(), cache, labels, vw, k, part_weights, capacity, powers, targets,
                                   cbucket.get(), replicas);
            });
            GPART_LAUNCH_CHECK();
            profile_end(ctx, GPART_PROFILE_REBALANCE, 0.0);
        });
        run.phase(-1, [&] {
            hipLaunchKernelGGL(bucket_boundaries_kernel<false>, dim3(k), dim3(kBucketScanThreads), 0, ctx->stream, replicas, k,
                               part_weights, capacity, boundary.get(), before.get());
            hipLaunchKernelGGL(balance_sources_kernel<W>, dim3(slices), dim3(kSliceThreads), 0, ctx->stream, st_ptr,
                               cand.get(), cbucket.get(), leaving.get(), targets, vw, boundary.get(), sums.get());
            auto ranks = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(slices), dim3(kSliceThreads), 0, ctx->stream, st_ptr, cand.get(),
                                   cbucket.get(), leaving.get(), targets, vw, part_weights, k, capacity, before.get(),
                                   sums.get(), left_vertex.get(), left_code.get(), left_count.get(),
                                   destination_replicas);
            };
            if (few) {
                ranks(balance_source_ranks_kernel<W, false>);
                hipLaunchKernelGGL((balance_destinations_kernel<O, W>), dim3(1), dim3(kSelectThreads), 0, ctx->stream,
                                   st_ptr, slices, left_vertex.get(), left_code.get(), left_count.get(), labels, vw, off,
                                   k, part_weights, capacity, most, light.get(), heavy.get(), flags, state);
            } else {
                ranks(balance_source_ranks_kernel<W, true>);
                hipLaunchKernelGGL(bucket_boundaries_kernel<true>, dim3(k), dim3(kBucketScanThreads), 0, ctx->stream,
                                   destination_replicas, k, part_weights, capacity, boundary.get(), before.get());
                auto slice = [&](auto kernel) {
                    hipLaunchKernelGGL(kernel, dim3(slices), dim3(kSliceThreads), 0, ctx->stream, st_ptr,
                                       left_vertex.get(), left_code.get(), left_count.get(), labels, vw, off, k,
                                       part_weights, capacity, boundary.get(), before.get(), sums.get(), light.get(),
                                       heavy.get(), flags, state);
                };
                slice(balance_slices_kernel<O, W, false>);
                slice(balance_slices_kernel<O, W, true>);
            }
            GPART_LAUNCH_CHECK();
        });
        if (r)
            apply_rows(ctx, run, g, c, r, st_ptr, light.get(), heavy.get(), labels, targets, flags, k, cache,
                       part_weights, nullptr);
        else
            apply(ctx, run, g, c, st_ptr, light.get(), heavy.get(), labels, targets, flags, k, cache, part_weights,
                  nullptr);
        const bool done = finish(ctx, run, g, k, r != nullptr, out);
        ctx->rebalance_counters_zero = true;
        return done;
    }
};

}  // namespace
}  // namespace gpart_hip

// Device scratch of gpart_cut_noalloc, one copy per GPU for the life of the
// process: the directed total, the per-workgroup partials and the tile rows.
// Host code never passes this name to a kernel; it passes the device address
// that cut_scratch_setup looks up for each device.
namespace gpart_hip {
namespace {
constexpr std::int64_t kCutScratchTiles = std::int64_t{1} << 20;  // CSRs up to 2^20 * 4096 entries
constexpr std::size_t kCutScratchPartialsOffset = 0;
constexpr std::size_t kCutScratchTilesOffset = kCutScratchPartialsOffset + 8 * kCutBlocks;
constexpr std::size_t kCutScratchBytes = kCutScratchTilesOffset + 4 * kCutScratchTiles;  // 4 MiB + 8 KiB
constexpr int kCutScratchDevices = 64;

std::mutex& cut_scratch_mutex() {
    static std::mutex mutex;
    return mutex;
}
void* cut_scratch_address[kCutScratchDevices] = {};
}  // namespace
}  // namespace gpart_hip

static __device__ __align__(256) unsigned char scratch[gpart_hip::kCutScratchBytes];

namespace gpart_hip {
// Called once per context with its device current (gpart_ctx_create); the first
// call on a device resolves that device's copy of the array.
void cut_scratch_setup(int device) {
    if (device < 0 || device >= kCutScratchDevices)
        throw Error(GPART_ERR_RUNTIME, "device ordinal beyond the no-allocation scratch table");
    std::lock_guard<std::mutex> lock(cut_scratch_mutex());
    if (cut_scratch_address[device]) return;
    void* address = nullptr;
    GPART_HIP_CHECK(hipGetSymbolAddress(&address, HIP_SYMBOL(scratch)));
    cut_scratch_address[device] = address;
}
}  // namespace gpart_hip

using namespace gpart_hip;

#define GPART_WIDTH_DISPATCH(width, call)                            \
    do {                                                             \
        if ((width) == GPART_WIDTH_STANDARD) {                        \
            using OpsT = Ops<std::int32_t, std::uint32_t>;           \
            call;                                                    \
        } else {                                                     \
            using OpsT = Ops<std::int64_t, std::uint64_t>;           \
            call;                                                    \
        }                                                            \
    } while (0)

// Width of the entry points without an incremental cache (4-byte rows).
#define GPART_ROWS_DISPATCH(width, call)                                       \
    do {                                                                       \
        if ((width) == GPART_WIDTH_STANDARD) {                                  \
            using OpsT = Ops<std::int32_t, std::uint32_t, unsigned>;           \
            call;                                                              \
        } else {                                                               \
            using OpsT = Ops<std::int64_t, std::uint64_t, unsigned>;           \
            call;                                                              \
        }                                                                      \
    } while (0)

// Width and cache entry type (4 or 8 bytes) of the refinement entry points.
#define GPART_CACHE_DISPATCH(width, bytes, call)                                                      \
    do {                                                                                              \
        if ((bytes) != 4 && (bytes) != 8) throw Error(GPART_ERR_INVALID_ARGUMENT, "cache entries are 4 or 8 bytes"); \
        if ((width) == GPART_WIDTH_STANDARD && (bytes) == 4) {                                        \
            using OpsT = Ops<std::int32_t, std::uint32_t, unsigned>;                                  \
            using CacheT = unsigned;                                                                  \
            call;                                                                                     \
        } else if ((width) == GPART_WIDTH_STANDARD) {                                                 \
            using OpsT = Ops<std::int32_t, std::uint32_t, unsigned long long>;                        \
            using CacheT = unsigned long long;                                                        \
            call;                                                                                     \
        } else if ((bytes) == 4) {                                                                    \
            using OpsT = Ops<std::int64_t, std::uint64_t, unsigned>;                                  \
            using CacheT = unsigned;                                                                  \
            call;                                                                                     \
        } else {                                                                                      \
            using OpsT = Ops<std::int64_t, std::uint64_t, unsigned long long>;                        \
            using CacheT = unsigned long long;                                                        \
            call;                                                                                     \
        }                                                                                             \
    } while (0)

extern "C" {

int gpart_refine_set_rebuild(gpart_ctx* ctx, int64_t min_entries, int64_t share) {
    return guarded([&] {
        if (!ctx) throw Error(GPART_ERR_INVALID_ARGUMENT, "null context");
        ctx->rebuild_min_entries = min_entries < 0 ? 0 : min_entries;
        ctx->rebuild_share = share;
    });
}

int gpart_cut(gpart_ctx* ctx, const gpart_csr_view* g, const int32_t* labels, uint64_t* cut) {
    return guarded([&] { GPART_WIDTH_DISPATCH(g->width, OpsT::cut(ctx, g, labels, cut)); });
}

int gpart_cut_noalloc(gpart_ctx* ctx, const gpart_csr_view* g, const int32_t* labels, uint64_t* cut) {
    return guarded([&] {
        if (!ctx || !g || !cut) throw Error(GPART_ERR_INVALID_ARGUMENT, "null context, graph or output");
        if (g->m > gpart_cut_noalloc_max_entries())
            throw Error(GPART_ERR_INVALID_ARGUMENT,
                        "gpart_cut_noalloc: " + std::to_string(g->m) + " entries exceed its limit of " +
                            std::to_string(gpart_cut_noalloc_max_entries()));
        void* base = nullptr;
        if (ctx->device >= 0 && ctx->device < kCutScratchDevices) {
            std::lock_guard<std::mutex> lock(cut_scratch_mutex());
            base = cut_scratch_address[ctx->device];
        }
        if (!base) throw Error(GPART_ERR_RUNTIME, "gpart_cut_noalloc: scratch of this device was not set up");
        auto* bytes = static_cast<unsigned char*>(base);
        auto* partials = reinterpret_cast<unsigned long long*>(bytes + kCutScratchPartialsOffset);
        auto* tile_row = reinterpret_cast<std::int32_t*>(bytes + kCutScratchTilesOffset);
        GPART_WIDTH_DISPATCH(g->width, OpsT::cut_with(ctx, g, labels, tile_row, partials, cut));
    });
}

int64_t gpart_cut_noalloc_max_entries(void) { return kCutScratchTiles * kTileEdges; }

int gpart_part_weights(gpart_ctx* ctx, const gpart_csr_view* g, const int32_t* labels, int k,
                       uint64_t* part_weights) {
    return guarded([&] {
        if (k < 1 || k > 32) throw Error(GPART_ERR_INVALID_ARGUMENT, "part count must be in [1, 32]");
        fill_bytes(ctx, part_weights, 0, static_cast<std::size_t>(k) * 8);
        if (g->n <= 0) return;
        const unsigned blocks = std::min<unsigned>(grid_for(g->n), 1024);
        auto* pw = reinterpret_cast<unsigned long long*>(part_weights);
        if (g->width == GPART_WIDTH_STANDARD)
            hipLaunchKernelGGL(part_weights_kernel<std::uint32_t>, dim3(blocks), dim3(kBlock), 0, ctx->stream, g->n,
                               labels, static_cast<const std::uint32_t*>(g->vertex_weights), k, pw);
        else
            hipLaunchKernelGGL(part_weights_kernel<std::uint64_t>, dim3(blocks), dim3(kBlock), 0, ctx->stream, g->n,
                               labels, static_cast<const std::uint64_t*>(g->vertex_weights), k, pw);
        GPART_LAUNCH_CHECK();
    });
}

int gpart_project(gpart_ctx* ctx, int64_t n, const int32_t* map, const int32_t* coarse_labels, int32_t* fine_labels) {
    return guarded([&] {
        if (n <= 0) return;
        hipLaunchKernelGGL(project_kernel, dim3(grid_for(n)), dim3(kBlock), 0, ctx->stream, n, map, coarse_labels,
                           fine_labels);
        GPART_LAUNCH_CHECK();
    });
}

int gpart_refine_build_cache(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes,
                             const int32_t* labels, int k, void* cache, int cache_bytes) {
    return guarded([&] {
        GPART_CACHE_DISPATCH(g->width, cache_bytes,
                             OpsT::build_cache(ctx, g, classes, labels, k, static_cast<CacheT*>(cache)));
    });
}

int gpart_refine_lp_round(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes,
                          void* cache, int cache_bytes, int32_t* labels, int k, double filter, int32_t* locks,
                          int32_t* targets, int64_t* gains, int32_t* flags, uint64_t* part_weights,
                          gpart_refine_status* status) {
    return guarded([&] {
        if (k < 1 || k > 32) throw Error(GPART_ERR_INVALID_ARGUMENT, "part count must be in [1, 32]");
        if (g->n <= 0) throw Error(GPART_ERR_INVALID_ARGUMENT, "refinement round needs vertices");
        GPART_CACHE_DISPATCH(g->width, cache_bytes,
                             OpsT::lp_round(ctx, g, classes, static_cast<CacheT*>(cache), labels, k, filter, locks,
                                            targets, reinterpret_cast<long long*>(gains), flags,
                                            reinterpret_cast<unsigned long long*>(part_weights), nullptr, status));
        complete_outputs(ctx);
    });
}

int gpart_refine_rows_create(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes, int k,
                             int cache_bytes, gpart_refine_rows** rows) {
    return guarded([&] {
        if (!ctx || !g || !classes || !rows) throw Error(GPART_ERR_INVALID_ARGUMENT, "null argument");
        if (k < 1 || k > 32) throw Error(GPART_ERR_INVALID_ARGUMENT, "part count must be in [1, 32]");
        *rows = nullptr;
        if (cache_bytes != 4 || g->n <= 0 || g->m < kRowsMinDegree * g->n || g->n > kRowsMaxVertices) return;
        auto made = std::make_unique<gpart_refine_rows>();
        made->n = g->n;
        made->m = g->m;
        made->high_count = classes->high_count;
        made->width = g->width;
        made->k = k;
        made->form = g->n <= kStateBytes ? kByteState
                     : k <= 8 && g->n <= 2 * kStateBytes ? kNibbleState
                                                         : kMemoryState;
        made->states.reset(ctx, (g->n + 15) / 16 * 16);
        made->hubs = classes->max_degree > kHubChunk;
        if (made->hubs) {
            if (g->width == GPART_WIDTH_STANDARD)
                build_hub_chunks(ctx, static_cast<const std::int32_t*>(g->offsets), classes->high, classes->high_count,
                                 classes->high_edges, kHubChunk, made->chunks);
            else
                build_hub_chunks(ctx, static_cast<const std::int64_t*>(g->offsets), classes->high, classes->high_count,
                                 classes->high_edges, kHubChunk, made->chunks);
        }
        *rows = made.release();
    });
}

void gpart_refine_rows_destroy(gpart_refine_rows* rows) { delete rows; }

int gpart_refine_rows_reset(gpart_refine_rows* rows) {
    return guarded([&] {
        if (!rows) throw Error(GPART_ERR_INVALID_ARGUMENT, "null rows");
        rows->ready = false;
    });
}

int gpart_refine_rows_check(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes,
                            gpart_refine_rows* rows, uint32_t* cache, const int32_t* labels, int k,
                            const uint64_t* part_weights, uint64_t capacity, const uint32_t* expected,
                            int64_t* differing) {
    return guarded([&] {
        if (!rows) throw Error(GPART_ERR_INVALID_ARGUMENT, "null rows");
        rows->check(g, classes, k);
        GPART_ROWS_DISPATCH(g->width, {
            OpsT::prepare_rows(ctx, g, classes, rows, labels, k, cache);
            *differing = OpsT::check_rows(ctx, g, classes, rows, labels, k, cache,
                                          reinterpret_cast<const unsigned long long*>(part_weights), capacity, expected);
        });
        rows->ready = true;
    });
}

int gpart_refine_lp_round_rows(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes,
                               gpart_refine_rows* rows, uint32_t* cache, int32_t* labels, int k, double filter,
                               int32_t* locks, int32_t* targets, int64_t* gains, int32_t* flags,
                               uint64_t* part_weights, gpart_refine_status* status) {
    return guarded([&] {
        if (!rows) throw Error(GPART_ERR_INVALID_ARGUMENT, "null rows");
        rows->check(g, classes, k);
        GPART_ROWS_DISPATCH(g->width, {
            OpsT::prepare_rows(ctx, g, classes, rows, labels, k, cache);
            OpsT::lp_round(ctx, g, classes, cache, labels, k, filter, locks, targets,
                           reinterpret_cast<long long*>(gains), flags,
                           reinterpret_cast<unsigned long long*>(part_weights), rows, status);
        });
        rows->ready = true;
        complete_outputs(ctx);
    });
}

int gpart_refine_rebalance_round_rows(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes,
                                      gpart_refine_rows* rows, uint32_t* cache, int32_t* labels, int k,
                                      uint64_t* part_weights, uint64_t capacity, int32_t* targets, int32_t* flags,
                                      gpart_refine_status* status) {
    return guarded([&] {
        if (!rows) throw Error(GPART_ERR_INVALID_ARGUMENT, "null rows");
        rows->check(g, classes, k);
        GPART_ROWS_DISPATCH(g->width, {
            OpsT::prepare_rows(ctx, g, classes, rows, labels, k, cache);
            OpsT::rebalance_round(ctx, g, classes, cache, labels, k,
                                  reinterpret_cast<unsigned long long*>(part_weights), capacity, targets, flags,
                                  rows, status);
        });
        rows->ready = true;
        complete_outputs(ctx);
    });
}

int gpart_refine_set_balance_blocks(gpart_ctx* ctx, int64_t blocks) {
    return guarded([&] {
        if (blocks < 1 || blocks > (int64_t{1} << 20)) throw Error(GPART_ERR_INVALID_ARGUMENT, "block count out of range");
        ctx->balance_blocks = blocks;
    });
}

int gpart_refine_set_few_leaving(gpart_ctx* ctx, int64_t vertices) {
    return guarded([&] {
        if (!ctx || vertices < -1 || vertices > (int64_t{1} << 28))
            throw Error(GPART_ERR_INVALID_ARGUMENT, "leaving vertices out of range");
        ctx->few_leaving = vertices;
    });
}

int gpart_refine_selection_stats(gpart_ctx* ctx, int64_t* single, int64_t* slices, int64_t* refused) {
    return guarded([&] {
        if (!ctx) throw Error(GPART_ERR_INVALID_ARGUMENT, "null context");
        if (single) *single = ctx->single_selections;
        if (slices) *slices = ctx->slice_selections;
        if (refused) *refused = ctx->refused_selections;
    });
}

int gpart_refine_set_graphs(gpart_ctx* ctx, int enabled) {
    return guarded([&] {
        GPART_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        ctx->round_plans.reset();
        ctx->round_graphs = enabled != 0;
    });
}

int gpart_refine_graphs_enabled(gpart_ctx* ctx) { return ctx && ctx->round_graphs ? 1 : 0; }

int gpart_refine_graph_stats(gpart_ctx* ctx, int64_t* plans, int64_t* captures, int64_t* replays) {
    return guarded([&] {
        const RoundPlans* set = ctx->round_plans ? static_cast<const RoundPlans*>(ctx->round_plans.get()) : nullptr;
        if (plans) *plans = set ? static_cast<int64_t>(set->plans.size()) : 0;
        if (captures) *captures = set ? set->captures : 0;
        if (replays) *replays = set ? set->replays : 0;
    });
}

int gpart_refine_rebalance_round(gpart_ctx* ctx, const gpart_csr_view* g, const gpart_degree_classes* classes,
                                 void* cache, int cache_bytes, int32_t* labels, int k, uint64_t* part_weights,
                                 uint64_t capacity, int32_t* targets, int32_t* flags, gpart_refine_status* status) {
    return guarded([&] {
        if (k < 1 || k > 32) throw Error(GPART_ERR_INVALID_ARGUMENT, "part count must be in [1, 32]");
        if (g->n <= 0) throw Error(GPART_ERR_INVALID_ARGUMENT, "refinement round needs vertices");
        GPART_CACHE_DISPATCH(g->width, cache_bytes,
                             OpsT::rebalance_round(ctx, g, classes, static_cast<CacheT*>(cache), labels, k,
                                                   reinterpret_cast<unsigned long long*>(part_weights), capacity,
                                                   targets, flags, nullptr, status));
        complete_outputs(ctx);
    });
}

int gpart_max_edge_weight(gpart_ctx* ctx, const gpart_csr_view* g, uint64_t* maximum) {
    return guarded([&] {
        unsigned long long h = 0;
        if (g->m > 0)
            with_weights(g->width, g->edge_weights, [&](auto load) { reduce_read<MaxU64>(ctx, load, g->m, &h); });
        *maximum = h;
    });
}

int gpart_edge_weight_sum(gpart_ctx* ctx, const gpart_csr_view* g, uint64_t* checked, uint64_t* limited) {
    return guarded([&] {
        unsigned long long h[2] = {0, 0};
        if (g->m > 0)
            with_weights(g->width, g->edge_weights,
                         [&](auto load) { reduce_read<CheckedSumU64, LimitedSumU64>(ctx, load, g->m, h); });
        *checked = h[0];
        *limited = h[1];
    });
}

int gpart_vertex_weight_stats(gpart_ctx* ctx, const gpart_csr_view* g, uint64_t* total, uint64_t* maximum,
                              uint64_t* minimum) {
    return guarded([&] {
        unsigned long long h[3] = {0, 0, 0};
        if (g->n > 0)
            with_weights(g->width, g->vertex_weights,
                         [&](auto load) { reduce_read<CheckedSumU64, MaxU64, MinU64>(ctx, load, g->n, h); });
        *total = h[0];
        *maximum = h[1];
        *minimum = h[2];
    });
}

}  // extern "C"
