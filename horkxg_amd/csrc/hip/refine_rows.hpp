// refine_rows.hpp -- connectivity rows computed when they are read.
//
// The incremental cache pays two device-scope atomics per entry of a mover's row
// (about 10 G atomics/s on MI355X, whatever the addresses). On a dense level (tens of
// entries per vertex and up) a rebalance iteration moves vertices holding a tenth of
// the level's entries, while it reads the rows of the overloaded parts only. There
// nothing is updated: a rebalance iteration sums its candidates' rows from the CSR,
// an LP round every row, and a round's movers are walked once for the cut. Rows are
// sums of the same integers either way.
//
// What bounds such a pass is the gather of a neighbour's part: 4-byte labels from the
// L2 reached 115 G entries/s (0.9 TB/s of CSR). So the parts are kept as a byte per
// vertex, and every workgroup, one or two per CU, first copies all of them into its
// LDS, a byte each, or half a byte for k <= 8, and gathers there while the CSR streams
// past: 240 G entries/s. Levels that do not fit gather the bytes from memory.
//
// Rows of more than 256 entries take a wave each, rows above kHubChunk entries a wave
// per chunk with the parts' sums added to the row; a workgroup lists the wanted ones of
// its share and its waves draw them from a counter in LDS, since a rebalance iteration
// wants a tenth of the rows, of any length up to the chunk (fixed shares left most waves
// waiting for the longest). Every wave sums into LDS words of its own, several copies
// per part: neighbours mostly share one part, and the lanes of one LDS atomic that meet
// in a word are served one by one.
#pragma once

#include "hubs.hpp"
#include "internal.hpp"
#include "refine_device.hpp"

namespace gpart_hip {
namespace {

constexpr int kRowsThreads = 1024;
constexpr int kRowsWaves = kRowsThreads / kWave;
constexpr int kRowsGroups = 256;  // workgroups of a launch at most: one per CU,
constexpr std::size_t kRowsPairLds = 74 * 1024;  // two where their LDS allows it
// LDS words of a wave: the sums of 8 rows (8 lanes each), of 4 rows in 2 copies (16
// lanes each) or of one row in 8 copies (the wave), 32 parts each; then a list of 64.
constexpr int kRowsWaveWords = 8 * 32 + kWave;
constexpr std::size_t kRowsWaveBytes = static_cast<std::size_t>(kRowsWaves) * kRowsWaveWords * 4;
constexpr std::int64_t kStateBytes = 128 * 1024;
static_assert(kRowsWaveBytes % 16 == 0, "the states behind the waves' words are aligned to 16 bytes");
static_assert(kRowsWaveBytes + kStateBytes + 9 * 1024 <= 160 * 1024, "with the row list they fit a CU's 160 KB");
// Dense: from this many entries per vertex. R-MAT levels have 29 and more (refinement of
// R-MAT 18, k = 8: 36 -> 20 ms); the mesh levels' 17 and less stay with the cache, whose
// rows are shorter than theirs. Up to as many vertices as an XCD's 4 MB L2 holds states:
// R-MAT 22 at 4.2 M vertices takes 16.9 ms against 17.4 with the cache, at 785 k 23.4
// against 28.9; R-MAT 24 at 16.8 M takes 119 against 104.
constexpr std::int64_t kRowsMinDegree = 24;
constexpr std::int64_t kRowsMaxVertices = std::int64_t{4} << 20;

// A vertex's state byte: its part, with the top bit for a mover of the round that is
// ending (the part is then its new one). Every round's first pass over the vertices
// rewrites it from the labels, the selections mark their movers.
constexpr unsigned kMovedBit = 0x80;
__device__ __forceinline__ void mark_mover(unsigned char* state, std::int32_t v, std::int32_t target) {
    if (state) state[v] = static_cast<unsigned char>(kMovedBit | static_cast<unsigned>(target));
}

// Where a pass gathers the states: bytes in LDS, half bytes in LDS, bytes in memory.
enum StateForm { kByteState, kNibbleState, kMemoryState };

// The states of all vertices as a pass reads them.
template <int Form>
struct States {
    const unsigned* words;        // LDS
    const unsigned char* memory;  // kMemoryState
    __device__ __forceinline__ unsigned raw(std::int32_t v) const {
        if constexpr (Form == kNibbleState) return words[v >> 3] >> ((v & 7) * 4) & 15U;
        else if constexpr (Form == kByteState) return reinterpret_cast<const unsigned char*>(words)[v];
        else return memory[v];
    }
    static constexpr unsigned kMoved = Form == kNibbleState ? 8U : kMovedBit;
    static constexpr unsigned kPart = Form == kNibbleState ? 7U : 31U;
    __device__ __forceinline__ int part(std::int32_t v) const { return static_cast<int>(raw(v) & kPart); }
};

// Four state bytes as four half bytes.
__device__ __forceinline__ unsigned pack_states(unsigned x) {
    unsigned out = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const unsigned b = x >> (8 * j);
        out |= ((b & 7U) | (b >> 4 & 8U)) << (4 * j);
    }
    return out;
}

// Copies the states (padded to whole 16 bytes) into LDS. Called by the workgroup.
template <int Form>
__device__ __forceinline__ void stage_states(const unsigned char* state, std::int64_t n, unsigned* words) {
    if constexpr (Form == kMemoryState) return;
    const auto* in = reinterpret_cast<const uint4*>(state);
    const int chunks = static_cast<int>((n + 15) / 16);
#pragma unroll 4
    for (int i = threadIdx.x; i < chunks; i += kRowsThreads) {
        const uint4 x = in[i];
        if constexpr (Form == kNibbleState) {
            reinterpret_cast<uint2*>(words)[i] =
                make_uint2(pack_states(x.x) | pack_states(x.y) << 16, pack_states(x.z) | pack_states(x.w) << 16);
        } else {
            reinterpret_cast<uint4*>(words)[i] = x;
        }
    }
}
inline std::size_t state_lds_bytes(std::int64_t n, int form) {
    const auto chunks = static_cast<std::size_t>((n + 15) / 16);
    return form == kMemoryState ? 0 : chunks * (form == kNibbleState ? 8 : 16);
}

// Adds the entries [begin, end) with stride G, those of v itself aside, to the sums
// of their parts: sums[part * Copies + copy]. A lane's loads of a trip are independent.
template <int G, int Copies, int Unroll, int Form, typename W>
__device__ __forceinline__ void add_row(std::int32_t v, std::int64_t begin, std::int64_t end, int sub,
                                        const std::int32_t* neighbors, const W* weights,
                                        const States<Form>& state, unsigned* sums) {
    const int copy = sub & (Copies - 1);
    for (std::int64_t e = begin + sub; e < end; e += G * Unroll) {
        std::int32_t nb[Unroll];
        unsigned w[Unroll];
#pragma unroll
        for (int u = 0; u < Unroll; ++u) {
            const bool in = e + u * G < end;
            nb[u] = in ? neighbors[e + u * G] : v;
            w[u] = in ? static_cast<unsigned>(weights[e + u * G]) : 0U;
        }
        int part[Unroll];
#pragma unroll
        for (int u = 0; u < Unroll; ++u) part[u] = state.part(nb[u]);
#pragma unroll
        for (int u = 0; u < Unroll; ++u)
            if (nb[u] != v) atomicAdd(&sums[part[u] * Copies + copy], w[u]);
    }
}

// The row of a group's sums into the cache, the sums cleared for the next row.
template <int G, int Copies, bool Add>
__device__ __forceinline__ void store_row(std::int32_t v, int sub, int k, unsigned* sums, unsigned* cache) {
    for (int p = sub; p < k; p += G) {
        unsigned total = 0;
#pragma unroll
        for (int c = 0; c < Copies; ++c) {
            total += sums[p * Copies + c];
            sums[p * Copies + c] = 0;
        }
        unsigned* out = cache + static_cast<std::int64_t>(v) * k + p;
        if constexpr (Add) {
            if (total) atomicAdd(out, total);
        } else {
            *out = total;
        }
    }
}

// The rows of a level by degree class and the chunks of its hub rows.
struct RowLists {
    const std::int32_t* low;
    const std::int32_t* medium;
    const std::int32_t* high;
    std::int64_t low_count, medium_count, high_count;
    const std::int64_t* chunk_total;  // null: no hub rows
    const std::int64_t* chunk_start;
    const std::int32_t* chunk_hub;
};

// Visits the list entries [0, count): a wave looks up `Lookups` of them at once, gathers
// the wanted ones in its LDS list and gives them to its groups of G lanes. Every lane
// of the wave calls body(v, sub) or skips it as its group does.
template <int G, int Lookups, typename Wanted, typename Body>
__device__ __forceinline__ void visit_rows(const std::int32_t* list, std::int64_t count, std::int64_t wave,
                                           std::int64_t waves, int* slots, Wanted wanted, Body body) {
    const int lane = lane_id();
    for (std::int64_t base = wave * Lookups; base < count; base += waves * Lookups) {
        const std::int64_t row = base + lane;
        std::int32_t v = 0;
        bool want = false;
        if (lane < Lookups && row < count) {
            v = list[row];
            want = wanted(v);
        }
        const unsigned long long lanes = __ballot(want);
        const int rows = __popcll(lanes);
        if (want) slots[__popcll(lanes & lanemask_lt())] = v;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int r = lane / G; r < rows; r += kWave / G) body(slots[r], lane & (G - 1));
        __builtin_amdgcn_wave_barrier();
    }
}

// Rows to be summed a wave each, as a workgroup lists them.
struct RowQueue {
    std::int32_t item[kRowsThreads];
    int count;
    int next;
};

// Visits the items [0, count) strided over the workgroups, one wave per wanted item: a
// thread looks up one item per pass (wanted(i)), the waves draw the wanted ones and call
// body(i) with every lane. Called by the whole workgroup.
template <typename Wanted, typename Body>
__device__ __forceinline__ void visit_wave_rows(std::int64_t count, RowQueue& queue, Wanted wanted, Body body) {
    const int lane = lane_id();
    const std::int64_t groups = gridDim.x;
    for (std::int64_t base = blockIdx.x; base < count; base += groups * kRowsThreads) {
        if (threadIdx.x == 0) queue.count = queue.next = 0;
        __syncthreads();
        const std::int64_t i = base + static_cast<std::int64_t>(threadIdx.x) * groups;
        const bool want = i < count && wanted(i);
        const unsigned long long lanes = __ballot(want);
        int at = 0;
        if (lane == 0 && lanes) at = atomicAdd(&queue.count, __popcll(lanes));
        at = __builtin_amdgcn_readfirstlane(at);
        if (want) queue.item[at + __popcll(lanes & lanemask_lt())] = static_cast<std::int32_t>(i);
        __syncthreads();
        for (;;) {
            int x = 0;
            if (lane == 0) x = atomicAdd(&queue.next, 1);
            x = __builtin_amdgcn_readfirstlane(x);
            if (x >= queue.count) break;
            body(static_cast<std::int64_t>(queue.item[x]));
        }
        __syncthreads();
    }
}

// Rows into the cache: every vertex's, or (part_weights) those of the vertices of parts
// above capacity. Hub rows must be zero before.
template <typename O, typename W, int Form>
__global__ void __launch_bounds__(kRowsThreads) rows_kernel(RowLists lists, const unsigned char* states,
                                                            std::int64_t n, const O* offsets,
                                                            const std::int32_t* neighbors, const W* weights, int k,
                                                            unsigned* cache, const unsigned long long* part_weights,
                                                            std::uint64_t capacity) {
    extern __shared__ __align__(16) unsigned lds[];  // stage_states stores 16 bytes at once
    __shared__ RowQueue queue;
    const int lane = lane_id(), wave_in = threadIdx.x / kWave;
    unsigned* sums = lds + wave_in * kRowsWaveWords;
    int* slots = reinterpret_cast<int*>(sums + 8 * 32);
    unsigned* words = lds + kRowsWaves * kRowsWaveWords;
    stage_states<Form>(states, n, words);
    for (int i = lane; i < 8 * 32; i += kWave) sums[i] = 0;
    unsigned wanted = ~0U;
    if (part_weights)
        wanted = static_cast<unsigned>(__ballot(lane < k && part_weights[lane < k ? lane : 0] > capacity));
    __syncthreads();
    const States<Form> state{words, states};
    const std::int64_t wave = static_cast<std::int64_t>(wave_in) * gridDim.x + blockIdx.x;
    const std::int64_t waves = static_cast<std::int64_t>(gridDim.x) * kRowsWaves;
    auto want = [&](std::int32_t v) -> bool { return wanted >> state.part(v) & 1U; };
    if (lists.chunk_total)
        visit_wave_rows(
            *lists.chunk_total, queue, [&](std::int64_t c) { return want(lists.high[lists.chunk_hub[c]]); },
            [&](std::int64_t c) {
                std::int32_t i, v;
                std::int64_t begin, end;
                hub_chunk_range(offsets, lists.high, lists.chunk_start, lists.chunk_hub, c, &i, &v, &begin, &end);
                add_row<kWave, 8, 8>(v, begin, end, lane, neighbors, weights, state, sums);
                store_row<kWave, 8, true>(v, lane, k, sums, cache);
            });
    visit_wave_rows(
        lists.high_count, queue,
        [&](std::int64_t i) {
            const std::int32_t v = lists.high[i];
            return want(v) && offsets[v + 1] - offsets[v] <= kHubChunk;
        },
        [&](std::int64_t i) {
            const std::int32_t v = lists.high[i];
            add_row<kWave, 8, 8>(v, static_cast<std::int64_t>(offsets[v]), static_cast<std::int64_t>(offsets[v + 1]),
                                 lane, neighbors, weights, state, sums);
            store_row<kWave, 8, false>(v, lane, k, sums, cache);
        });
    visit_rows<16, 16>(lists.medium, lists.medium_count, wave, waves, slots, want, [&](std::int32_t v, int sub) {
        unsigned* mine = sums + (lane / 16) * 64;
        add_row<16, 2, 4>(v, static_cast<std::int64_t>(offsets[v]), static_cast<std::int64_t>(offsets[v + 1]), sub,
                          neighbors, weights, state, mine);
        store_row<16, 2, false>(v, sub, k, mine, cache);
    });
    visit_rows<8, kWave>(lists.low, lists.low_count, wave, waves, slots, want, [&](std::int32_t v, int sub) {
        unsigned* mine = sums + (lane / 8) * 32;
        add_row<8, 1, 1>(v, static_cast<std::int64_t>(offsets[v]), static_cast<std::int64_t>(offsets[v + 1]), sub,
                         neighbors, weights, state, mine);
        store_row<8, 1, false>(v, sub, k, mine, cache);
    });
}

// Before a level's first round: the states (where given) from the labels, every hub row
// of the cache to zero (as each round leaves them).
__global__ void __launch_bounds__(256) rows_prepare_kernel(RowLists lists, std::int64_t n, const std::int32_t* labels,
                                                           unsigned char* states, int k, unsigned* cache) {
    const std::int64_t threads = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    if (states)
        for (std::int64_t v = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; v < n; v += threads)
            states[v] = static_cast<unsigned char>(labels[v]);
    if (!lists.chunk_total) return;
    for (std::int64_t c = blockIdx.x; c < *lists.chunk_total; c += gridDim.x) {
        const std::int32_t i = lists.chunk_hub[c];
        if (c != lists.chunk_start[i]) continue;  // a hub's first chunk clears its row
        if (threadIdx.x < static_cast<unsigned>(k))
            cache[static_cast<std::int64_t>(lists.high[i]) * k + threadIdx.x] = 0;
    }
}

// Whether entry i of the rows that rows_kernel sums differs from the expected one.
struct RowsDiffer {
    const unsigned* cache;
    const unsigned* expected;
    const std::int32_t* labels;
    const unsigned long long* part_weights;  // null: every row
    std::uint64_t capacity;
    int k;
    __device__ __forceinline__ unsigned long long operator()(std::int64_t i) const {
        if (part_weights && part_weights[labels[i / k]] <= capacity) return 0;
        return cache[i] != expected[i];
    }
};

// The cut change of a mover's entries [begin, end) with stride G (the lanes' shares), as
// update_cache_movers counts it: a neighbour that moves too counts once, at the lower
// id, and only then its old part is fetched.
template <int G, int Unroll, int Form, typename W>
__device__ __forceinline__ long long mover_gain(std::int32_t v, std::int32_t source, std::int32_t target,
                                                std::int64_t begin, std::int64_t end, int sub,
                                                const std::int32_t* neighbors, const W* weights,
                                                const States<Form>& state, const std::int32_t* flags) {
    long long gain = 0;
    for (std::int64_t e = begin + sub; e < end; e += G * Unroll) {
        std::int32_t nb[Unroll];
        unsigned states[Unroll];
        W w[Unroll];
#pragma unroll
        for (int u = 0; u < Unroll; ++u) {
            const bool in = e + u * G < end;
            nb[u] = in ? neighbors[e + u * G] : v;
            w[u] = in ? weights[e + u * G] : W{0};
        }
#pragma unroll
        for (int u = 0; u < Unroll; ++u) states[u] = state.raw(nb[u]);
#pragma unroll
        for (int u = 0; u < Unroll; ++u) {
            const unsigned raw = states[u];
            const bool moved = raw & States<Form>::kMoved;
            const int after = static_cast<int>(raw & States<Form>::kPart);
            if (nb[u] == v || (moved && nb[u] < v)) continue;
            const int before = moved ? flags[nb[u]] - 1 : after;
            gain += static_cast<long long>(w[u]) * ((source != before) - (target != after));
        }
    }
    return gain;
}

}  // namespace
}  // namespace gpart_hip

// A level in this form: its sizes, the chunk map of its hub rows and the states of its
// vertices.
struct gpart_refine_rows {
    std::int64_t n, m, high_count;
    int width, k;
    gpart_hip::HubChunks chunks;
    gpart_hip::Scratch<unsigned char> states;  // n, rounded up to 16
    bool hubs = false;
    int form = gpart_hip::kByteState;
    // States and hub rows are as a round expects them: not before the first round, not
    // after a round that failed, nor once the caller has changed labels.
    bool ready = false;

    // The arrays' sizes depend on these, so a round of another level is refused.
    void check(const gpart_csr_view* g, const gpart_degree_classes* c, int parts) const {
        if (g->n != n || g->m != m || g->width != width || c->high_count != high_count || parts != k)
            throw gpart_hip::Error(GPART_ERR_INVALID_ARGUMENT, "the rows belong to another level or part count");
    }
};
