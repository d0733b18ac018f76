// initial.hip -- weighted recursive spectral bisection for gfx950
// (src/initial_partition_gpu.cu of the reference).
//
// Both forms keep the reference's FP64 summation order so that results are
// reproducible and identical between forms:
//   * a vertex is owned by 32 lanes (half a wave64); lane l accumulates entries
//     e = begin+l, begin+l+32, ... in increasing e, then a 32-lane shuffle-down
//     tree (16, 8, 4, 2, 1) combines them;
//   * moments are combined per 8 consecutive vertices with the reference's
//     block tree ((z0+z4)+(z2+z6))+((z1+z5)+(z3+z7)), z = m + 0.0;
//   * the normalisation sums those partials with 256 strided accumulators and
//     the same trees.
// Multiply-adds are fused only where written with fma() (the SpMV accumulation
// and the variance); the library is built with -ffp-contract=off.
//
// Plain form: the reference's launch structure, one task at a time (start, then
// per step: SpMV, finish_moments, normalize).
// Batched form: all tasks of one recursion depth share every launch. Small sparse tasks
// take a single one (the solo form below), else a depth is 66 launches whatever its task
// count: start, 64 steps (each also finishing the previous step's moments and
// normalising on read), and one 1024-thread workgroup per task for the (x, id) sort
// (LDS bitonic), the weight prefix, the feasible split and the label assignment,
// emitting the child tasks.
#include "internal.hpp"
#include "scan.hpp"
#include "spectral_device.hpp"

#include <algorithm>
#include <cstring>
#include <cmath>

namespace gpart_hip {
namespace {

// ------------------------------------------------------------------ plain form

template <typename O, typename W>
__global__ void __launch_bounds__(256) spectral_start_kernel(int count, const int* ids, const int* labels, int group,
                                                             const O* offsets, const int* neighbors, const W* weights,
                                                             double* degree, double* x, unsigned seed,
                                                             Moments* partials, unsigned long long* entries) {
    __shared__ Moments vm[8];
    const int lane = threadIdx.x & 31, hw = threadIdx.x >> 5;
    const int i = blockIdx.x * 8 + hw;
    double d = 0;
    if (i < count) {
        const int v = ids[i];
        for (std::int64_t e = static_cast<std::int64_t>(offsets[v]) + lane; e < offsets[v + 1]; e += 32)
            if (labels[neighbors[e]] == group) d += static_cast<double>(weights[e]);
    }
    d = tree32(d);
    if (lane == 0) {
        Moments m{0, 0, 0};
        if (i < count) {
            const int v = ids[i];
            // CSR entries each diffusion step scans, for the family's algorithmic bytes:
            // counted under profiling only, the atomics of all rows meet in one word
            // (7,429 rows: 48 us of the launch's 52)
            if (entries) atomicAdd(entries, static_cast<unsigned long long>(offsets[v + 1] - offsets[v]));
            const double a = static_cast<double>(mix32(static_cast<unsigned>(v) ^ seed)) / 4294967296.0 - 0.5;
            degree[v] = d;
            x[v] = a;
            const double mass = d > 0 ? d : 1.0;
            m = Moments{mass, mass * a, mass * a * a};
        }
        vm[hw] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = block_partial(vm, 0, 8);
}

template <typename O, typename W, typename T>
__global__ void __launch_bounds__(256) spectral_step_kernel(int count, const int* ids, const int* labels, int group,
                                                            const O* offsets, const int* neighbors, const W* weights,
                                                            const double* degree, const T* x, T* y,
                                                            Moments* partials) {
    __shared__ Moments vm[8];
    const int lane = threadIdx.x & 31, hw = threadIdx.x >> 5;
    const int i = blockIdx.x * 8 + hw;
    double sum = 0;
    if (i < count) {
        const int v = ids[i];
        for (std::int64_t e = static_cast<std::int64_t>(offsets[v]) + lane; e < offsets[v + 1]; e += 32) {
            const int u = neighbors[e];
            if (labels[u] == group) sum = fma(static_cast<double>(weights[e]), static_cast<double>(x[u]), sum);
        }
    }
    sum = tree32(sum);
    if (lane == 0) {
        Moments m{0, 0, 0};
        if (i < count) {
            const int v = ids[i];
            const double d = degree[v];
            const double a = d > 0 ? 0.5 * (static_cast<double>(x[v]) + sum / d) : static_cast<double>(x[v]);
            y[v] = static_cast<T>(a);
            const double mass = d > 0 ? d : 1.0;
            m = Moments{mass, mass * a, mass * a * a};
        }
        vm[hw] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = block_partial(vm, 0, 8);
}

__global__ void __launch_bounds__(256) finish_moments_kernel(int count, const Moments* partials, Norm* norm) {
    __shared__ double shared8[24];
    __shared__ Norm shared_norm;
    const Norm r = finish_block(partials, count, shared8, &shared_norm);
    if (threadIdx.x == 0) *norm = r;
}

__global__ void normalize_kernel(int count, const int* ids, double* x, const Norm* norm) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        const int v = ids[i];
        x[v] = (x[v] - norm->mean) * norm->scale;
    }
}

__global__ void sort_keys_kernel(int count, const int* ids, const double* x, std::uint64_t* keys, std::uint64_t* vals,
                                 bool by_id) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int v = ids[i];
    keys[i] = by_id ? static_cast<std::uint64_t>(v) : ordered_bits(x[v]);
    vals[i] = static_cast<std::uint64_t>(v);
}

__global__ void copy_ids_kernel(int count, const std::uint64_t* vals, int* ids) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) ids[i] = static_cast<int>(vals[i]);
}

struct OrderWeightLoad {
    const int* ids;
    const std::uint64_t* weights;
    __device__ __forceinline__ std::uint64_t operator()(std::int64_t i) const { return weights[ids[i]]; }
};

__global__ void assign_split_kernel(int count, const int* ids, int boundary, int left, int right, int* labels) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) labels[ids[i]] = i < boundary ? left : right;
}

// ------------------------------------------------------------------ batched form

// All tasks of one depth share each launch: the grid is the concatenation of the
// tasks' 8-vertex blocks (the reference's own mapping), so every task, small or
// large, is spread over the whole GPU. One step is one launch: each workgroup
// first recomputes its task's normalisation from the previous step's block
// partials (finish_block, the reference's fixed order) and normalises x values as
// it reads them, (x - mean) * scale, the same expression the reference stores.
constexpr int kMaxDepthTasks = 32;

struct DepthTasks {
    int count;
    int first_block[kMaxDepthTasks + 1];  // prefix of ceil(task.count / 8)
    gpart_bisect_task task[kMaxDepthTasks];
};

__device__ __forceinline__ int task_of_block(const DepthTasks& dt, int block) {
    int t = 0;
    while (t + 1 < dt.count && dt.first_block[t + 1] <= block) ++t;
    return t;
}

// spectral_start (:81-107) for every task of the depth.
template <typename O, typename W, typename T>
__global__ void __launch_bounds__(256) depth_start_kernel(DepthTasks dt, const int* order, const int* labels,
                                                          const O* offsets, const int* neighbors, const W* weights,
                                                          unsigned seed, double* degree, T* x, Moments* partials,
                                                          unsigned long long* entries) {
    __shared__ Moments vm[8];
    const int t = task_of_block(dt, blockIdx.x);
    const gpart_bisect_task task = dt.task[t];
    const int* ids = order + task.begin;
    const int group = task.first_part;
    const unsigned tseed = seed ^ static_cast<unsigned>(task.first_part);
    const int lane = threadIdx.x & 31, hw = threadIdx.x >> 5;
    const int i = (blockIdx.x - dt.first_block[t]) * 8 + hw;
    double d = 0;
    if (i < task.count) {
        const int v = ids[i];
        for (std::int64_t e = static_cast<std::int64_t>(offsets[v]) + lane; e < offsets[v + 1]; e += 32)
            if (labels[neighbors[e]] == group) d += static_cast<double>(weights[e]);
    }
    d = tree32(d);
    if (lane == 0) {
        Moments m{0, 0, 0};
        if (i < task.count) {
            const int v = ids[i];
            if (entries) atomicAdd(entries, static_cast<unsigned long long>(offsets[v + 1] - offsets[v]));
            const double a = static_cast<double>(mix32(static_cast<unsigned>(v) ^ tseed)) / 4294967296.0 - 0.5;
            degree[v] = d;
            x[v] = static_cast<T>(a);
            const double av = static_cast<double>(static_cast<T>(a));
            const double mass = d > 0 ? d : 1.0;
            m = Moments{mass, mass * av, mass * av * av};
        }
        vm[hw] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = block_partial(vm, 0, 8);
}

// finish_moments (:65-79) of the previous step, normalize (:138-142) on read, and
// spectral_step (:109-136), for every task of the depth.
template <typename O, typename W, typename T>
__global__ void __launch_bounds__(256) depth_step_kernel(DepthTasks dt, const int* order, const int* labels,
                                                         const O* offsets, const int* neighbors, const W* weights,
                                                         const double* degree, const T* x, T* y,
                                                         const Moments* previous, Moments* partials) {
    __shared__ Moments vm[8];
    __shared__ double shared8[24];
    __shared__ Norm shared_norm;
    const int t = task_of_block(dt, blockIdx.x);
    const gpart_bisect_task task = dt.task[t];
    const int first = dt.first_block[t];
    const Norm norm = finish_block(previous + first, dt.first_block[t + 1] - first, shared8, &shared_norm);
    const int* ids = order + task.begin;
    const int group = task.first_part;
    const int lane = threadIdx.x & 31, hw = threadIdx.x >> 5;
    const int i = (blockIdx.x - first) * 8 + hw;
    T sum = 0;
    if (i < task.count) {
        const int v = ids[i];
        const auto end = static_cast<std::int64_t>(offsets[v + 1]);
        std::int64_t e = static_cast<std::int64_t>(offsets[v]) + lane;
        // the next neighbour under way while this one's label and value are: a long row is a
        // chain of such loads, which normalising on read lengthens (a row of 4,096 entries
        // took 12% longer than with the normalisation in a launch of its own)
        int u = e < end ? neighbors[e] : -1;
        while (u >= 0) {
            const std::int64_t next = e + 32;
            const int then = next < end ? neighbors[next] : -1;
            if (labels[u] == group) sum = VecTraits<T>::fmadd(static_cast<T>(weights[e]), normalized(x, u, norm), sum);
            e = next;
            u = then;
        }
    }
    const double sd = static_cast<double>(tree32(sum));
    if (lane == 0) {
        Moments m{0, 0, 0};
        if (i < task.count) {
            const int v = ids[i];
            const double d = degree[v];
            const T xv = normalized(x, v, norm);
            double a;
            if constexpr (sizeof(T) == 8) {
                a = d > 0 ? 0.5 * (static_cast<double>(xv) + sd / d) : static_cast<double>(xv);
            } else {
                const float df = static_cast<float>(d);
                const float af = d > 0 ? 0.5f * (xv + static_cast<float>(sd) / df) : xv;
                a = static_cast<double>(af);
            }
            y[v] = static_cast<T>(a);
            const double mass = d > 0 ? d : 1.0;
            m = Moments{mass, mass * a, mass * a * a};
        }
        vm[hw] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = block_partial(vm, 0, 8);
}

// The last normalisation of one task, in place.
__global__ void __launch_bounds__(256) depth_normalize_kernel(int count, const int* ids, double* x,
                                                              const Moments* partials, int blocks) {
    __shared__ double shared8[24];
    __shared__ Norm shared_norm;
    const Norm norm = finish_block(partials, blocks, shared8, &shared_norm);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) x[ids[i]] = normalized(x, ids[i], norm);
}

// The last normalisation, the (x, id) sort (:143-148, :230), the weight prefix and
// feasible split (:231-248) and the label assignment (:149-153): one workgroup per
// task, emitting the child tasks of the next depth.
template <typename T>
__global__ void __launch_bounds__(kBatchThreads) depth_finish_kernel(DepthTasks dt, int* labels, int* order,
                                                                     const std::uint64_t* vertex_weights,
                                                                     std::uint64_t capacity, const T* x,
                                                                     const Moments* partials, double* coords,
                                                                     gpart_bisect_task* next, int* next_count,
                                                                     int* status) {
    __shared__ BatchShared sh;
    const int t = blockIdx.x;
    const gpart_bisect_task task = dt.task[t];
    const int first = dt.first_block[t];
    const Norm norm = finish_block(partials + first, dt.first_block[t + 1] - first, sh.shared8, &sh.norm);
    const int st = split_task<T>(
        task, order + task.begin, labels, vertex_weights, capacity, coords, sh,
        [&](int, int v) { return normalized(x, v, norm); },
        [&](const gpart_bisect_task& child) { next[atomicAdd(next_count, 1)] = child; });
    if (st && threadIdx.x == 0) atomicMax(status, st);
}

// ------------------------------------------------------------------- solo form
//
// A step of a small sparse task is a few microseconds of launch and of dependent loads
// (id, row, neighbour, label, value) around a few hundred nanoseconds of work: 5.0-6.5
// us per launch, 64 per depth. Here one workgroup does a task's whole depth, start,
// steps and split, in one launch. The vector stays in LDS; a thread owns up to four
// rows, and their entries, resolved to positions inside the task once, lie in slots of
// one lane each (sliced ELL: rows of a wave share the width of the longest), so that a
// step reads them in runs from the L2. Values are bit-identical to the launch form: a
// thread sums its row's 32 strided accumulators and their tree itself (absent entries
// and other tasks' neighbours are zero terms), eight neighbouring lanes form a block's
// partial, and finish_block is the same. A step waits for its two barriers and the
// normalisation's chain (1.3 us at 460 rows), from about 2,000 rows on for the slots and
// the LDS reads. Bisection of a 7,429-vertex weighted mesh into 32, with its four depths
// below the root: 3.29 -> 2.33 ms.
constexpr int kSoloThreads = 1024;
constexpr int kSoloGroups = kMaxBatchedTask / kWave;  // groups of 64 rows, one width each
// Where every task of a depth is small and sparse enough the form is tried: up to this
// many entries by the task's share of the graph's vertices. Weighted 3D meshes, FP64, a
// depth of tasks of 3,700 vertices and 21,000 entries: 500 us, the launch form 500; of
// 1,860 and 10,500: 300 and 500; of 930 and 5,300: 190 and 490; of 460 and 2,600: 145 and
// 490.
constexpr double kSoloEntries = 16384;
// The share says nothing of how a skewed graph's entries lie, so the depth is measured
// first and left to the launch form where a task has more slots, or a longer row, than
// these: slots are padded to the longest row of each 64, and a wave has its groups to
// itself while the launch form spreads rows over all CUs. Bisections of one task, the
// launch form and the solo one in us: mesh, 216 rows of slots, 463 and 367; 344, 543 and
// 490; 424, 557 and 563; random, 16 entries a vertex, 488, 392 and 352; 664, 459 and 502;
// 936, 465 and 599; R-MAT 8, 248 and a row of 94, 384 and 371; 384 and a row of 119, 403
// and 449; R-MAT 9, 584 and 141, 434 and 506.
constexpr int kSoloRows = 416;  // slots of a task, in rows of 64
constexpr int kSoloWidth = 96;  // longest row, padded

struct SoloTasks {
    int count;
    gpart_bisect_task task[kMaxDepthTasks];
};

// The sum of a row's terms in the reference's order: accumulator l takes terms l,
// l + 32, ..., then a tree (16, 8, 4, 2, 1) whose absent leaves would add zero.
// terms(first, part) adds the terms from `first` on to a run of accumulators, whose
// loads are so under way together.
template <typename A, int N, int Run, typename Terms>
__device__ __forceinline__ A tree_sum(int width, Terms terms) {
    A v[N];
#pragma unroll
    for (int l = 0; l < N; ++l) v[l] = A(0);
    for (int first = 0; first < width; first += N) {
#pragma unroll
        for (int c = 0; c < N; c += Run) {
            A part[Run];
#pragma unroll
            for (int l = 0; l < Run; ++l) part[l] = v[c + l];
            terms(first + c, part);
#pragma unroll
            for (int l = 0; l < Run; ++l) v[c + l] = part[l];
            // no more than a run's loads at once: the registers do not hold them
            if constexpr (Run < N) __builtin_amdgcn_sched_barrier(0);
        }
        if (N < 32) break;
    }
#pragma unroll
    for (int h = 16; h > 0; h /= 2)
#pragma unroll
        for (int l = 0; l < h; ++l)
            if (l + h < N) v[l] += v[l + h];
    return v[0];
}
// over slots, the same width for a wave
template <typename A, typename Terms>
__device__ __forceinline__ A row_sum(int width, Terms terms) {
    if (width <= 4) return tree_sum<A, 4, 4>(width, terms);
    if (width <= 8) return tree_sum<A, 8, 8>(width, terms);
    if (width <= 12) return tree_sum<A, 12, 12>(width, terms);
    if (width <= 16) return tree_sum<A, 16, 8>(width, terms);
    if (width <= 24) return tree_sum<A, 24, 8>(width, terms);
    return tree_sum<A, 32, 8>(width, terms);
}
// the slots that row_sum reads for a row of `width` entries
__device__ __forceinline__ int padded_width(int width) {
    if (width <= 16) return (width + 3) / 4 * 4;
    return width <= 24 ? 24 : (width + 31) / 32 * 32;
}

// A slot: position in the low 12 bits, weight above. Of 4 bytes while a group's weights
// are below 2^20 (a step's time is the slots' way from the L2), else of 8, up to 2^52.
constexpr int kSlotShift = 12;
static_assert(kMaxBatchedTask <= 1 << kSlotShift, "a task's positions fit");

template <typename T>
struct SoloShared {
    BatchShared batch;  // its keys hold the degrees until the split
    T x[kMaxBatchedTask];   // normalised
    T y[kMaxBatchedTask];   // a step's result
    Moments partials[kMaxBatchedTask / 8];
    int width[kSoloGroups];  // of a group of 64 rows: its longest
    int slots[kSoloGroups];  // its first slot, in rows of 64
    int slot_bytes[kSoloGroups];
};

// Whether a task is one for the solo form, by its rows: refused[task] is 1 where one is
// longer than kSoloWidth, where the padded groups together need more than kSoloRows, or
// where a weight does not fit a slot. Also clears the depth's counters (two words).
template <typename O, typename W>
__global__ void __launch_bounds__(kSoloThreads) depth_measure_kernel(SoloTasks st, const int* order, const O* offsets,
                                                                     const W* weights, int* refused,
                                                                     unsigned long long* counters) {
    __shared__ int wave_rows[kSoloThreads / kWave];
    const gpart_bisect_task task = st.task[blockIdx.x];
    const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
    if (blockIdx.x == 0 && t < 2) counters[t] = 0;
    int rows = 0;
    bool unfit = false;
    for (int first = wave * kWave; first < task.count; first += kSoloThreads) {
        int width = 0;
        if (first + lane < task.count) {
            const int v = order[task.begin + first + lane];
            const auto begin = static_cast<std::int64_t>(offsets[v]), end = static_cast<std::int64_t>(offsets[v + 1]);
            width = static_cast<int>(end - begin < kSoloWidth + 1 ? end - begin : kSoloWidth + 1);
            if constexpr (sizeof(W) == 8) {
                std::uint64_t bits = 0;
                for (int e = 0; e < width; ++e) bits |= weights[begin + e];
                unfit = unfit || bits >> (64 - kSlotShift) != 0;
            }
        }
#pragma unroll
        for (int m = kWave / 2; m > 0; m /= 2) width = max(width, __shfl_xor(width, m, kWave));
        width = padded_width(width);
        unfit = unfit || width > kSoloWidth;
        rows += width;
    }
    if (lane == 0) wave_rows[wave] = rows;
    unfit = __syncthreads_or(unfit);
    if (t == 0) {
        int total = 0;
        for (int w = 0; w < kSoloThreads / kWave; ++w) total += wave_rows[w];
        refused[blockIdx.x] = unfit || total > kSoloRows;
    }
}

constexpr int kSoloRefused = -1;  // status of a depth with a refused task: nothing was done

template <typename O, typename W, typename T>
__global__ void __launch_bounds__(kSoloThreads) depth_solo_kernel(
    SoloTasks st, const int* refused, int* labels, int* order, const O* offsets, const int* neighbors,
    const W* weights, const std::uint64_t* vertex_weights, unsigned seed, std::uint64_t capacity, double* coords,
    int* position, std::uint64_t* slot, gpart_bisect_task* next, int* next_count, int* status,
    unsigned long long* entries) {
    __shared__ SoloShared<T> sh;
    if (__syncthreads_or(static_cast<int>(threadIdx.x) < st.count && refused[threadIdx.x])) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *status = kSoloRefused;
        return;
    }
    const gpart_bisect_task task = st.task[blockIdx.x];
    const int count = task.count, group = task.first_part, blocks = (count + 7) / 8;
    const int rounds = (count + kSoloThreads - 1) / kSoloThreads;
    int* ids = order + task.begin;
    double* degree = reinterpret_cast<double*>(sh.batch.keys);
    const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
    unsigned long long scanned = 0;
    if (t < kSoloGroups) sh.width[t] = 0;
    __syncthreads();
    for (int r = t, g = wave; g < rounds * (kSoloThreads / kWave); r += kSoloThreads, g += kSoloThreads / kWave) {
        int width = 0;
        if (r < count) {
            const int v = ids[r];
            position[v] = r;
            width = static_cast<int>(offsets[v + 1] - offsets[v]);
        }
        scanned += static_cast<unsigned long long>(width);
#pragma unroll
        for (int m = kWave / 2; m > 0; m /= 2) width = max(width, __shfl_xor(width, m, kWave));
        if (lane == 0) sh.width[g] = width;
    }
    scanned = group_sum_u64<kWave>(scanned);
    if (entries && lane == 0 && scanned) atomicAdd(entries, scanned);
    __syncthreads();  // widths and positions
    if (wave == 0) {
        const int width = padded_width(sh.width[lane]);
        sh.slots[lane] = static_cast<int>(blockIdx.x) * kSoloRows + wave_scan(width) - width;
    }
    __syncthreads();
    static_assert(kSoloGroups == kWave, "one wave places the groups");
    // four terms of row r from the CSR: weight (0: no entry, or another task's neighbour) and position
    auto resolve = [&](int r, int first, W (&w)[4], int (&pos)[4]) {
        std::int64_t e = 0, end = 0;
        if (r < count) {
            const int v = ids[r];
            e = static_cast<std::int64_t>(offsets[v]) + first;
            end = static_cast<std::int64_t>(offsets[v + 1]);
        }
        int u[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) u[l] = e + l < end ? neighbors[e + l] : -1;
#pragma unroll
        for (int l = 0; l < 4; ++l) w[l] = u[l] >= 0 ? weights[e + l] : W(0);
#pragma unroll
        for (int l = 0; l < 4; ++l)
            if (u[l] >= 0 && labels[u[l]] != group) u[l] = -1;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            pos[l] = u[l] >= 0 ? position[u[l]] : 0;
            w[l] = u[l] >= 0 ? w[l] : W(0);
        }
    };
    // row r's entries into its slots; returns all its weights or-ed
    auto fill = [&](int r, auto* slots) {
        using S = std::remove_pointer_t<decltype(slots)>;
        const int width = __builtin_amdgcn_readfirstlane(padded_width(sh.width[r / kWave]));
        std::uint64_t bits = 0;
#pragma unroll 1
        for (int first = 0; first < width; first += 4) {
            W w[4];
            int pos[4];
            resolve(r, first, w, pos);
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                bits |= w[l];
                slots[(first + l) * kWave + lane] = static_cast<S>(w[l]) << 12 | static_cast<S>(pos[l]);
            }
        }
        return bits;
    };
    // the sum of term(weight, position, accumulator) over row r
    auto over_row = [&](int r, auto zero, auto term) {
        using A = decltype(zero);
        const int g = r / kWave;
        const int width = __builtin_amdgcn_readfirstlane(sh.width[g]);
        auto stored = [&](const auto* at) {
            return row_sum<A>(width, [&](int first, auto& acc) {
                constexpr int N = sizeof(acc) / sizeof(A);
                std::remove_cv_t<std::remove_pointer_t<decltype(at)>> s[N];
#pragma unroll
                for (int l = 0; l < N; ++l) s[l] = at[(first + l) * kWave];
#pragma unroll
                for (int l = 0; l < N; ++l)
                    acc[l] = term(s[l] >> kSlotShift, static_cast<int>(s[l] & ((1 << kSlotShift) - 1)), acc[l]);
            });
        };
        const int bytes = __builtin_amdgcn_readfirstlane(sh.slot_bytes[g]);
        const std::uint64_t* at = slot + static_cast<std::int64_t>(sh.slots[g]) * kWave;
        return bytes == 4 ? stored(reinterpret_cast<const std::uint32_t*>(at) + lane) : stored(at + lane);
    };
    // a row's moments into its block of eight rows
    auto absorb = [&](int r, double mass, double a) {
        Moments m{0, 0, 0};
        if (r < count) m = Moments{mass, mass * a, mass * a * a};
        auto total = [](double v) {
            v = z(v);
            v += lane_down<4>(v);
            v += lane_down<2>(v);
            return v + lane_down<1>(v);
        };
        m = Moments{total(m.mass), total(m.sum), total(m.squares)};
        if ((t & 7) == 0 && r / 8 < blocks) sh.partials[r / 8] = m;
    };
    // spectral_start (:81-107)
    const unsigned tseed = seed ^ static_cast<unsigned>(task.first_part);
#pragma unroll 1
    for (int r = t; r < rounds * kSoloThreads; r += kSoloThreads) {
        const int g = r / kWave;
        std::uint64_t* slots = slot + static_cast<std::int64_t>(sh.slots[g]) * kWave;
        const std::uint64_t bits = fill(r, reinterpret_cast<std::uint32_t*>(slots));
        const bool wide = __any(bits >> (32 - kSlotShift) != 0);
        if (wide) fill(r, slots);
        if (lane == 0) sh.slot_bytes[g] = wide ? 8 : 4;
        const double d = over_row(r, 0.0, [](auto w, int, double acc) { return acc + static_cast<double>(w); });
        T x = 0;
        if (r < count) {
            x = static_cast<T>(static_cast<double>(mix32(static_cast<unsigned>(ids[r]) ^ tseed)) / 4294967296.0 - 0.5);
            degree[r] = d;
            sh.y[r] = x;
        }
        absorb(r, d > 0 ? d : 1.0, static_cast<double>(x));
    }
    __syncthreads();
    // finish_moments (:65-79), normalize (:138-142) and spectral_step (:109-136)
#pragma unroll 1
    for (int step = 0;; ++step) {
        const Norm norm = finish_block(sh.partials, blocks, sh.batch.shared8, &sh.batch.norm);
        for (int r = t; r < count; r += kSoloThreads)
            sh.x[r] = static_cast<T>((static_cast<double>(sh.y[r]) - norm.mean) * norm.scale);
        __syncthreads();
        if (step == 64) break;
#pragma unroll 1
        for (int r = t; r < rounds * kSoloThreads; r += kSoloThreads) {
            const T sum = over_row(r, T(0), [&](auto w, int pos, T acc) {
                return VecTraits<T>::fmadd(static_cast<T>(w), sh.x[pos], acc);
            });
            double a = 0, d = 0;
            if (r < count) {
                d = degree[r];
                const T x = sh.x[r];
                if constexpr (sizeof(T) == 8) {
                    a = d > 0 ? 0.5 * (x + sum / d) : x;
                } else {
                    a = static_cast<double>(d > 0 ? 0.5f * (x + sum / static_cast<float>(d)) : x);
                }
                sh.y[r] = static_cast<T>(a);
            }
            absorb(r, d > 0 ? d : 1.0, a);
        }
        __syncthreads();
    }
    const int failed = split_task<T>(
        task, ids, labels, vertex_weights, capacity, coords, sh.batch, [&](int i, int) { return sh.x[i]; },
        [&](const gpart_bisect_task& child) { next[atomicAdd(next_count, 1)] = child; });
    if (failed && t == 0) atomicMax(status, failed);
}

// Single tasks of at most this size take their steps through the depth's fused launches:
// one per step where step, moments and normalisation are three. Each workgroup reads all
// partials, 3 bytes a vertex, so the form's cost grows with the square of the size.
// Bisections of one task in us, three launches a step and one: 2D grids of 4,096 vertices
// 810 and 561, 8,281 940 and 784, 12,100 989 and 887, 13,924 1018 and 986, 15,876 1033 and
// 1061, 24,025 1235 and 1550; 3D meshes and random graphs of 16 and 64 entries a vertex
// cross at the same sizes, 14,000 to 16,000. With rows of half the vertices, whose chain of
// loads normalising on read lengthens, they are level from 6,000 (3305 and 3280) to 8,192
// (4228 and 4395) and one launch is behind above: the line lies there.
constexpr int kMaxFusedTask = 8192;

template <typename O, typename W>
void plain_task(gpart_ctx* ctx, const gpart_csr_view* g, const int32_t* labels, int32_t* order,
                const std::uint64_t* vertex_weights, const gpart_bisect_task* task, uint32_t seed, double* x,
                double* y, double* degree, std::uint64_t* prefix) {
    const int count = task->count;
    if (count <= 0) return;
    int* ids = order + task->begin;
    const auto* off = static_cast<const O*>(g->offsets);
    const auto* w = static_cast<const W*>(g->edge_weights);
    const int blocks = (count + 255) / 256;
    const int spectral_blocks = (count + 7) / 8;
    Scratch<Moments> partials(ctx, spectral_blocks);
    Scratch<Norm> norm(ctx, 1);
    Scratch<unsigned long long> entries(ctx, 1);
    fill_bytes(ctx, entries.get(), 0, 8);
    profile_begin(ctx, GPART_PROFILE_SPECTRAL);
    unsigned long long* scanned = ctx->profile[GPART_PROFILE_SPECTRAL].enabled ? entries.get() : nullptr;
    if (count <= kMaxFusedTask) {
        DepthTasks dt{};
        dt.count = 1;
        dt.first_block[1] = spectral_blocks;
        dt.task[0] = *task;
        Scratch<Moments> partials_alt(ctx, spectral_blocks);
        Moments* p = partials.get();
        Moments* q = partials_alt.get();
        hipLaunchKernelGGL((depth_start_kernel<O, W, double>), dim3(spectral_blocks), dim3(256), 0, ctx->stream, dt,
                           order, labels, off, g->neighbors, w, seed, degree, x, p, scanned);
        for (int step = 0; step < 64; ++step) {
            hipLaunchKernelGGL((depth_step_kernel<O, W, double>), dim3(spectral_blocks), dim3(256), 0, ctx->stream, dt,
                               order, labels, off, g->neighbors, w, degree, x, y, p, q);
            std::swap(x, y);
            std::swap(p, q);
        }
        hipLaunchKernelGGL(depth_normalize_kernel, dim3(blocks), dim3(256), 0, ctx->stream, count, ids, x, p,
                           spectral_blocks);
        GPART_LAUNCH_CHECK();
    } else {
        hipLaunchKernelGGL((spectral_start_kernel<O, W>), dim3(spectral_blocks), dim3(256), 0, ctx->stream, count, ids,
                           labels, task->first_part, off, g->neighbors, w, degree, x,
                           seed ^ static_cast<unsigned>(task->first_part), partials.get(), scanned);
        hipLaunchKernelGGL(finish_moments_kernel, dim3(1), dim3(256), 0, ctx->stream, spectral_blocks, partials.get(),
                           norm.get());
        GPART_LAUNCH_CHECK();
        for (int iteration = 0; iteration <= 64; ++iteration) {
            hipLaunchKernelGGL(normalize_kernel, dim3(blocks), dim3(256), 0, ctx->stream, count, ids, x, norm.get());
            if (iteration == 64) break;
            hipLaunchKernelGGL((spectral_step_kernel<O, W, double>), dim3(spectral_blocks), dim3(256), 0, ctx->stream,
                               count, ids, labels, task->first_part, off, g->neighbors, w, degree, x, y, partials.get());
            hipLaunchKernelGGL(finish_moments_kernel, dim3(1), dim3(256), 0, ctx->stream, spectral_blocks, partials.get(),
                               norm.get());
            GPART_LAUNCH_CHECK();
            std::swap(x, y);
        }
    }
    profile_end(ctx, GPART_PROFILE_SPECTRAL, 0.0);
    if (ctx->profile[GPART_PROFILE_SPECTRAL].enabled)
        profile_add_bytes(ctx, GPART_PROFILE_SPECTRAL,
                          64.0 * step_bytes(count, 1, static_cast<double>(read_scalar(ctx, entries.get())), sizeof(O),
                                            sizeof(W), sizeof(double)));
    // (x, id) total order: stable sort by id, then stable sort by x
    Scratch<std::uint64_t> keys(ctx, count), keys_alt(ctx, count), vals(ctx, count), vals_alt(ctx, count);
    hipLaunchKernelGGL(sort_keys_kernel, dim3(blocks), dim3(256), 0, ctx->stream, count, ids, x, keys.get(), vals.get(),
                       true);
    GPART_LAUNCH_CHECK();
    std::uint64_t* cur_v = vals.get();
    if (radix_sort_pairs(ctx, keys.get(), keys_alt.get(), vals.get(), vals_alt.get(), count, 0, 31))
        cur_v = vals_alt.get();
    hipLaunchKernelGGL(copy_ids_kernel, dim3(blocks), dim3(256), 0, ctx->stream, count, cur_v, ids);
    hipLaunchKernelGGL(sort_keys_kernel, dim3(blocks), dim3(256), 0, ctx->stream, count, ids, x, keys.get(), vals.get(),
                       false);
    GPART_LAUNCH_CHECK();
    cur_v = vals.get();
    if (radix_sort_pairs(ctx, keys.get(), keys_alt.get(), vals.get(), vals_alt.get(), count, 0, 64))
        cur_v = vals_alt.get();
    hipLaunchKernelGGL(copy_ids_kernel, dim3(blocks), dim3(256), 0, ctx->stream, count, cur_v, ids);
    GPART_LAUNCH_CHECK();
    device_scan<std::uint64_t, SumOp<std::uint64_t>>(ctx, OrderWeightLoad{ids, vertex_weights},
                                                      InclusiveStore<std::uint64_t>{prefix}, count,
                                                      SumOp<std::uint64_t>{});
    // x now holds the final coordinates (the caller's x pointer after an even swap count)
}

}  // namespace
}  // namespace gpart_hip

using namespace gpart_hip;

extern "C" {

int gpart_spectral_task(gpart_ctx* ctx, const gpart_csr_view* g, const int32_t* labels, int32_t* order,
                        const uint64_t* vertex_weights, const gpart_bisect_task* task, uint32_t seed, double* x,
                        double* y, double* degree, uint64_t* prefix) {
    return guarded([&] {
        if (g->width == GPART_WIDTH_STANDARD)
            plain_task<std::int32_t, std::uint32_t>(ctx, g, labels, order, vertex_weights, task, seed, x, y, degree,
                                                    prefix);
        else
            plain_task<std::int64_t, std::uint64_t>(ctx, g, labels, order, vertex_weights, task, seed, x, y, degree,
                                                    prefix);
    });
}

int gpart_spectral_assign(gpart_ctx* ctx, const int32_t* order, const gpart_bisect_task* task, int32_t boundary,
                          int32_t left_parts, int32_t* labels) {
    return guarded([&] {
        const int count = task->count;
        if (count <= 0) return;
        hipLaunchKernelGGL(assign_split_kernel, dim3((count + 255) / 256), dim3(256), 0, ctx->stream, count,
                           order + task->begin, boundary, task->first_part, task->first_part + left_parts, labels);
        GPART_LAUNCH_CHECK();
    });
}

int64_t gpart_spectral_depth_max_task(void) { return kMaxBatchedTask; }

int gpart_spectral_depth(gpart_ctx* ctx, const gpart_csr_view* g, int32_t* labels, int32_t* order,
                         const uint64_t* vertex_weights, const gpart_bisect_task* tasks, int32_t task_count,
                         uint32_t seed, uint64_t capacity, int precision, double* coords, gpart_bisect_task* next,
                         int32_t* next_count, int32_t* status) {
    return guarded([&] {
        *next_count = 0;
        *status = 0;
        if (task_count <= 0) return;
        if (task_count > kMaxDepthTasks) throw Error(GPART_ERR_INVALID_ARGUMENT, "too many tasks in one depth");
        DepthTasks dt{};
        dt.count = task_count;
        dt.first_block[0] = 0;
        for (int t = 0; t < task_count; ++t) {
            if (tasks[t].count < 1 || tasks[t].count > kMaxBatchedTask)
                throw Error(GPART_ERR_INVALID_ARGUMENT, "batched bisection task size out of range");
            dt.task[t] = tasks[t];
            dt.first_block[t + 1] = dt.first_block[t] + (tasks[t].count + 7) / 8;
        }
        const int blocks = dt.first_block[task_count];
        const std::int64_t n = g->n;
        Scratch<double> degree(ctx, n), xa(ctx, n), xb(ctx, n);
        Scratch<Moments> pa(ctx, blocks), pb(ctx, blocks);
        // next_count and status (two ints), then the scanned CSR entries
        Scratch<unsigned long long> counters(ctx, 2);
        int* next_and_status = reinterpret_cast<int*>(counters.get());
        unsigned long long* entries = ctx->profile[GPART_PROFILE_SPECTRAL].enabled ? counters.get() + 1 : nullptr;
        int vertices = 0;
        for (int t = 0; t < task_count; ++t) vertices += tasks[t].count;
        auto launch = [&](auto o_tag, auto w_tag, auto t_tag) {
            using O = decltype(o_tag);
            using W = decltype(w_tag);
            using T = decltype(t_tag);
            const auto* off = static_cast<const O*>(g->offsets);
            const auto* w = static_cast<const W*>(g->edge_weights);
            T* x = reinterpret_cast<T*>(xa.get());
            T* y = reinterpret_cast<T*>(xb.get());
            Moments* p = pa.get();
            Moments* q = pb.get();
            hipLaunchKernelGGL((depth_start_kernel<O, W, T>), dim3(blocks), dim3(256), 0, ctx->stream, dt, order,
                               labels, off, g->neighbors, w, seed, degree.get(), x, p, entries);
            for (int step = 0; step < 64; ++step) {
                hipLaunchKernelGGL((depth_step_kernel<O, W, T>), dim3(blocks), dim3(256), 0, ctx->stream, dt, order,
                                   labels, off, g->neighbors, w, degree.get(), x, y, p, q);
                std::swap(x, y);
                std::swap(p, q);
            }
            hipLaunchKernelGGL((depth_finish_kernel<T>), dim3(task_count), dim3(kBatchThreads), 0, ctx->stream, dt,
                               labels, order, vertex_weights, capacity, x, p, coords, next, next_and_status,
                               next_and_status + 1);
            GPART_LAUNCH_CHECK();
        };
        // one workgroup per task where every task is small and sparse enough
        SoloTasks solo{};
        solo.count = task_count;
        bool alone = true;
        for (int t = 0; t < task_count; ++t) {
            const double share = static_cast<double>(g->m) * tasks[t].count / static_cast<double>(n);
            alone = alone && share <= kSoloEntries;
            solo.task[t] = tasks[t];
        }
        Scratch<int> position(ctx, alone ? n : 0), refused(ctx, alone ? task_count : 0);
        Scratch<std::uint64_t> slot(ctx, alone ? std::int64_t{task_count} * kSoloRows * kWave : 0);
        auto launch_solo = [&](auto o_tag, auto w_tag, auto t_tag) {
            using O = decltype(o_tag);
            using W = decltype(w_tag);
            using T = decltype(t_tag);
            const auto* off = static_cast<const O*>(g->offsets);
            const auto* w = static_cast<const W*>(g->edge_weights);
            hipLaunchKernelGGL((depth_measure_kernel<O, W>), dim3(task_count), dim3(kSoloThreads), 0, ctx->stream, solo,
                               order, off, w, refused.get(), counters.get());
            hipLaunchKernelGGL((depth_solo_kernel<O, W, T>), dim3(task_count), dim3(kSoloThreads), 0, ctx->stream, solo,
                               refused.get(), labels, order, off, g->neighbors, w, vertex_weights, seed, capacity,
                               coords, position.get(), slot.get(), next, next_and_status, next_and_status + 1, entries);
            GPART_LAUNCH_CHECK();
        };
        const bool fp32 = precision == GPART_SPECTRAL_FP32;
        unsigned long long h[2];
        int ns[2];
        auto run = [&](auto&& form) {
            profile_begin(ctx, GPART_PROFILE_SPECTRAL);
            const bool standard = g->width == GPART_WIDTH_STANDARD;
            if (standard && fp32) form(std::int32_t{}, std::uint32_t{}, float{});
            else if (standard) form(std::int32_t{}, std::uint32_t{}, double{});
            else if (fp32) form(std::int64_t{}, std::uint64_t{}, float{});
            else form(std::int64_t{}, std::uint64_t{}, double{});
            profile_end(ctx, GPART_PROFILE_SPECTRAL, 0.0);
            read_back(ctx, h, counters.get(), sizeof(h));
            std::memcpy(ns, h, sizeof(ns));
        };
        if (alone) run(launch_solo);
        if (!alone || ns[1] == kSoloRefused) {
            fill_bytes(ctx, counters.get(), 0, 16);
            run(launch);
        }
        *next_count = ns[0];
        *status = ns[1];
        const std::size_t o_size = g->width == GPART_WIDTH_STANDARD ? 4 : 8;
        profile_add_bytes(ctx, GPART_PROFILE_SPECTRAL,
                          64.0 * step_bytes(vertices, task_count, static_cast<double>(h[1]), o_size, o_size,
                                            fp32 ? sizeof(float) : sizeof(double)));
    });
}

}  // extern "C"
