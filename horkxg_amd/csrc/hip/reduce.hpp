// reduce.hpp -- contention-free device-wide reductions.
//
// A single global address updated by every wave serialises in L2 (a CAS loop
// per wave costs tens of milliseconds at 10^5 waves). Reductions here run a
// capped grid with grid-stride loops, combine inside each workgroup through LDS
// and store one partial per workgroup; the workgroup that finishes last folds the
// partials and publishes the results to the host, which waits for them. One launch
// for partials, fold and read-back, and for several reductions over the same values.
#pragma once

#include "internal.hpp"

#include <algorithm>

namespace gpart_hip {

constexpr int kReduceThreads = 256;
constexpr int kReduceMaxBlocks = 2048;
constexpr int kReduceLoads = 4;  // of a thread, under way together

// Op: T identity(); T operator()(T, T).
template <typename T, typename Op>
__device__ T block_reduce(T value, Op op, T* shared) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
#pragma unroll
    for (int m = kWave / 2; m > 0; m /= 2) {
        T other;
        static_assert(sizeof(T) == 8, "block_reduce handles 8-byte values");
        const auto bits = shfl_xor_u64(*reinterpret_cast<unsigned long long*>(&value), m, kWave);
        *reinterpret_cast<unsigned long long*>(&other) = bits;
        value = op(value, other);
    }
    if (lane == 0) shared[wave] = value;
    __syncthreads();
    T total = op.identity();
    if (threadIdx.x == 0)
        for (int w = 0; w < static_cast<int>(blockDim.x) / kWave; ++w) total = op(total, shared[w]);
    return total;  // valid in thread 0
}

struct MaxU64 {
    __device__ __forceinline__ unsigned long long identity() const { return 0; }
    __device__ __forceinline__ unsigned long long operator()(unsigned long long a, unsigned long long b) const {
        return a > b ? a : b;
    }
};
struct MinU64 {
    __device__ __forceinline__ unsigned long long identity() const { return ~0ULL; }
    __device__ __forceinline__ unsigned long long operator()(unsigned long long a, unsigned long long b) const {
        return a < b ? a : b;
    }
};
struct SumU64 {
    __device__ __forceinline__ unsigned long long identity() const { return 0; }
    __device__ __forceinline__ unsigned long long operator()(unsigned long long a, unsigned long long b) const {
        return a + b;
    }
};
// Saturating at UINT64_MAX (CheckedSum, src/initial_partition_gpu.cu:31-35).
struct CheckedSumU64 {
    __device__ __forceinline__ unsigned long long identity() const { return 0; }
    __device__ __forceinline__ unsigned long long operator()(unsigned long long a, unsigned long long b) const {
        return ~0ULL - a < b ? ~0ULL : a + b;
    }
};
// Saturating at INT64_MAX/2 + 1 (RefinementWeightSum, src/refine.cu:367-372).
struct LimitedSumU64 {
    static constexpr unsigned long long kLimit = 0x7fffffffffffffffULL / 2;
    __device__ __forceinline__ unsigned long long identity() const { return 0; }
    __device__ __forceinline__ unsigned long long operator()(unsigned long long a, unsigned long long b) const {
        return a > kLimit || b > kLimit || a > kLimit - b ? kLimit + 1 : a + b;
    }
};

template <typename W>
struct WidenLoad {
    const W* data;
    __device__ __forceinline__ unsigned long long operator()(std::int64_t i) const {
        return static_cast<unsigned long long>(data[i]);
    }
};

// Calls use(load) for the weights of a graph of this width.
template <typename Use>
void with_weights(int width, const void* weights, Use use) {
    if (width == GPART_WIDTH_STANDARD)
        use(WidenLoad<std::uint32_t>{static_cast<const std::uint32_t*>(weights)});
    else
        use(WidenLoad<std::uint64_t>{static_cast<const std::uint64_t*>(weights)});
}

struct NonzeroLoad {
    const unsigned long long* data;
    __device__ __forceinline__ unsigned long long operator()(std::int64_t i) const { return data[i] != 0; }
};

// The values in words 1.. are complete: makes the publication visible. One thread.
__device__ __forceinline__ void publish_sequence(const Publication& to) {
    __threadfence_system();
    const unsigned long long seq = *to.counter + 1;
    *to.counter = seq;
    __hip_atomic_store(to.words, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <typename... Ops>
struct Reduction {
    static constexpr int kValues = sizeof...(Ops);
    unsigned long long v[kValues];
    __device__ __forceinline__ Reduction() : v{Ops{}.identity()...} {}
    // the same value for each op, or a partial of each
    __device__ __forceinline__ void add(unsigned long long x) {
        int j = 0;
        ((v[j] = Ops{}(v[j], x), ++j), ...);
    }
    template <typename Partial>
    __device__ __forceinline__ void fold(Partial partial) {
        int j = 0;
        ((v[j] = Ops{}(v[j], partial(j)), ++j), ...);
    }
    // over the workgroup, valid in thread 0
    __device__ __forceinline__ void combine(unsigned long long (*shared)[kReduceThreads / kWave]) {
        int j = 0;
        ((v[j] = block_reduce(v[j], Ops{}, shared[j]), ++j), ...);
    }
};

// `known` (words of earlier kernels) and the reductions of n loaded values to the host.
template <typename Load, typename... Ops>
__global__ void __launch_bounds__(kReduceThreads) reduce_publish_kernel(Load load, std::int64_t n,
                                                                        unsigned long long* partials,
                                                                        const unsigned long long* known, int known_count,
                                                                        Publication to) {
    using R = Reduction<Ops...>;
    __shared__ unsigned long long shared[R::kValues][kReduceThreads / kWave];
    __shared__ bool last;
    R acc;
    const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += kReduceLoads * stride) {
        unsigned long long x[kReduceLoads];
#pragma unroll
        for (int u = 0; u < kReduceLoads; ++u) x[u] = i + u * stride < n ? load(i + u * stride) : 0;
#pragma unroll
        for (int u = 0; u < kReduceLoads; ++u)
            if (i + u * stride < n) acc.add(x[u]);
    }
    acc.combine(shared);
    if (gridDim.x > 1) {
        unsigned long long* arrivals = to.counter + 1;
        if (threadIdx.x == 0) {
            for (int j = 0; j < R::kValues; ++j)
                __hip_atomic_store(partials + blockIdx.x * R::kValues + j, acc.v[j], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_s_waitcnt(0);
            last = __hip_atomic_fetch_add(arrivals, 1ULL, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 == gridDim.x;
        }
        __syncthreads();
        if (!last) return;
        acc = R();
        for (unsigned b = threadIdx.x; b < gridDim.x; b += blockDim.x)
            acc.fold([&](int j) {
                return __hip_atomic_load(partials + b * R::kValues + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            });
        acc.combine(shared);
        if (threadIdx.x == 0) __hip_atomic_store(arrivals, 0ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (threadIdx.x == 0) {
        for (int j = 0; j < known_count; ++j) to.words[1 + j] = known[j];
        for (int j = 0; j < R::kValues; ++j) to.words[1 + known_count + j] = acc.v[j];
        publish_sequence(to);
    }
}

// The reductions of n loaded values (the identities for none) after known_count device
// words, to the host. Waits for them.
template <typename... Ops, typename Load>
void reduce_read(gpart_ctx* ctx, Load load, std::int64_t n, unsigned long long* out,
                 const unsigned long long* known = nullptr, int known_count = 0) {
    constexpr std::int64_t kTile = kReduceThreads * kReduceLoads;
    const auto blocks =
        static_cast<int>(std::min<std::int64_t>(std::max<std::int64_t>((n + kTile - 1) / kTile, 1), kReduceMaxBlocks));
    Scratch<unsigned long long> partials(ctx, blocks > 1 ? blocks * static_cast<std::int64_t>(sizeof...(Ops)) : 0);
    hipLaunchKernelGGL((reduce_publish_kernel<Load, Ops...>), dim3(blocks), dim3(kReduceThreads), 0, ctx->stream, load,
                       n, partials.get(), known, known_count, publication(ctx));
    GPART_LAUNCH_CHECK();
    read_published(ctx, out, (known_count + sizeof...(Ops)) * 8);
}

}  // namespace gpart_hip
