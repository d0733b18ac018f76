// common.hpp -- device helpers shared by the gfx950 kernels.
//
// CDNA4 executes 64-lane wavefronts. Kernels here map a vertex to a "group" of
// G lanes (G in {4, 8, 16, 32, 64}) or to a whole workgroup; group reductions use
// DPP moves where the pattern has one, else width-limited shuffles.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace gpart_hip {

constexpr int kWave = 64;
constexpr std::int32_t kSclpInvalid = 0x7fffffff;
constexpr std::uint64_t kInvalidKey = ~std::uint64_t{0};

// The public "lowbias32" integer hash.
__device__ __forceinline__ std::uint32_t mix32(std::uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352dU;
    x ^= x >> 15;
    x *= 0x846ca68bU;
    return x ^ (x >> 16);
}

__device__ __forceinline__ int lane_id() { return static_cast<int>(threadIdx.x & (kWave - 1)); }

__device__ __forceinline__ std::uint64_t lanemask_lt() {
    const int lane = lane_id();
    return lane == 0 ? 0ULL : (~0ULL >> (64 - lane));
}

// Lane exchanges. __shfl_* go through the LDS crossbar (ds_bpermute, two per 64-bit
// value and step); DPP operands move data between neighbouring lanes inside a
// vector instruction. Patterns with a DPP form use it: xor 1 and 2 (quad_perm),
// xor 8 (rotation by half a row of 16) and the prefix steps of wave_scan below.
// Every lane that a pattern reads must be active, as with __shfl_*.
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppRowRor8 = 0x128;
constexpr int kDppRowShr1 = 0x111, kDppRowShr2 = 0x112, kDppRowShr4 = 0x114, kDppRowShr8 = 0x118;
constexpr int kDppRowShl = 0x100;  // + 1..15
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143;

// Lanes without a source (and rows outside RowMask) receive 0.
template <int Control, int RowMask = 0xf>
__device__ __forceinline__ unsigned dpp_or_zero(unsigned v) {
    return static_cast<unsigned>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(v), Control, RowMask, 0xf, false));
}
template <int Control, int RowMask = 0xf>
__device__ __forceinline__ unsigned long long dpp_or_zero(unsigned long long v) {
    const unsigned lo = dpp_or_zero<Control, RowMask>(static_cast<unsigned>(v));
    const unsigned hi = dpp_or_zero<Control, RowMask>(static_cast<unsigned>(v >> 32));
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

// Inclusive prefix sums over the wave: four steps inside each row of 16 lanes, then
// the last lane of rows 0 and 2 into rows 1 and 3, then lane 31 into rows 2 and 3.
// Every lane of the wave must be active.
template <typename T>
__device__ __forceinline__ T wave_scan(T v) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4- or 8-byte integers");
    using U = std::conditional_t<sizeof(T) == 4, unsigned, unsigned long long>;
    U x = static_cast<U>(v);
    x += dpp_or_zero<kDppRowShr1>(x);
    x += dpp_or_zero<kDppRowShr2>(x);
    x += dpp_or_zero<kDppRowShr4>(x);
    x += dpp_or_zero<kDppRowShr8>(x);
    x += dpp_or_zero<kDppBcast15, 0xa>(x);
    x += dpp_or_zero<kDppBcast31, 0xc>(x);
    return static_cast<T>(x);
}

// Lane `src`'s value, the same src on every lane.
__device__ __forceinline__ unsigned read_lane(unsigned v, int src) {
    return static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v), src));
}
__device__ __forceinline__ unsigned long long read_lane(unsigned long long v, int src) {
    const unsigned lo = read_lane(static_cast<unsigned>(v), src);
    const unsigned hi = read_lane(static_cast<unsigned>(v >> 32), src);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

// __shfl_xor(v, mask, width) for mask < width; mask is a constant after inlining.
__device__ __forceinline__ unsigned lane_xor(unsigned v, int mask, int width) {
    if (mask == 1) return dpp_or_zero<kDppXor1>(v);
    if (mask == 2) return dpp_or_zero<kDppXor2>(v);
    if (mask == 8) return dpp_or_zero<kDppRowRor8>(v);
    return __shfl_xor(v, mask, width);
}

__device__ __forceinline__ unsigned long long shfl_u64(unsigned long long v, int src, int width) {
    const unsigned lo = __shfl(static_cast<unsigned>(v), src, width);
    const unsigned hi = __shfl(static_cast<unsigned>(v >> 32), src, width);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

__device__ __forceinline__ unsigned long long shfl_xor_u64(unsigned long long v, int mask, int width) {
    const unsigned lo = lane_xor(static_cast<unsigned>(v), mask, width);
    const unsigned hi = lane_xor(static_cast<unsigned>(v >> 32), mask, width);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

__device__ __forceinline__ unsigned long long shfl_up_u64(unsigned long long v, int delta, int width) {
    const unsigned lo = __shfl_up(static_cast<unsigned>(v), delta, width);
    const unsigned hi = __shfl_up(static_cast<unsigned>(v >> 32), delta, width);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

template <int G>
__device__ __forceinline__ unsigned long long group_sum_u64(unsigned long long v) {
    if constexpr (G == kWave) return read_lane(wave_scan(v), kWave - 1);
#pragma unroll
    for (int m = G / 2; m > 0; m /= 2) v += shfl_xor_u64(v, m, G);
    return v;
}

template <int G>
__device__ __forceinline__ long long group_sum_i64(long long v) {
    return static_cast<long long>(group_sum_u64<G>(static_cast<unsigned long long>(v)));
}

template <int G>
__device__ __forceinline__ unsigned long long group_max_u64(unsigned long long v) {
#pragma unroll
    for (int m = G / 2; m > 0; m /= 2) {
        const auto o = shfl_xor_u64(v, m, G);
        v = o > v ? o : v;
    }
    return v;
}

template <int G>
__device__ __forceinline__ bool group_any(bool p) {
    int v = p ? 1 : 0;
#pragma unroll
    for (int m = G / 2; m > 0; m /= 2) v |= __shfl_xor(v, m, G);
    return v != 0;
}

// Width traits: Standard = int32 offsets / uint32 weights, Big = int64 / uint64.
template <int Width>
struct WidthTypes;
template <>
struct WidthTypes<0> {
    using O = std::int32_t;
    using W = std::uint32_t;
};
template <>
struct WidthTypes<1> {
    using O = std::int64_t;
    using W = std::uint64_t;
};

inline int ceil_div_int(std::int64_t a, std::int64_t b) { return static_cast<int>((a + b - 1) / b); }

}  // namespace gpart_hip
