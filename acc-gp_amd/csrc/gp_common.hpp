// Shared definitions for the gfx950 partitioner: error handling, wave64
// helpers and the hash used by every deterministic tie-break.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

namespace gp {

struct HipError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

#define GP_HIP(call)                                                                   \
    do {                                                                               \
        const hipError_t gp_err__ = (call);                                            \
        if (gp_err__ != hipSuccess)                                                    \
            throw ::gp::HipError(std::string("HIP failure at ") + __FILE__ + ":" +     \
                                 std::to_string(__LINE__) + " for " #call ": " +       \
                                 hipGetErrorString(gp_err__));                         \
    } while (0)

// Kernel launches made by the calling host thread: every launch site goes
// through GP_LAUNCH_CHECK, and a partition reads the count before and after.
std::uint64_t& thread_launches();
#define GP_LAUNCH_CHECK()              \
    do {                               \
        ++::gp::thread_launches();     \
        GP_HIP(hipGetLastError());     \
    } while (0)

constexpr int kWave = 64;          // CDNA wavefront width
constexpr int kMaxParts = 128;
constexpr std::int32_t kInvalid = 0x7fffffff;

inline int ceil_div(std::int64_t a, std::int64_t b) { return static_cast<int>((a + b - 1) / b); }

// mix32: the integer hash behind every tie-break (src/coarsen.cu:173-179).
__host__ __device__ inline std::uint32_t mix32(std::uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352dU;
    x ^= x >> 15;
    x *= 0x846ca68bU;
    return x ^ (x >> 16);
}

__device__ inline std::uint64_t ew_at(const std::uint32_t* ew, std::int64_t e) {
    return ew ? static_cast<std::uint64_t>(ew[e]) : 1ULL;
}

__device__ inline int lane_id() { return static_cast<int>(__lane_id()); }

// Orders LDS traffic between lanes of one wavefront.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Barrier of the block after which every store made by its threads before it
// has left the CU, so that a release by one of them covers them all.  (A
// release by every wave writes the XCD's L2 back once per wave: an edge cut
// whose 16-wave blocks ended that way took 580 us instead of its own time.)
__device__ inline void block_stores_done() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// ------------------------------------------------ lane exchanges
// The value of lane ^ d (d a power of two below 64) without the LDS crossbar
// that __shfl_xor goes through: DPP within rows of 16 lanes (quad_perm for 1
// and 2, half mirror i <-> 7 - i followed by the quad mirror for 4, rotation
// by 8 for 8), row and half-wave swaps above (v_permlane16_swap_b32 and
// v_permlane32_swap_b32 on gfx950).  d has to be a constant after unrolling;
// the lanes that exchange have to be active.  The crossbar is one unit for a
// CU's four SIMDs: a 512-entry bitonic row sort issues 624 of these moves, and
// the contraction of rows of 257 to 512 entries (R-MAT scale 20) took 33 us a
// launch with shuffles and takes 26, their affinity on scale 18 28 and 24.
constexpr int kDppQuadXor1 = 0xB1;
constexpr int kDppQuadXor2 = 0x4E;
constexpr int kDppQuadMirror = 0x1B;
constexpr int kDppRowHalfMirror = 0x141;
constexpr int kDppRowRor8 = 0x128;

template <int Ctrl>
__device__ inline int dpp_word(int x) {
    return __builtin_amdgcn_update_dpp(x, x, Ctrl, 0xf, 0xf, false);
}
__device__ inline int lane_xor_word(int x, int d) {
    switch (d) {
        case 1: return dpp_word<kDppQuadXor1>(x);
        case 2: return dpp_word<kDppQuadXor2>(x);
        case 4: return dpp_word<kDppQuadMirror>(dpp_word<kDppRowHalfMirror>(x));
        case 8: return dpp_word<kDppRowRor8>(x);
        case 16: {
            // [0]: rows 0 0 2 2, [1]: rows 1 1 3 3
            const auto r = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
            return (int)((lane_id() & 16) ? r[0] : r[1]);
        }
        default: {
            // [0]: the lower half twice, [1]: the upper half twice
            const auto r = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
            return (int)((lane_id() & 32) ? r[0] : r[1]);
        }
    }
}
template <typename T>
__device__ inline T lane_xor(const T& v, int d) {
    static_assert(sizeof(T) % 4 == 0, "lane moves are 32-bit words");
    constexpr int words = sizeof(T) / 4;
    int in[words], out[words];
    __builtin_memcpy(in, &v, sizeof(T));
#pragma unroll
    for (int i = 0; i < words; ++i) out[i] = lane_xor_word(in[i], d);
    T r;
    __builtin_memcpy(&r, out, sizeof(T));
    return r;
}

template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
    for (int d = kWave / 2; d; d >>= 1) v += lane_xor(v, d);
    return v;
}
template <typename T>
__device__ inline T wave_max(T v) {
#pragma unroll
    for (int d = kWave / 2; d; d >>= 1) {
        const T o = lane_xor(v, d);
        v = o > v ? o : v;
    }
    return v;
}
// Reduction within aligned groups of W lanes (W divides 64).
template <int W, typename T>
__device__ inline T group_sum(T v) {
#pragma unroll
    for (int d = W / 2; d; d >>= 1) v += lane_xor(v, d);
    return v;
}

// Every lane gets combine() over the 64 lanes' values.  combine must be
// associative and commutative (a sum, or the better of two under a total
// order), so the result does not depend on the pairing.  Called from
// converged control flow only.
template <typename T, typename Combine>
__device__ inline T wave_allreduce(T v, Combine combine) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) v = combine(v, lane_xor(v, d));
    return v;
}

struct PlusU64 {
    __device__ unsigned long long operator()(unsigned long long x, unsigned long long y) const { return x + y; }
};
struct PlusI64 {
    __device__ std::int64_t operator()(std::int64_t x, std::int64_t y) const { return x + y; }
};

}  // namespace gp
