// Shared host/device helpers for the C-IPC HIP library: error handling, grow-only
// device buffers, launch helpers and the device-primitive entry points (scan, radix
// sort, deterministic reductions) implemented in prims.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>
#include <stdexcept>
#include <vector>

namespace cipc {

struct HipError : std::runtime_error {
    int code;
    HipError(const std::string& m, int c) : std::runtime_error(m), code(c) {}
};

#define CIPC_HIP(call)                                                                          \
    do {                                                                                        \
        hipError_t e_ = (call);                                                                 \
        if (e_ != hipSuccess)                                                                   \
            throw ::cipc::HipError(std::string(#call) + ": " + hipGetErrorString(e_), (int)e_); \
    } while (0)

#define CIPC_LAUNCH_CHECK() CIPC_HIP(hipGetLastError())

constexpr int kBlock = 256;
inline int nblocks(long n, int bs = kBlock) { return (int)((n + bs - 1) / bs); }
// Grow-only device allocation; contents are not preserved on growth.
template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t cap = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { if (p) (void)hipFree(p); }
    T* ensure(size_t n) {
        if (n <= cap && p) return p;
        if (p) CIPC_HIP(hipFree(p));
        p = nullptr;
        size_t c = n < 64 ? 64 : n + n / 4;
        CIPC_HIP(hipMalloc(&p, c * sizeof(T)));
        cap = c;
        return p;
    }
    T* ensure_exact(size_t n) {
        if (n <= cap && p) return p;
        if (p) CIPC_HIP(hipFree(p));
        p = nullptr;
        size_t c = n < 1 ? 1 : n;
        CIPC_HIP(hipMalloc(&p, c * sizeof(T)));
        cap = c;
        return p;
    }
    operator T*() const { return p; }
};

template <class T>
inline void upload(DevBuf<T>& b, const T* h, size_t n, hipStream_t s) {
    b.ensure_exact(n);
    if (n) CIPC_HIP(hipMemcpyAsync(b.p, h, n * sizeof(T), hipMemcpyHostToDevice, s));
}
template <class T>
inline void upload(DevBuf<T>& b, const std::vector<T>& h, hipStream_t s) { upload(b, h.data(), h.size(), s); }

// Scratch memory shared by the primitives.
struct PrimWork {
    DevBuf<uint32_t> scanBlocks, scanBlocks2, hist, histScan;
    DevBuf<uint64_t> keyAlt;
    DevBuf<uint32_t> valAlt;
    DevBuf<double> redPartial;
    DevBuf<uint32_t> u32tmp;
};

// exclusive prefix sum of n uint32 values; total (if not null) written to device memory
void scan_exclusive(const uint32_t* in, uint32_t* out, long n, uint32_t* total, PrimWork& w, hipStream_t s);
// stable sort of the keys with their positions 0, 1, ..., on the low `bits` bits of the keys,
// no bit set above them; `vals` is room for n positions.  The sorted pairs are either in
// `keys` and `vals` or in the work buffers, valid until the next sort.
struct SortedPairs {
    uint64_t* keys;
    uint32_t* vals;
};
SortedPairs radix_sort_pairs(uint64_t* keys, uint32_t* vals, long n, int bits, PrimWork& w, hipStream_t s);
// deterministic sums: chunks of 256 values folded by halving strides, chunk partials
// added in chunk order by one thread; result written to device memory `out`
void chunk_sum(const double* in, long n, double* out, PrimWork& w, hipStream_t s);
// sum of per-block partials already in device memory (fixed order)
void sum_partials(const double* partials, int n, double* out, hipStream_t s);

// a slot in an output list for every active lane of the wave: the active lanes are found
// by a ballot, the lowest adds their count to the counter, and each lane takes base + its
// rank among them (one atomic per wave; the slot order is arbitrary)
__device__ __forceinline__ uint32_t wave_reserve(uint32_t* cnt) {
    const uint64_t act = __ballot(1);
    const int lane = (int)__lane_id();
    const int leader = __ffsll((unsigned long long)act) - 1;
    const uint32_t rank = (uint32_t)__popcll(act & ((1ull << lane) - 1ull));
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(cnt, (uint32_t)__popcll(act));
    base = (uint32_t)__shfl((int)base, leader, 64);
    return base + rank;
}

// device reductions inside kernels.  Lanes exchange values through DPP moves (VALU) instead
// of LDS permutes (__shfl_xor): a dependent step costs a few cycles instead of an LDS round
// trip, which is what the short PCG kernels' reductions consist of.  Measured (us per
// launch): PCG SpMV on 4,247 vertices 4.8 -> 4.1, restriction to 612 aggregates 6.4 -> 4.8.
// All lanes of the wave must be active.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
// sum over aligned groups of LANES (2, 4, 8 or 16) lanes, in every lane of the group.  A row
// of 16: rotations by 8, 4, 2, 1 -- after the rotation by 8 the values repeat every 8 lanes,
// so each next rotation meets the partner of an xor butterfly.  Eight lanes start with the
// mirrored half row (lane i and 7 - i, another association than lanes ^ 4), four and two with
// the quad permutations (lanes ^ 2, lanes ^ 1).  Every lane of a group adds the same pairs in
// every step, so all hold the same bits, and a launch shape gives the same bits every time.
template <int LANES, class V>
__device__ __forceinline__ V lane_sum(V v) {
    static_assert(LANES == 2 || LANES == 4 || LANES == 8 || LANES == 16, "");
    if (LANES == 16) {
        v += dpp_move<0x128>(v);
        v += dpp_move<0x124>(v);
        v += dpp_move<0x122>(v);
        v += dpp_move<0x121>(v);
        return v;
    }
    if (LANES == 8) v += dpp_move<0x141>(v);
    if (LANES >= 4) v += dpp_move<0x4E>(v);
    v += dpp_move<0xB1>(v);
    return v;
}
// v + (v of lane ^ 32), v + (v of lane ^ 16): the swap instructions exchange halves (rows)
// between two registers, here two copies of v
__device__ __forceinline__ double add_half(double v) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double add_row(double v) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// sum over the wave, the same value in every lane: the xor butterfly 32, 16, 8, 4, 2, 1
__device__ __forceinline__ double wave_sum(double v) { return lane_sum<16>(add_row(add_half(v))); }
// block-wide sum for blockDim = 256; result valid in thread 0.  Fixed association order.
__device__ __forceinline__ double block_sum_256(double v, double* lds /*[4]*/) {
    v = wave_sum(v);
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) lds[wid] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0) r = (lds[0] + lds[1]) + (lds[2] + lds[3]);
    __syncthreads();
    return r;
}
__device__ __forceinline__ double block_min_256(double v, double* lds) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { double u = __shfl_xor(v, o, 64); v = u < v ? u : v; }
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) lds[wid] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0) {
        r = lds[0];
        for (int i = 1; i < 4; ++i) r = lds[i] < r ? lds[i] : r;
    }
    __syncthreads();
    return r;
}

}  // namespace cipc
