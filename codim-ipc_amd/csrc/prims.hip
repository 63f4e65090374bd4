// Device primitives: exclusive scan, stable LSD radix sort of (key, value) pairs and
// deterministic reductions.  Written for 64-wide wavefronts: within-wave ranking uses
// 64-bit ballots, block-level structures are 256 threads (four waves).
#include "common.hpp"

namespace cipc {

constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = kBlock * SCAN_ITEMS;   // 2048 values per block

__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t v) {
    int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}
// exclusive scan of one value per thread over a 256-thread block; returns block total
__device__ __forceinline__ uint32_t block_excl_scan_u32(uint32_t v, uint32_t& excl, uint32_t* lds /*[4]*/) {
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t inc = wave_incl_scan_u32(v);
    if (lane == 63) lds[wid] = inc;
    __syncthreads();
    uint32_t base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t t = lds[w];
        if (w < wid) base += t;
        total += t;
    }
    __syncthreads();
    excl = base + inc - v;
    return total;
}

__global__ void k_scan_block_sums(const uint32_t* __restrict__ in, long n, uint32_t* __restrict__ sums) {
    __shared__ uint32_t lds[4];
    long base = (long)blockIdx.x * SCAN_TILE;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        long idx = base + (long)i * kBlock + threadIdx.x;
        if (idx < n) s += in[idx];
    }
    uint32_t excl;
    uint32_t tot = block_excl_scan_u32(s, excl, lds);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// single-block exclusive scan of up to any count (serial chunks per thread)
__global__ void k_scan_single(uint32_t* __restrict__ a, long n, uint32_t* __restrict__ total) {
    __shared__ uint32_t lds[4];
    long per = (n + kBlock - 1) / kBlock;
    long b = threadIdx.x * per, e = b + per < n ? b + per : n;
    uint32_t s = 0;
    for (long i = b; i < e; ++i) s += a[i];
    uint32_t excl;
    uint32_t tot = block_excl_scan_u32(s, excl, lds);
    uint32_t run = excl;
    for (long i = b; i < e; ++i) { uint32_t v = a[i]; a[i] = run; run += v; }
    if (threadIdx.x == 0 && total) *total = tot;
}

__global__ void k_scan_apply(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, long n,
                             const uint32_t* __restrict__ blockOff) {
    __shared__ uint32_t lds[4];
    long base = (long)blockIdx.x * SCAN_TILE + (long)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        long idx = base + i;
        v[i] = idx < n ? in[idx] : 0;
        s += v[i];
    }
    uint32_t excl;
    block_excl_scan_u32(s, excl, lds);
    uint32_t run = excl + blockOff[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        long idx = base + i;
        if (idx < n) out[idx] = run;
        run += v[i];
    }
}

// up to kScanSmall values in one workgroup of 1024 threads, 16 consecutive values each: one
// launch instead of three where the launches are the time
constexpr int kScanSmall = 16384;
__global__ __launch_bounds__(1024) void k_scan_small(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int n,
                                                     uint32_t* __restrict__ total) {
    __shared__ uint32_t lds[16];
    const int base = 16 * threadIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t v[16], s = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = base + i < n ? in[base + i] : 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += v[i];
    const uint32_t inc = wave_incl_scan_u32(s);
    if (lane == 63) lds[wid] = inc;
    __syncthreads();
    uint32_t run = inc - s;
#pragma unroll
    for (int w = 0; w < 16; ++w)
        if (w < wid) run += lds[w];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (total && threadIdx.x == 1023) *total = run;
}

void scan_exclusive(const uint32_t* in, uint32_t* out, long n, uint32_t* total, PrimWork& w, hipStream_t s) {
    if (n <= 0) {
        if (total) CIPC_HIP(hipMemsetAsync(total, 0, sizeof(uint32_t), s));
        return;
    }
    if (n <= kScanSmall) {
        hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, in, out, (int)n, total);
        CIPC_LAUNCH_CHECK();
        return;
    }
    int nb = (int)((n + SCAN_TILE - 1) / SCAN_TILE);
    uint32_t* sums = w.scanBlocks.ensure(nb);
    hipLaunchKernelGGL(k_scan_block_sums, dim3(nb), dim3(kBlock), 0, s, in, n, sums);
    CIPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(kBlock), 0, s, sums, (long)nb, total);
    CIPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(kBlock), 0, s, in, out, n, sums);
    CIPC_LAUNCH_CHECK();
}

// ------------------------------------------------------------------ sort
// Least-significant-digit radix sort, digits of up to kMaxDigit bits: the key's bits are
// split evenly, so 18 bits take two passes and 35 bits four (three and five with 8-bit
// digits); the passes' launches and their scans are the time on all but the largest inputs.
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = kBlock * RS_ITEMS;
constexpr int kMaxDigit = 9, kBins = 1 << kMaxDigit, kBinsPer = kBins / kBlock;

__global__ void k_rs_hist(const uint64_t* __restrict__ keys, long n, int shift, uint32_t mask, uint32_t* __restrict__ hist, int nb) {
    __shared__ uint32_t h[kBins];
#pragma unroll
    for (int k = 0; k < kBinsPer; ++k) h[threadIdx.x + k * kBlock] = 0;
    __syncthreads();
    long base = (long)blockIdx.x * RS_TILE;
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i) {
        long idx = base + (long)i * kBlock + threadIdx.x;
        if (idx < n) atomicAdd(&h[(uint32_t)(keys[idx] >> shift) & mask], 1u);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kBinsPer; ++k) {
        const uint32_t d = threadIdx.x + k * kBlock;
        if (d <= mask) hist[(long)d * nb + blockIdx.x] = h[d];
    }
}

// vin == nullptr: the values are the positions 0, 1, ...
__global__ void k_rs_scatter(const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                             uint64_t* __restrict__ kout, uint32_t* __restrict__ vout, long n, int shift, int digitBits,
                             const uint32_t* __restrict__ histScan, int nb) {
    __shared__ uint32_t next[kBins];         // output position of the digit's next key
    __shared__ uint32_t wcnt[4][kBins];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const uint32_t mask = (1u << digitBits) - 1;
#pragma unroll
    for (int k = 0; k < kBinsPer; ++k) {
        const uint32_t d = tid + k * kBlock;
        next[d] = d <= mask ? histScan[(long)d * nb + blockIdx.x] : 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) wcnt[w][d] = 0;
    }
    const uint64_t ltmask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    long base = (long)blockIdx.x * RS_TILE;
    uint64_t key[RS_ITEMS];
    uint32_t val[RS_ITEMS];
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const long idx = base + (long)r * kBlock + tid;
        key[r] = idx < n ? kin[idx] : 0;
        val[r] = idx < n ? (vin ? vin[idx] : (uint32_t)idx) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const bool valid = base + (long)r * kBlock + tid < n;
        const uint32_t dig = (uint32_t)(key[r] >> shift) & mask;
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < digitBits; ++b) {
            uint64_t m = __ballot((dig >> b) & 1u);
            peers &= ((dig >> b) & 1u) ? m : ~m;
        }
        const uint32_t rankInWave = (uint32_t)__popcll(peers & ltmask);
        if (valid && rankInWave == 0) wcnt[wid][dig] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (valid) {
            uint32_t dst = next[dig] + rankInWave;
            for (int k = 0; k < wid; ++k) dst += wcnt[k][dig];
            kout[dst] = key[r];
            vout[dst] = val[r];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kBinsPer; ++k) {
            const uint32_t d = tid + k * kBlock;
            next[d] += (wcnt[0][d] + wcnt[1][d]) + (wcnt[2][d] + wcnt[3][d]);
#pragma unroll
            for (int w = 0; w < 4; ++w) wcnt[w][d] = 0;
        }
        __syncthreads();
    }
}

// Short inputs by counting: an element's place is the number of smaller keys plus the equal
// ones before it.  64 elements per workgroup, each of its four waves compares them with a
// quarter of the keys (uniform addresses: scalar loads); one launch instead of five per
// digit.  kRankSort: keys at most, by the number of digits that the passes would take: the
// counting is quadratic in the keys and does not see their length.  The lines are those of
// whole calls (us, counting / passes), where the card idles between calls:
//   2 digits, gradient by vertex   1,600 slots 122 / 134   3,200 137 / 137   4,800 159 / 143   8,000 180 / 146
//   3 digits, barrier Hessian      3,200 slots 581 / 630   6,400 745 / 746   8,000 813 / 794   16,000 1,229 / 1,094
//   4 digits, constraint set, edge pairs 7,500 (2,400 point-triangle pairs)  338 / 426
//             9,900 (3,100) 385 / 457   15,400 (4,900) 480 / 478   22,100 (7,000) 608 / 530:
//             the edge pairs alone cross near 9,600
// Back to back the counting is a third faster (2 digits cross at 5,000, 3 at 9,600, 4 at
// 15,000, 1 at 1,900), which sets the lines for 1, 5 and 6 digits in proportion.
constexpr long kRankSort[] = {0, 1200, 3200, 6400, 9600, 12800, 16000};
__global__ __launch_bounds__(kBlock) void k_rank_sort(const uint64_t* __restrict__ kin, uint64_t* __restrict__ kout,
                                                      uint32_t* __restrict__ vout, int n) {
    __shared__ uint32_t part[4][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int first = blockIdx.x * 64, i = first + lane;
    const uint64_t mine = i < n ? kin[i] : 0;
    const int per = (n + 3) / 4, j0 = w * per, j1 = min(n, j0 + per);
    // keys before this workgroup's count when not larger, keys behind it when smaller
    uint32_t r = 0;
    const int a = min(max(first, j0), j1), b = min(max(first + 64, j0), j1);
#pragma unroll 8
    for (int j = j0; j < a; ++j) r += kin[j] <= mine;
    for (int j = a; j < b; ++j) r += kin[j] < mine || (kin[j] == mine && j < i);
#pragma unroll 8
    for (int j = b; j < j1; ++j) r += kin[j] < mine;
    part[w][lane] = r;
    __syncthreads();
    if (w != 0 || i >= n) return;
    r = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    kout[r] = mine;
    vout[r] = (uint32_t)i;
}

SortedPairs radix_sort_pairs(uint64_t* keys, uint32_t* vals, long n, int bits, PrimWork& w, hipStream_t s) {
    if (n <= 0) return {keys, vals};
    uint64_t* k2 = w.keyAlt.ensure(n);
    uint32_t* v2 = w.valAlt.ensure(n);
    const int passes = (bits + kMaxDigit - 1) / kMaxDigit, rb = (bits + passes - 1) / passes;
    if (n <= kRankSort[std::min(passes, 6)]) {
        hipLaunchKernelGGL(k_rank_sort, dim3((unsigned)((n + 63) / 64)), dim3(kBlock), 0, s, keys, k2, v2, (int)n);
        CIPC_LAUNCH_CHECK();
        return {k2, v2};
    }
    int nb = (int)((n + RS_TILE - 1) / RS_TILE);
    uint32_t* hist = w.hist.ensure((size_t)nb << rb);
    uint32_t* hs = w.histScan.ensure((size_t)nb << rb);
    uint64_t *ka = keys, *kb = k2;
    uint32_t *va = vals, *vb = v2;
    for (int p = 0; p < passes; ++p) {
        hipLaunchKernelGGL(k_rs_hist, dim3(nb), dim3(kBlock), 0, s, ka, n, rb * p, (1u << rb) - 1, hist, nb);
        CIPC_LAUNCH_CHECK();
        scan_exclusive(hist, hs, (long)nb << rb, nullptr, w, s);
        hipLaunchKernelGGL(k_rs_scatter, dim3(nb), dim3(kBlock), 0, s, ka, p == 0 ? nullptr : va, kb, vb, n, rb * p, rb, hs, nb);
        CIPC_LAUNCH_CHECK();
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    return {ka, va};
}

// ------------------------------------------------------------------ reductions
__global__ void k_chunk_sum(const double* __restrict__ in, long n, double* __restrict__ partial) {
    __shared__ double a[kBlock];
    long idx = (long)blockIdx.x * kBlock + threadIdx.x;
    a[threadIdx.x] = idx < n ? in[idx] : 0.0;
    __syncthreads();
    for (int st = kBlock / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) a[threadIdx.x] += a[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = a[0];
}
// Sequential sum in index order (the order the deterministic reductions define); the
// partials are staged through LDS by the whole workgroup so the single summing thread
// reads LDS instead of waiting on one global load per term.
__global__ void k_serial_sum(const double* __restrict__ partial, int n, double* __restrict__ out) {
    constexpr int kTile = 4096;
    __shared__ double buf[kTile];
    double t = 0;
    for (int base = 0; base < n; base += kTile) {
        const int m = n - base < kTile ? n - base : kTile;
        for (int i = threadIdx.x; i < m; i += blockDim.x) buf[i] = partial[base + i];
        __syncthreads();
        if (threadIdx.x == 0)
            for (int i = 0; i < m; ++i) t += buf[i];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = t;
}
void chunk_sum(const double* in, long n, double* out, PrimWork& w, hipStream_t s) {
    int nb = n > 0 ? nblocks(n) : 0;
    double* part = w.redPartial.ensure(nb > 0 ? nb : 1);
    if (nb > 0) {
        hipLaunchKernelGGL(k_chunk_sum, dim3(nb), dim3(kBlock), 0, s, in, n, part);
        CIPC_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_serial_sum, dim3(1), dim3(kBlock), 0, s, part, nb, out);
    CIPC_LAUNCH_CHECK();
}
void sum_partials(const double* partials, int n, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_serial_sum, dim3(1), dim3(kBlock), 0, s, partials, n, out);
    CIPC_LAUNCH_CHECK();
}

}  // namespace cipc
