// Candidate walk shared by the constraint-set queries (contact.hip) and the CCD (ccd.hip):
// every item (point or edge) meets the primitives listed in the grid cells of its query
// box, each once (in the first cell common to both boxes), plus the large primitives that
// are kept out of the cell lists.
//
// 16 lanes share an item.  One lane per cell reads the cell's range, a prefix sum over the
// 16 lanes joins the ranges, and the lanes step through the joined list together, so they
// read consecutive 32-byte records.  The cheap test on the records rejects almost all
// candidates; the rest goes to a queue in LDS, from which the exact test takes whole
// workgroups' worth of pairs: no lane waits for another's exact test, and a scene of a few
// thousand primitives is not a serial chain of loads per thread.
// Bound: the latency of the cell ranges and records, then the exact tests' arithmetic.
// Measured against one item per thread, which loaded a primitive's box, its first cell and
// its vertices one after the other (us): edge-edge query of 492,000 edges with 1.25 million
// constraints 6,550 -> 1,000, point-triangle 1,920 -> 256; edge-edge CCD of 129,000 edges
// 743 -> 333; on 12,600 edges 176 -> 27 (query) and 294 -> 29 (CCD).
#pragma once
#include "ctx.hpp"
#include <algorithm>
#include <stdexcept>

namespace cipc {

constexpr int kWalkLanes = 16, kWalkItems = kBlock / kWalkLanes;
constexpr int kWalkUnroll = 4;                            // candidates per lane between two looks at the queue
constexpr int kWalkQueue = kBlock * (kWalkUnroll + 1);    // what one pass adds to less than a workgroup's worth
constexpr int kWalkGrid = 2048;                           // workgroups at most (items grid-stride)
inline int walk_grid(long n) { return (int)std::max(1l, std::min((long)kWalkGrid, (n + kWalkItems - 1) / kWalkItems)); }

// A cell entry's value: the primitive and, per axis, whether the cell is the first one of
// the primitive's box.  A cell is the first common one of two boxes when on every axis it
// is the first of one of them.  (Flags in the record's unused word, 32 bits for the primitive:
// a fourth register per record read ahead, constraint set of 492,000 edges 5.10 -> 5.30 ms,
// CCD of 129,000 edges 0.80 -> 0.83.)  More primitives than the 29 bits number are refused.
constexpr int kWalkIdBits = 29;
constexpr uint32_t kWalkId = (1u << kWalkIdBits) - 1;
__device__ __forceinline__ uint32_t walk_entry(int prim, bool fx, bool fy, bool fz) {
    return (uint32_t)prim | ((fx ? 1u : 0u) | (fy ? 2u : 0u) | (fz ? 4u : 0u)) << kWalkIdBits;
}

struct CellGrid {
    int dim[3];
    const uint32_t* start;    // per cell: first record (and, of the next cell, last + 1)
    const int4* rec;          // records in cell order: box (6 words), entry value, unused
    const int4* box;          // the same per primitive
    const int* lgList;        // large primitives
    const uint32_t* lgCount;
};

// Cell lists by counting: primitives count their cells, a prefix sum over the cells gives
// every list its place, and the entries take places in their lists in any order -- what is
// found does not depend on the order within a cell (the constraint set is sorted by key, the
// CCD takes a minimum), so no sort of the entries by cell is needed.
__device__ __forceinline__ void walk_put(int4* __restrict__ rec, const uint32_t* __restrict__ start, uint32_t* __restrict__ count, long cell,
                                         const int4& a, const int4& b, uint32_t entry) {
    const long k = (long)start[cell] + atomicSub(&count[cell], 1u) - 1;
    rec[2 * k] = a;
    rec[2 * k + 1] = make_int4(b.x, b.y, (int)entry, 0);
}
// Eight lanes share a primitive while its cells are counted and filled: one after the other
// they were a serial chain of atomics and stores (12,600 edges 47 -> 9.7 us to fill and 12 ->
// 6 to count, 492,000 edges 204 -> 85 and 70 -> 55).
constexpr int kCellLanes = 8;
inline dim3 cell_blocks(int n) { return dim3(nblocks((long)n * kCellLanes)); }
__device__ __forceinline__ int cell_prim() { return (int)(((long)blockIdx.x * blockDim.x + threadIdx.x) / kCellLanes); }
// f(cell, whether it is the first of the box a..b on x, y, z)
template <class F>
__device__ __forceinline__ void for_prim_cells(const int* a, const int* b, const int* dim, F f) {
    const int nx = b[0] - a[0] + 1, ny = b[1] - a[1] + 1, nc = nx * ny * (b[2] - a[2] + 1);
    for (int ci = threadIdx.x % kCellLanes; ci < nc; ci += kCellLanes) {
        const int iz = ci / (nx * ny), r = ci - iz * nx * ny, iy = r / nx, ix = r - iy * nx;
        f((a[0] + ix) + (long)dim[0] * ((a[1] + iy) + (long)dim[1] * (a[2] + iz)), ix == 0, iy == 0, iz == 0);
    }
}
// per-cell counters cleared; room for the lists' starts
inline void walk_cells_begin(Ctx& c, long nCells, int n, DevBuf<uint32_t>& start, DevBuf<uint32_t>& count, DevBuf<int>& box,
                             DevBuf<uint8_t>& lgFlag, DevBuf<int>& lgList) {
    if ((uint32_t)n > kWalkId) throw std::length_error("more than 2^29 - 1 boundary triangles, edges or particles");
    start.ensure(nCells + 1);
    count.ensure(nCells);
    CIPC_HIP(hipMemsetAsync(count.p, 0, nCells * sizeof(uint32_t), c.s));
    lgFlag.ensure((size_t)n + 1);
    lgList.ensure((size_t)n + 1);
    box.ensure(8 * (size_t)std::max(n, 1));
}
// starts from the counters; the total number of entries is copied to *hTotal (pinned)
inline void walk_cells_scan(Ctx& c, long nCells, DevBuf<uint32_t>& start, DevBuf<uint32_t>& count, uint32_t* hTotal) {
    scan_exclusive(count.p, start.p, nCells, start.p + nCells, c.pw, c.s);
    CIPC_HIP(hipMemcpyAsync(hTotal, start.p + nCells, sizeof(uint32_t), hipMemcpyDeviceToHost, c.s));
}

// P: bool begin(item, qlo, qhi)           load the item; false: not listed in the cells (large)
//    bool accept(item, prim, a, b, large) the cheap test on a record, and the order of pairs
//    void exact(item, prim)               full test, any lanes of the workgroup active
//    void flush(all)                      after a batch of exact tests, the whole workgroup
// Called by whole workgroups of kBlock threads.
template <class P>
__device__ __forceinline__ void walk_pairs(P& T, int nItems, const CellGrid& G) {
    __shared__ int2 queue[kWalkQueue];
    __shared__ int qn;
    const int tid = threadIdx.x, lane = tid % kWalkLanes, grp = tid / kWalkLanes;
    if (tid == 0) qn = 0;
    const uint32_t nl = *G.lgCount;
    __syncthreads();
    auto push = [&](int item, int prim) { queue[atomicAdd(&qn, 1)] = make_int2(item, prim); };
    // whole workgroups' worth of pairs; the last call takes what is left
    auto drain = [&](bool all) {
        __syncthreads();
        for (;;) {
            const int n = qn;
            const int m = min(n, kBlock);
            const bool on = tid < m;
            const int2 e = on ? queue[n - m + tid] : make_int2(0, 0);
            __syncthreads();   // qn and the entries are read by all before either changes
            if (all ? n == 0 : n < kBlock) break;
            if (tid == 0) qn = n - m;
            if (on) T.exact(e.x, e.y);
            __syncthreads();
            T.flush(false);
        }
    };
    for (int base = blockIdx.x * kWalkItems; base < nItems; base += gridDim.x * kWalkItems) {
        const int item = base + grp;
        const bool live = item < nItems;
        int qlo[3] = {0, 0, 0}, qhi[3] = {-1, -1, -1};
        const bool walks = live && T.begin(item, qlo, qhi);
        const int nx = qhi[0] - qlo[0] + 1, ny = qhi[1] - qlo[1] + 1;
        const int nc = walks ? nx * ny * (qhi[2] - qlo[2] + 1) : 0;
        for (int c0 = 0; __syncthreads_or(c0 < nc); c0 += kWalkLanes) {
            uint32_t st = 0, len = 0;
            int first = 0;
            if (c0 + lane < nc) {
                const int ci = c0 + lane, iz = ci / (nx * ny), r = ci - iz * nx * ny, iy = r / nx, ix = r - iy * nx;
                const long cell = (qlo[0] + ix) + (long)G.dim[0] * ((qlo[1] + iy) + (long)G.dim[1] * (qlo[2] + iz));
                st = G.start[cell];
                len = G.start[cell + 1] - st;
                first = (ix == 0 ? 1 : 0) | (iy == 0 ? 2 : 0) | (iz == 0 ? 4 : 0);
            }
            uint32_t pre = len;   // inclusive prefix over the item's lanes
#pragma unroll
            for (int o = 1; o < kWalkLanes; o <<= 1) {
                const uint32_t u = __shfl_up(pre, o, kWalkLanes);
                if (lane >= o) pre += u;
            }
            const uint32_t total = __shfl(pre, kWalkLanes - 1, kWalkLanes);
            const uint32_t off = st - (pre - len);   // record of joined position t: off + t
            for (uint32_t t0 = 0; __syncthreads_or(t0 < total); t0 += kWalkLanes * kWalkUnroll) {
                int4 ra[kWalkUnroll], rb[kWalkUnroll];
                int fm[kWalkUnroll];
#pragma unroll
                for (int u = 0; u < kWalkUnroll; ++u) {
                    const uint32_t t = t0 + u * kWalkLanes + lane;
                    int j = 0;   // the lane whose cell holds position t
#pragma unroll
                    for (int s = kWalkLanes / 2; s > 0; s >>= 1)
                        if ((uint32_t)__shfl(pre, j + s - 1, kWalkLanes) <= t) j += s;
                    const uint32_t k = (uint32_t)__shfl(off, j, kWalkLanes) + t;
                    const int f = __shfl(first, j, kWalkLanes);
                    fm[u] = t < total ? f : -1;
                    if (t < total) {
                        ra[u] = G.rec[2l * k];
                        rb[u] = G.rec[2l * k + 1];
                    }
                }
#pragma unroll
                for (int u = 0; u < kWalkUnroll; ++u) {
                    if (fm[u] < 0) continue;
                    const uint32_t v = (uint32_t)rb[u].z;
                    if ((fm[u] | (int)(v >> kWalkIdBits)) != 7) continue;
                    const int prim = (int)(v & kWalkId);
                    if (T.accept(item, prim, ra[u], rb[u], false)) push(item, prim);
                }
                drain(false);
            }
        }
        for (uint32_t k0 = 0; k0 < nl; k0 += kWalkLanes) {
            const uint32_t k = k0 + lane;
            if (live && k < nl) {
                const int prim = G.lgList[k];
                if (T.accept(item, prim, G.box[2l * prim], G.box[2l * prim + 1], walks)) push(item, prim);
            }
            drain(false);
        }
    }
    drain(true);
    T.flush(true);
}

}  // namespace cipc
