// Contact kernels: spatial-grid broad phase, point-triangle and edge-edge narrow
// phase with compaction, PP/PE deduplication with multiplicity, barrier energy /
// gradient / Hessian (per-stencil PSD projection), minimum distance.
//
// Reference: FEM/IPC.h:19-740 (Compute_Constraint_Set), :742-941, :943-1256,
// :1258-1731 (Compute_Barrier{,_Gradient,_Hessian}), :2246-2388 (Compute_Min_Dist2).
//
// Broad phase: a uniform grid (cell = mean rest boundary-edge length, grown so the
// grid has at most 2^23 cells) holds each triangle / edge in every cell its AABB
// touches, cell after cell (counted, prefix sum, placed).  A query visits the cells of its box (walk.hpp) and
// accepts a candidate only in the first cell common to both boxes, so every pair is
// tested once; indices are clamped into the grid, which keeps the search complete
// for points outside it.  The active set is defined by the reference's predicates
// (AABB filter with d_hat + offset, region type, d^2 < (d_hat + offset)^2), so it does
// not depend on the grid.
//
// Output order (deterministic): point-triangle by (boundary node, triangle),
// edge-edge family by (edge, edge), then deduplicated PP/PE entries in the
// lexicographic int4 order of the reference's std::map.
#include "ctx.hpp"
#include "dev_math.hpp"
#include "walk.hpp"
#include <algorithm>
#include <chrono>
#include <cmath>

namespace cipc {

__device__ __forceinline__ int cell_of(double v, double lb, double inv, int dim) {
    double f = floor((v - lb) * inv);
    if (!(f >= 0.0)) return 0;
    if (f >= (double)(dim - 1)) return dim - 1;
    return (int)f;
}

// ------------------------------------------------------------------ grid build
// Primitives are triangles (3 vertices, SoA), boundary edges (2) or particles (1).  Each gets
// a box record of outward-rounded floats: a test on it can only accept too much, the exact
// predicates decide on what it accepts.  Primitives whose box covers more than kLargeCells
// cells get count 0 and go to the large list.
__device__ __forceinline__ float float_below(double v) {
    const float f = (float)v;
    return f - fabsf(f) * 2.4e-7f - 1e-30f;
}
__device__ __forceinline__ float float_above(double v) {
    const float f = (float)v;
    return f + fabsf(f) * 2.4e-7f + 1e-30f;
}
__device__ __forceinline__ void prim_minmax(const double* __restrict__ x, const int* __restrict__ verts, int n, int nv, int i, double* mn,
                                            double* mx) {
#pragma unroll
    for (int d = 0; d < 3; ++d) { mn[d] = 1e300; mx[d] = -1e300; }
    for (int k = 0; k < nv; ++k) {
        int v = verts[(long)k * n + i];
#pragma unroll
        for (int d = 0; d < 3; ++d) { double c = x[3 * v + d]; mn[d] = c < mn[d] ? c : mn[d]; mx[d] = c > mx[d] ? c : mx[d]; }
    }
}
__global__ void k_prim_range(const double* __restrict__ x, const int* __restrict__ verts, int n, int nv, GridParams G,
                             int4* __restrict__ box, uint32_t* __restrict__ count, uint8_t* __restrict__ lgFlag,
                             int* __restrict__ lgList, uint32_t* __restrict__ lgCount) {   // count: per cell
    const int i = cell_prim();
    if (i >= n) return;
    double mn[3], mx[3];
    prim_minmax(x, verts, n, nv, i, mn, mx);
    uint64_t cnt = 1;
    int a[3], b[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        a[d] = cell_of(mn[d], G.lb[d], G.inv, G.dim[d]);
        b[d] = cell_of(mx[d], G.lb[d], G.inv, G.dim[d]);
        cnt *= (uint64_t)(b[d] - a[d] + 1);
    }
    const bool large = cnt > kLargeCells;
    if (threadIdx.x % kCellLanes == 0) {
        box[2l * i] = make_int4(__float_as_int(float_below(mn[0])), __float_as_int(float_below(mn[1])), __float_as_int(float_below(mn[2])),
                                __float_as_int(float_above(mx[0])));
        box[2l * i + 1] = make_int4(__float_as_int(float_above(mx[1])), __float_as_int(float_above(mx[2])), 0, 0);
        lgFlag[i] = large ? 1 : 0;
        if (large) lgList[atomicAdd(lgCount, 1u)] = i;
    }
    if (large) return;
    for_prim_cells(a, b, G.dim, [&](long cell, bool, bool, bool) { atomicAdd(&count[cell], 1u); });
}
__global__ void k_prim_emit(const double* __restrict__ x, const int* __restrict__ verts, int n, int nv, GridParams G,
                            const uint8_t* __restrict__ lgFlag, const int4* __restrict__ box, const uint32_t* __restrict__ start,
                            uint32_t* __restrict__ count, int4* __restrict__ rec) {
    const int i = cell_prim();
    if (i >= n || lgFlag[i]) return;
    double mn[3], mx[3];
    prim_minmax(x, verts, n, nv, i, mn, mx);
    int a[3], b[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) { a[d] = cell_of(mn[d], G.lb[d], G.inv, G.dim[d]); b[d] = cell_of(mx[d], G.lb[d], G.inv, G.dim[d]); }
    const int4 ba = box[2l * i], bb = box[2l * i + 1];
    for_prim_cells(a, b, G.dim, [&](long cell, bool fx, bool fy, bool fz) { walk_put(rec, start, count, cell, ba, bb, walk_entry(i, fx, fy, fz)); });
}
static int bits_for(uint64_t n) {
    int b = 1;
    while (b < 64 && (1ull << b) < n) ++b;
    return b;
}

// cell lists of one primitive kind (large primitives listed apart, their count left in
// device memory at lgCount): counts and starts, then, once the host knows the number of
// entries, the records
struct CellBuild {
    const int* verts;
    int n, nv;
    DevBuf<int>&box, &rec;
    DevBuf<uint32_t>&start, &count;
    DevBuf<uint8_t>& lgFlag;
    DevBuf<int>& lgList;
    uint32_t *lgCount, *hTotal;
};
static void cells_count(Ctx& c, const double* x, const GridParams& G, const CellBuild& b) {
    const long nCells = (long)G.dim[0] * G.dim[1] * G.dim[2];
    walk_cells_begin(c, nCells, b.n, b.start, b.count, b.box, b.lgFlag, b.lgList);
    if (b.n) {
        hipLaunchKernelGGL(k_prim_range, cell_blocks(b.n), dim3(kBlock), 0, c.s, x, b.verts, b.n, b.nv, G, (int4*)b.box.p, b.count.p,
                           b.lgFlag.p, b.lgList.p, b.lgCount);
        CIPC_LAUNCH_CHECK();
    }
    walk_cells_scan(c, nCells, b.start, b.count, b.hTotal);
}
static void cells_emit(Ctx& c, const double* x, const GridParams& G, const CellBuild& b) {
    b.rec.ensure(8 * (size_t)std::max(*b.hTotal, 1u));
    if (*b.hTotal == 0) return;
    hipLaunchKernelGGL(k_prim_emit, cell_blocks(b.n), dim3(kBlock), 0, c.s, x, b.verts, b.n, b.nv, G, (const uint8_t*)b.lgFlag.p,
                       (const int4*)b.box.p, (const uint32_t*)b.start.p, b.count.p, (int4*)b.rec.p);
    CIPC_LAUNCH_CHECK();
}

// ------------------------------------------------------------------ narrow phase
struct CSOut {
    uint64_t* key; int* c4; uint32_t* cnt; uint32_t cap;   // kept entries
    uint64_t* dkey; uint32_t* dcnt; uint32_t dcap;          // PP/PE entries to deduplicate
};

__device__ __forceinline__ uint64_t dup_key(int c0, int c1, int c2, int nV) {
    // lexicographic order of (c0 < 0, c1 >= 0, c2 >= -1) as signed ints
    uint64_t a = (uint64_t)(nV - 1 - (-c0 - 1)), b = (uint64_t)c1, d = (uint64_t)(c2 + 1);
    return (a * (uint64_t)nV + b) * (uint64_t)(nV + 1) + d;
}
// Output slots reserved once per wavefront (wave_reserve).  The slot order is arbitrary; the
// set is sorted by key afterwards, so the result is deterministic.
struct WaveOut {
    CSOut o;
    __device__ __forceinline__ void dup(uint64_t key) const {
        const uint32_t i = wave_reserve(o.dcnt);
        if (i < o.dcap) o.dkey[i] = key;
    }
};
// Output gathered in LDS and written out a few hundred entries at a time: one atomic on the
// counter per flush.  (One per wavefront and emission was most of the queries' time on a
// state with 10^6 constraints: atomics on one address take about 15 ns each.)
constexpr int kOutCap = 2 * kBlock;   // a batch adds up to kBlock entries to at most kBlock
struct OutBuf {
    uint64_t key[kOutCap], dkey[kOutCap];
    int4 c4[kOutCap];
    int n, nd;
    uint32_t base, dbase;
};
struct BlockOut {
    CSOut o;
    OutBuf* b;
    __device__ __forceinline__ void init() const {
        if (threadIdx.x == 0) b->n = b->nd = 0;   // the walk's first barrier orders it
    }
    __device__ __forceinline__ void kept(uint64_t key, int c0, int c1, int c2, int c3) const {
        const int i = atomicAdd(&b->n, 1);
        b->key[i] = key;
        b->c4[i] = make_int4(c0, c1, c2, c3);
    }
    __device__ __forceinline__ void dup(uint64_t key) const { b->dkey[atomicAdd(&b->nd, 1)] = key; }
    // whole workgroup, after a barrier
    __device__ __forceinline__ void flush(bool all) const {
        const int n = b->n, nd = b->nd, lim = all ? 0 : kOutCap - kBlock;
        const bool fk = n > lim, fd = nd > lim;
        if (fk || fd) {
            if (threadIdx.x == 0) {
                if (fk) b->base = atomicAdd(o.cnt, (uint32_t)n);
                if (fd) b->dbase = atomicAdd(o.dcnt, (uint32_t)nd);
            }
            __syncthreads();
            if (fk)
                for (int i = threadIdx.x; i < n; i += kBlock) {
                    const uint32_t k = b->base + i;
                    if (k >= o.cap) break;
                    o.key[k] = b->key[i];
                    reinterpret_cast<int4*>(o.c4)[k] = b->c4[i];
                }
            if (fd)
                for (int i = threadIdx.x; i < nd; i += kBlock) {
                    const uint32_t k = b->dbase + i;
                    if (k < o.dcap) o.dkey[k] = b->dkey[i];
                }
            __syncthreads();
            if (threadIdx.x == 0) {
                if (fk) b->n = 0;
                if (fd) b->nd = 0;
            }
        }
        __syncthreads();   // the counts are read by all before the next batch adds to them
    }
};

#pragma clang fp contract(off)
__device__ __forceinline__ bool pt_cd_broadphase(d3 p, d3 t0, d3 t1, d3 t2, double dist) {
    double mx, mn;
    mx = dmax(dmax(t0.x, t1.x), t2.x); mn = dmin(dmin(t0.x, t1.x), t2.x);
    if (p.x - mx > dist || mn - p.x > dist) return false;
    mx = dmax(dmax(t0.y, t1.y), t2.y); mn = dmin(dmin(t0.y, t1.y), t2.y);
    if (p.y - mx > dist || mn - p.y > dist) return false;
    mx = dmax(dmax(t0.z, t1.z), t2.z); mn = dmin(dmin(t0.z, t1.z), t2.z);
    if (p.z - mx > dist || mn - p.z > dist) return false;
    return true;
}
__device__ __forceinline__ bool ee_cd_broadphase(d3 a0, d3 a1, d3 b0, d3 b1, double dist) {
    if (dmin(a0.x, a1.x) - dmax(b0.x, b1.x) > dist || dmin(b0.x, b1.x) - dmax(a0.x, a1.x) > dist) return false;
    if (dmin(a0.y, a1.y) - dmax(b0.y, b1.y) > dist || dmin(b0.y, b1.y) - dmax(a0.y, a1.y) > dist) return false;
    if (dmin(a0.z, a1.z) - dmax(b0.z, b1.z) > dist || dmin(b0.z, b1.z) - dmax(a0.z, a1.z) > dist) return false;
    return true;
}

// point vI (boundary-node slot svI) against triangle t: IPC.h:57-140
template <class O>
__device__ __forceinline__ void pt_candidate(const O& o, const double* __restrict__ x, const int* __restrict__ tri, int nT,
                                             const uint8_t* __restrict__ dbc, int svI, int vI, d3 p, int t, double dHat,
                                             double dHat2, int nV) {
    int a = tri[t], b = tri[nT + t], cc = tri[2 * nT + t];
    if (vI == a || vI == b || vI == cc) return;
    if (dbc[vI] && dbc[a] && dbc[b] && dbc[cc]) return;
    d3 t0 = ld3(x, a), t1 = ld3(x, b), t2 = ld3(x, cc);
    if (!pt_cd_broadphase(p, t0, t1, t2, dHat)) return;
    int ty = pt_type(p, t0, t1, t2);
    double d;
    int c1 = -1, c2 = -1;
    switch (ty) {
        case 0: d = dist2_pp(p, t0); c1 = a; break;
        case 1: d = dist2_pp(p, t1); c1 = b; break;
        case 2: d = dist2_pp(p, t2); c1 = cc; break;
        case 3: d = dist2_pe(p, t0, t1); c1 = a; c2 = b; break;
        case 4: d = dist2_pe(p, t1, t2); c1 = b; c2 = cc; break;
        case 5: d = dist2_pe(p, t2, t0); c1 = cc; c2 = a; break;
        default: d = dist2_pt(p, t0, t1, t2); break;
    }
    if (!(d < dHat2)) return;
    if (ty == 6) o.kept((uint64_t)svI * (uint64_t)nT + (uint64_t)t, -vI - 1, a, b, cc);
    else o.dup(dup_key(-vI - 1, c1, c2, nV));
}

// edge pair eA < eB: IPC.h:142-330 (edge A supplies a0/a1 of the encoding)
template <class O>
__device__ __forceinline__ void ee_candidate(const O& o, const double* __restrict__ x, const double* __restrict__ X0,
                                             const int* __restrict__ bEdge, int nBE, const uint8_t* __restrict__ dbc, int eA, int a0,
                                             int a1, d3 ea0, d3 ea1, int eB, double dHat, double dHat2, int nV) {
    int b0 = bEdge[eB], b1 = bEdge[nBE + eB];
    if (a0 == b0 || a0 == b1 || a1 == b0 || a1 == b1) return;
    if (dbc[a0] && dbc[a1] && dbc[b0] && dbc[b1]) return;
    d3 eb0 = ld3(x, b0), eb1 = ld3(x, b1);
    if (!ee_cd_broadphase(ea0, ea1, eb0, eb1, dHat)) return;
    double crossN = ee_cross_norm2(ea0, ea1, eb0, eb1);
    double eps = ee_mollifier_threshold(ld3(X0, a0), ld3(X0, a1), ld3(X0, b0), ld3(X0, b1));
    bool moll = crossN < eps;
    double d;
    int c[4];
    switch (ee_type(ea0, ea1, eb0, eb1)) {
        case 0: d = dist2_pp(ea0, eb0);
            if (moll) { c[0] = a0; c[1] = b0; c[2] = -a1 - 1; c[3] = -b1 - 1; } else { c[0] = -a0 - 1; c[1] = b0; c[2] = -1; c[3] = -1; } break;
        case 1: d = dist2_pp(ea0, eb1);
            if (moll) { c[0] = a0; c[1] = b1; c[2] = -a1 - 1; c[3] = -b0 - 1; } else { c[0] = -a0 - 1; c[1] = b1; c[2] = -1; c[3] = -1; } break;
        case 2: d = dist2_pe(ea0, eb0, eb1);
            if (moll) { c[0] = a0; c[1] = b0; c[2] = b1; c[3] = -a1 - 1; } else { c[0] = -a0 - 1; c[1] = b0; c[2] = b1; c[3] = -1; } break;
        case 3: d = dist2_pp(ea1, eb0);
            if (moll) { c[0] = a1; c[1] = b0; c[2] = -a0 - 1; c[3] = -b1 - 1; } else { c[0] = -a1 - 1; c[1] = b0; c[2] = -1; c[3] = -1; } break;
        case 4: d = dist2_pp(ea1, eb1);
            if (moll) { c[0] = a1; c[1] = b1; c[2] = -a0 - 1; c[3] = -b0 - 1; } else { c[0] = -a1 - 1; c[1] = b1; c[2] = -1; c[3] = -1; } break;
        case 5: d = dist2_pe(ea1, eb0, eb1);
            if (moll) { c[0] = a1; c[1] = b0; c[2] = b1; c[3] = -a0 - 1; } else { c[0] = -a1 - 1; c[1] = b0; c[2] = b1; c[3] = -1; } break;
        case 6: d = dist2_pe(eb0, ea0, ea1);
            if (moll) { c[0] = b0; c[1] = a0; c[2] = a1; c[3] = -b1 - 1; } else { c[0] = -b0 - 1; c[1] = a0; c[2] = a1; c[3] = -1; } break;
        case 7: d = dist2_pe(eb1, ea0, ea1);
            if (moll) { c[0] = b1; c[1] = a0; c[2] = a1; c[3] = -b0 - 1; } else { c[0] = -b1 - 1; c[1] = a0; c[2] = a1; c[3] = -1; } break;
        default: d = dist2_ee(ea0, ea1, eb0, eb1);
            if (moll) { c[0] = a0; c[1] = a1; c[2] = -b0 - 1; c[3] = b1; } else { c[0] = a0; c[1] = a1; c[2] = b0; c[3] = b1; } break;
    }
    if (!(d < dHat2)) return;
    if (c[0] >= 0) o.kept((uint64_t)eA * (uint64_t)nBE + (uint64_t)eB, c[0], c[1], c[2], c[3]);
    else o.dup(dup_key(c[0], c[1], c[2], nV));
}

// float box of the item grown by dHat against a record's box
struct QueryBox {
    float lo[3], hi[3];
    __device__ __forceinline__ void set(const double* mn, const double* mx, double dHat) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = float_below(mn[d] - dHat);
            hi[d] = float_above(mx[d] + dHat);
        }
    }
    __device__ __forceinline__ bool meets(const int4& a, const int4& b) const {
        return !(__int_as_float(a.x) > hi[0] || __int_as_float(a.w) < lo[0] || __int_as_float(a.y) > hi[1] || __int_as_float(b.x) < lo[1] ||
                 __int_as_float(a.z) > hi[2] || __int_as_float(b.y) < lo[2]);
    }
};
struct QueryPT {
    const double* __restrict__ x;
    const int* __restrict__ bNode;
    const int* __restrict__ tri;
    int nT;
    const uint8_t* __restrict__ dbc;
    GridParams G;
    double dHat, dHat2;
    int nV;
    BlockOut o;
    QueryBox q;
    __device__ __forceinline__ void flush(bool all) const { o.flush(all); }
    __device__ __forceinline__ bool begin(int slot, int* qlo, int* qhi) {
        const d3 p = ld3(x, bNode[slot]);
        const double pc[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            qlo[d] = cell_of(pc[d] - dHat, G.lb[d], G.inv, G.dim[d]);
            qhi[d] = cell_of(pc[d] + dHat, G.lb[d], G.inv, G.dim[d]);
        }
        q.set(pc, pc, dHat);
        return true;
    }
    __device__ __forceinline__ bool accept(int, int, const int4& a, const int4& b, bool) const { return q.meets(a, b); }
    __device__ __forceinline__ void exact(int slot, int t) const {
        const int vI = bNode[slot];
        pt_candidate(o, x, tri, nT, dbc, slot, vI, ld3(x, vI), t, dHat, dHat2, nV);
    }
};
__global__ __launch_bounds__(kBlock) void k_query_pt(QueryPT T, int nBN, CellGrid G) {
    __shared__ OutBuf buf;
    T.o.b = &buf;
    T.o.init();
    walk_pairs(T, nBN, G);
}

// Every unordered edge pair is tested once: a grid-listed edge finds grid-listed
// edges of larger index in the first common cell and every large edge from the
// list; a large edge only tests large edges of larger index.
struct QueryEE {
    const double* __restrict__ x;
    const double* __restrict__ X0;
    const int* __restrict__ bEdge;
    int nBE;
    const uint8_t* __restrict__ dbc;
    const uint8_t* __restrict__ lgFlag;
    GridParams G;
    double dHat, dHat2;
    int nV;
    BlockOut o;
    QueryBox q;
    __device__ __forceinline__ void flush(bool all) const { o.flush(all); }
    __device__ __forceinline__ bool begin(int e, int* qlo, int* qhi) {
        const d3 a = ld3(x, bEdge[e]), b = ld3(x, bEdge[nBE + e]);
        const double mn[3] = {dmin(a.x, b.x), dmin(a.y, b.y), dmin(a.z, b.z)}, mx[3] = {dmax(a.x, b.x), dmax(a.y, b.y), dmax(a.z, b.z)};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            qlo[d] = cell_of(mn[d] - dHat, G.lb[d], G.inv, G.dim[d]);
            qhi[d] = cell_of(mx[d] + dHat, G.lb[d], G.inv, G.dim[d]);
        }
        q.set(mn, mx, dHat);
        return !lgFlag[e];
    }
    __device__ __forceinline__ bool accept(int e, int other, const int4& a, const int4& b, bool anyOrder) const {
        return (anyOrder || other > e) && q.meets(a, b);
    }
    __device__ __forceinline__ void exact(int e, int other) const {
        const int eA = min(e, other), eB = max(e, other), a0 = bEdge[eA], a1 = bEdge[nBE + eA];
        ee_candidate(o, x, X0, bEdge, nBE, dbc, eA, a0, a1, ld3(x, a0), ld3(x, a1), eB, dHat, dHat2, nV);
    }
};
__global__ __launch_bounds__(kBlock) void k_query_ee(QueryEE T, CellGrid G) {
    __shared__ OutBuf buf;
    T.o.b = &buf;
    T.o.init();
    walk_pairs(T, T.nBE, G);
}
// rod nodes and particles (boundary-node slots >= codimBN0) against rod segments (the
// last nRod boundary edges), IPC.h:271-317; particles (slots >= codimBN1) against the
// particles after them, IPC.h:319-349.  All results are PP/PE entries for the
// multiplicity merge.  One item per thread: bound by its chain of loads (cell range, record,
// vertices).  4,800 rod segments and 3,600 particles in contact 185 us, 200,000 and 100,000
// without contacts 396 (233 and 494 with packed ids and the boxes' cells loaded per candidate).
__device__ __forceinline__ bool pe_cd_broadphase(d3 p, d3 e0, d3 e1, double dist) {
    if (p.x - dmax(e0.x, e1.x) > dist || dmin(e0.x, e1.x) - p.x > dist) return false;
    if (p.y - dmax(e0.y, e1.y) > dist || dmin(e0.y, e1.y) - p.y > dist) return false;
    if (p.z - dmax(e0.z, e1.z) > dist || dmin(e0.z, e1.z) - p.z > dist) return false;
    return true;
}
template <class O>
__device__ __forceinline__ void pe_codim_candidate(const O& o, const double* __restrict__ x, const int* __restrict__ bEdge, int nBE,
                                                   const uint8_t* __restrict__ dbc, int vI, d3 p, int eJ, double dHat, double dHat2,
                                                   int nV) {
    int a = bEdge[eJ], b = bEdge[nBE + eJ];
    if (vI == a || vI == b) return;
    if (dbc[vI] && dbc[a] && dbc[b]) return;
    d3 e0 = ld3(x, a), e1 = ld3(x, b);
    if (!pe_cd_broadphase(p, e0, e1, dHat)) return;
    double d;
    int c1, c2 = -1;
    switch (pe_type(p, e0, e1)) {
        case 0: d = dist2_pp(p, e0); c1 = a; break;
        case 1: d = dist2_pp(p, e1); c1 = b; break;
        default: d = dist2_pe(p, e0, e1); c1 = a; c2 = b; break;
    }
    if (d < dHat2) o.dup(dup_key(-vI - 1, c1, c2, nV));
}
__global__ void k_query_codim(const double* __restrict__ x, const int* __restrict__ bNode, int nBN, int codimBN0, int codimBN1,
                              const int* __restrict__ bEdge, int nBE, int nRod, const uint8_t* __restrict__ dbc, GridParams G,
                              const uint32_t* __restrict__ estart, const int4* __restrict__ erec,
                              const int* __restrict__ lgListE, const uint32_t* __restrict__ lgCountE,
                              const uint32_t* __restrict__ pstart, const int4* __restrict__ prec,
                              double dHat, double dHat2, int nV, CSOut out) {
    const WaveOut o{out};
    int s = codimBN0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nBN) return;
    int vI = bNode[s];
    d3 p = ld3(x, vI);
    int qlo[3], qhi[3];
    double pc[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) { qlo[d] = cell_of(pc[d] - dHat, G.lb[d], G.inv, G.dim[d]); qhi[d] = cell_of(pc[d] + dHat, G.lb[d], G.inv, G.dim[d]); }
    const int firstRod = nBE - nRod;
    for (int iz = qlo[2]; iz <= qhi[2]; ++iz)
        for (int iy = qlo[1]; iy <= qhi[1]; ++iy)
            for (int ix = qlo[0]; ix <= qhi[0]; ++ix) {
                uint64_t cell = (uint64_t)ix + (uint64_t)G.dim[0] * ((uint64_t)iy + (uint64_t)G.dim[1] * (uint64_t)iz);
                for (uint32_t k = estart[cell], e = estart[cell + 1]; k < e; ++k) {
                    const uint32_t entry = (uint32_t)erec[2l * k + 1].z;
                    const int eJ = (int)(entry & kWalkId), first = (int)(entry >> kWalkIdBits);
                    if (eJ < firstRod) continue;
                    if ((first | (ix == qlo[0] ? 1 : 0) | (iy == qlo[1] ? 2 : 0) | (iz == qlo[2] ? 4 : 0)) != 7) continue;
                    pe_codim_candidate(o, x, bEdge, nBE, dbc, vI, p, eJ, dHat, dHat2, nV);
                }
            }
    const uint32_t nl = *lgCountE;
    for (uint32_t k = 0; k < nl; ++k) {
        int eJ = lgListE[k];
        if (eJ >= firstRod) pe_codim_candidate(o, x, bEdge, nBE, dbc, vI, p, eJ, dHat, dHat2, nV);
    }
    if (s < codimBN1) return;
    // a point lies in exactly one cell, so each particle pair is met once
    for (int iz = qlo[2]; iz <= qhi[2]; ++iz)
        for (int iy = qlo[1]; iy <= qhi[1]; ++iy)
            for (int ix = qlo[0]; ix <= qhi[0]; ++ix) {
                uint64_t cell = (uint64_t)ix + (uint64_t)G.dim[0] * ((uint64_t)iy + (uint64_t)G.dim[1] * (uint64_t)iz);
                for (uint32_t k = pstart[cell], e = pstart[cell + 1]; k < e; ++k) {
                    int sJ = codimBN1 + (int)((uint32_t)prec[2l * k + 1].z & kWalkId);
                    if (sJ <= s) continue;
                    int vJ = bNode[sJ];
                    if (dbc[vI] && dbc[vJ]) continue;
                    double d = dist2_pp(p, ld3(x, vJ));
                    if (d < dHat2) o.dup(dup_key(-vI - 1, vJ, -1, nV));
                }
            }
}
#pragma clang fp contract(on)

// gather sorted kept entries into the SoA constraint array
__global__ void k_gather_c4(const uint32_t* __restrict__ idx, const int* __restrict__ c4, int n, int* __restrict__ C, int nC,
                            int offset) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    long s = idx[i];
#pragma unroll
    for (int k = 0; k < 4; ++k) C[(long)k * nC + offset + i] = c4[4 * s + k];
}
// the library's SoA sets and the callers' int4 rows, either way: the host copies rows as they
// are (transposing on the host was 0.24 of the 0.76 ms of a gradient call on 4 sheets of
// 101 x 101)
__global__ void k_constraint_rows(int* __restrict__ C, int4* __restrict__ rows, int nC, int toRows) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nC) return;
    if (toRows) {
        rows[i] = make_int4(C[i], C[(long)nC + i], C[2l * nC + i], C[3l * nC + i]);
    } else {
        const int4 r = rows[i];
        C[i] = r.x; C[(long)nC + i] = r.y; C[2l * nC + i] = r.z; C[3l * nC + i] = r.w;
    }
}
void constraint_rows(Ctx& c, int* C, int* rows, int nC, bool toRows) {
    hipLaunchKernelGGL(k_constraint_rows, dim3(nblocks(nC)), dim3(kBlock), 0, c.s, C, (int4*)rows, nC, toRows ? 1 : 0);
    CIPC_LAUNCH_CHECK();
}
__global__ void k_run_flags(const uint64_t* __restrict__ key, int n, uint32_t* __restrict__ head) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    head[i] = (i == 0 || key[i] != key[i - 1]) ? 1u : 0u;
}
__global__ void k_run_emit(const uint64_t* __restrict__ key, int n, const uint32_t* __restrict__ pos, int* __restrict__ C, int nC,
                           int offset, int nV) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (!(i == 0 || key[i] != key[i - 1])) return;
    int j = i + 1;
    while (j < n && key[j] == key[i]) ++j;
    uint64_t k = key[i];
    uint64_t d = k % (uint64_t)(nV + 1), r = k / (uint64_t)(nV + 1);
    uint64_t b = r % (uint64_t)nV, a = r / (uint64_t)nV;
    int c0 = -((int)(nV - 1 - (int)a)) - 1;
    long o = offset + pos[i];
    C[o] = c0;
    C[(long)nC + o] = (int)b;
    C[2l * nC + o] = (int)d - 1;
    C[3l * nC + o] = -(j - i);
}

static void constraint_set_impl(Ctx& c, const double* x, DevBuf<int>& out, int& nOut) {
    const double dHat = std::sqrt(c.dHat2) + c.P.xi;     // IPC.h:53-54
    const double dHat2 = dHat * dHat;
    // grid over the current bounding box of all vertices
    {
        double* bb = c.scal.p + 16;
        bbox_minmax(c, x, bb);
        CIPC_HIP(hipMemcpyAsync(c.hScal + 16, bb, 6 * sizeof(double), hipMemcpyDeviceToHost, c.s));
        CIPC_HIP(hipStreamSynchronize(c.s));
    }
    GridParams G;
    double cs = c.cellSize * c.cellMult;
    double rng[3];
    for (int d = 0; d < 3; ++d) { G.lb[d] = c.hScal[16 + d]; rng[d] = c.hScal[19 + d] - c.hScal[16 + d]; }
    for (;;) {
        double nc = 1;
        for (int d = 0; d < 3; ++d) nc *= std::floor(rng[d] / cs) + 1;
        if (nc <= (double)(1 << 23)) break;
        cs *= 1.25;
    }
    G.inv = 1.0 / cs;
    for (int d = 0; d < 3; ++d) G.dim[d] = (int)std::floor(rng[d] / cs) + 1;

    uint32_t* lgCountT = c.counters.p + 16;
    uint32_t* lgCountE = c.counters.p + 17;
    uint32_t* lgCountP = c.counters.p + 18;
    CIPC_HIP(hipMemsetAsync(lgCountT, 0, 3 * sizeof(uint32_t), c.s));
    const CellBuild bt = {c.btri.p, c.nBT, 3, c.csBoxT, c.csRecT, c.cellStart, c.cellCount, c.lgFlagT, c.lgListT, lgCountT, c.hCnt + 8};
    const CellBuild be = {c.bEdge.p, c.nBE, 2, c.csBoxE, c.csRecE, c.ecellStart, c.ecellCount, c.lgFlagE, c.lgListE, lgCountE, c.hCnt + 9};
    const CellBuild bp = {c.partSlot.p, c.nPart, 1, c.csBoxP, c.csRecP, c.pcellStart, c.pcellCount, c.lgFlagP, c.lgListP, lgCountP, c.hCnt + 10};
    cells_count(c, x, G, bt);
    cells_count(c, x, G, be);
    if (c.nPart) cells_count(c, x, G, bp);
    CIPC_HIP(hipStreamSynchronize(c.s));   // the three totals
    cells_emit(c, x, G, bt);
    cells_emit(c, x, G, be);
    if (c.nPart) cells_emit(c, x, G, bp);

    // narrow phase with capacity retry
    CSOut o;
    uint32_t cap = c.csCap;
    for (;;) {
        o.cap = cap; o.dcap = cap;
        o.key = c.csKey.ensure(2 * (size_t)cap);
        o.c4 = c.csC4.ensure(8 * (size_t)cap);
        o.dkey = c.csDKey.ensure((size_t)cap);
        o.cnt = c.counters.p;
        o.dcnt = c.counters.p + 1;
        CIPC_HIP(hipMemsetAsync(c.counters.p, 0, 4 * sizeof(uint32_t), c.s));
        // point-triangle kept entries fill [0, cap), edge-edge kept entries [cap, 2 cap)
        const CellGrid GT = {{G.dim[0], G.dim[1], G.dim[2]}, c.cellStart.p, (const int4*)c.csRecT.p, (const int4*)c.csBoxT.p,
                             c.lgListT.p, lgCountT};
        const CellGrid GE = {{G.dim[0], G.dim[1], G.dim[2]}, c.ecellStart.p, (const int4*)c.csRecE.p, (const int4*)c.csBoxE.p,
                             c.lgListE.p, lgCountE};
        const QueryPT pt = {x, c.bNode.p, c.btri.p, c.nBT, c.dbc.p, G, dHat, dHat2, c.nV, {o, nullptr}, {}};
        hipLaunchKernelGGL(k_query_pt, dim3(walk_grid(c.nBN)), dim3(kBlock), 0, c.s, pt, c.nBN, GT);
        CIPC_LAUNCH_CHECK();
        CSOut oEE = o;
        oEE.key = o.key + cap; oEE.c4 = o.c4 + 4 * (size_t)cap; oEE.cnt = c.counters.p + 2;
        const QueryEE ee = {x, c.X0.p, c.bEdge.p, c.nBE, c.dbc.p, c.lgFlagE.p, G, dHat, dHat2, c.nV, {oEE, nullptr}, {}};
        hipLaunchKernelGGL(k_query_ee, dim3(walk_grid(c.nBE)), dim3(kBlock), 0, c.s, ee, GE);
        CIPC_LAUNCH_CHECK();
        if (c.nBN > c.codimBN0) {
            hipLaunchKernelGGL(k_query_codim, dim3(nblocks(c.nBN - c.codimBN0)), dim3(kBlock), 0, c.s, x, c.bNode.p, c.nBN, c.codimBN0,
                               c.codimBN1, c.bEdge.p, c.nBE, c.nRod, c.dbc.p, G, c.ecellStart.p, (const int4*)c.csRecE.p,
                               c.lgListE.p, lgCountE, c.nPart ? c.pcellStart.p : c.ecellStart.p,
                               (const int4*)(c.nPart ? c.csRecP.p : c.csRecE.p), dHat, dHat2, c.nV, o);
            CIPC_LAUNCH_CHECK();
        }
        CIPC_HIP(hipMemcpyAsync(c.hCnt, c.counters.p, 4 * sizeof(uint32_t), hipMemcpyDeviceToHost, c.s));
        CIPC_HIP(hipStreamSynchronize(c.s));
        uint32_t nPT = c.hCnt[0], nDup = c.hCnt[1], nEE = c.hCnt[2];
        uint32_t need = std::max(std::max(nPT, nDup), nEE);
        if (need > cap) {
            while (cap < need) cap *= 2;
            c.csCap = cap;
            continue;
        }
        // deduplicate PP/PE entries: sort, run heads, scan
        uint32_t nUnique = 0;
        uint32_t* dpos = c.csPos.ensure((size_t)std::max<uint32_t>(nDup, 1) + 1);
        uint32_t* si = c.csIdx.ensure((size_t)std::max<uint32_t>(std::max(std::max(nPT, nEE), nDup), 1));
        const uint64_t* dkey = nullptr;
        if (nDup) {
            dkey = radix_sort_pairs(o.dkey, si, nDup, bits_for((uint64_t)c.nV * c.nV * (c.nV + 1)), c.pw, c.s).keys;
            uint32_t* h = c.csHead.ensure(nDup);
            hipLaunchKernelGGL(k_run_flags, dim3(nblocks(nDup)), dim3(kBlock), 0, c.s, dkey, (int)nDup, h);
            CIPC_LAUNCH_CHECK();
            scan_exclusive(h, dpos, nDup, c.counters.p + 4, c.pw, c.s);
            CIPC_HIP(hipMemcpyAsync(c.hCnt + 4, c.counters.p + 4, sizeof(uint32_t), hipMemcpyDeviceToHost, c.s));
            CIPC_HIP(hipStreamSynchronize(c.s));
            nUnique = c.hCnt[4];
        }
        int nC = (int)(nPT + nEE + nUnique);
        out.ensure((size_t)4 * std::max(nC, 1));
        if (nDup) {   // before the next sort, which may reuse dkey's buffer
            hipLaunchKernelGGL(k_run_emit, dim3(nblocks(nDup)), dim3(kBlock), 0, c.s, dkey, (int)nDup, dpos, out.p, nC,
                               (int)(nPT + nEE), c.nV);
            CIPC_LAUNCH_CHECK();
        }
        if (nPT) {
            const uint32_t* idx = radix_sort_pairs(o.key, si, nPT, bits_for((uint64_t)c.nBN * c.nBT), c.pw, c.s).vals;
            hipLaunchKernelGGL(k_gather_c4, dim3(nblocks(nPT)), dim3(kBlock), 0, c.s, idx, o.c4, (int)nPT, out.p, nC, 0);
            CIPC_LAUNCH_CHECK();
        }
        if (nEE) {
            const uint32_t* idx = radix_sort_pairs(oEE.key, si, nEE, bits_for((uint64_t)c.nBE * c.nBE), c.pw, c.s).vals;
            hipLaunchKernelGGL(k_gather_c4, dim3(nblocks(nEE)), dim3(kBlock), 0, c.s, idx, oEE.c4, (int)nEE, out.p, nC, (int)nPT);
            CIPC_LAUNCH_CHECK();
        }
        nOut = nC;
        return;
    }
}

// Autotuner of the grid cell size: while it runs, each call uses the next candidate
// multiplier of the mean rest edge length and its wall time is recorded (stream drained
// before and after; two rounds over the candidates); then the fastest multiplier is
// kept.  The constraint set itself does not depend on the cell size.
void constraint_set(Ctx& c, const double* x, DevBuf<int>& out, int& nOut) {
    Ctx::Tuner& T = c.tune;
    if (!T.cell) return constraint_set_impl(c, x, out, nOut);
    c.cellMult = T.cellCand[T.cellIdx];
    CIPC_HIP(hipStreamSynchronize(c.s));
    const auto t0 = std::chrono::steady_clock::now();
    constraint_set_impl(c, x, out, nOut);
    CIPC_HIP(hipStreamSynchronize(c.s));
    T.cellCost[T.cellIdx] = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (++T.cellIdx == (int)T.cellCand.size()) {
        // sum the rounds per multiplier
        const int m = (int)T.cellCand.size() / 2;
        int best = 0;
        for (int i = 1; i < m; ++i)
            if (T.cellCost[i] + T.cellCost[i + m] < T.cellCost[best] + T.cellCost[best + m]) best = i;
        c.cellMult = T.cellCand[best];
        T.cell = false;
    }
}

// ------------------------------------------------------------------ per-constraint evaluation
struct LocalC {
    int nv;
    int vid[4];
    double d2;
};

// decode a constraint (reference encoding) into its 4-vertex stencil; for mollified
// entries the stencil is the two edges (edgeVInd of IPC.h:831, 845, 859)
// entry k of constraint i at C[k * sk + i * si]: the library's SoA layout (sk = nC, si =
// 1) or int4 rows (sk = 1, si = 4)
__device__ __forceinline__ void decode(const int* __restrict__ C, long sk, long si, int i, int* cc, int& kind, int* vid, int& nv,
                                       double& mult) {
#pragma unroll
    for (int k = 0; k < 4; ++k) cc[k] = C[(long)k * sk + (long)i * si];
    mult = 1;
    if (cc[0] >= 0) {
        nv = 4;
        if (cc[2] >= 0 && cc[3] >= 0) { kind = 0; vid[0] = cc[0]; vid[1] = cc[1]; vid[2] = cc[2]; vid[3] = cc[3]; }                  // EE
        else if (cc[3] >= 0) { kind = 1; vid[0] = cc[0]; vid[1] = cc[1]; vid[2] = -cc[2] - 1; vid[3] = cc[3]; }                      // mollified EE
        else if (cc[2] >= 0) { kind = 2; vid[0] = cc[0]; vid[1] = -cc[3] - 1; vid[2] = cc[1]; vid[3] = cc[2]; }                      // mollified PE
        else { kind = 3; vid[0] = cc[0]; vid[1] = -cc[2] - 1; vid[2] = cc[1]; vid[3] = -cc[3] - 1; }                                 // mollified PP
    } else {
        vid[0] = -cc[0] - 1;
        if (cc[3] >= 0) { kind = 4; nv = 4; vid[1] = cc[1]; vid[2] = cc[2]; vid[3] = cc[3]; }                                        // PT
        else if (cc[2] >= 0) { kind = 5; nv = 3; vid[1] = cc[1]; vid[2] = cc[2]; vid[3] = -1; mult = -cc[3]; }                       // PE
        else { kind = 6; nv = 2; vid[1] = cc[1]; vid[2] = -1; vid[3] = -1; mult = -cc[3]; }                                          // PP
    }
}
__device__ __forceinline__ double con_dist2(const double* __restrict__ x, int kind, const int* vid) {
#pragma clang fp contract(off)
    switch (kind) {
        case 0: case 1: return dist2_ee(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), ld3(x, vid[3]));
        case 2: return dist2_pe(ld3(x, vid[0]), ld3(x, vid[2]), ld3(x, vid[3]));
        case 3: return dist2_pp(ld3(x, vid[0]), ld3(x, vid[2]));
        case 4: return dist2_pt(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), ld3(x, vid[3]));
        case 5: return dist2_pe(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]));
        default: return dist2_pp(ld3(x, vid[0]), ld3(x, vid[1]));
    }
}

// ROWS: C is int4 rows checked against [0, nV) after decoding (device-resident input the
// host never saw; an entry out of range contributes nothing and sets bit 2 of *bad),
// else the library's own SoA set
template <bool ROWS>
__global__ void k_barrier_energy(const double* __restrict__ x, const double* __restrict__ X0, const int* __restrict__ C, int nC,
                                 double kappa, double xi2, double shat, double* __restrict__ partial, uint32_t* __restrict__ bad,
                                 int nV) {
    __shared__ double lds[4];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0;
    if (i < nC) {
        int cc[4], vid[4], kind, nv;
        double mult;
        decode(C, ROWS ? 1 : nC, ROWS ? 4 : 1, i, cc, kind, vid, nv, mult);
        bool inRange = true;
        if (ROWS) {
#pragma unroll
            for (int k = 0; k < 4; ++k) inRange = inRange && cc[k] >= -nV && cc[k] < nV && (k >= nv || (vid[k] >= 0 && vid[k] < nV));
        }
        double d2 = inRange ? con_dist2(x, kind, vid) : 1.0;
        double s = d2 - xi2;
        if (!inRange) {
            atomicOr(bad, 2u);
        } else if (s <= 0) {
            atomicOr(bad, 1u);
        } else {
            double b = barrier_e(s, shat, kappa);
            if (kind >= 1 && kind <= 3) {
                double eps = ee_mollifier_threshold(ld3(X0, vid[0]), ld3(X0, vid[1]), ld3(X0, vid[2]), ld3(X0, vid[3]));
                double m = ee_mollifier(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), ld3(x, vid[3]), eps);
                e = b * m;
            } else {
                e = (cc[3] < -1) ? b * mult : b;
            }
        }
    }
    double t = block_sum_256(e, lds);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// distance gradient of a constraint embedded into its 4-vertex stencil
__device__ __forceinline__ void con_dist_grad(const double* __restrict__ x, int kind, const int* vid, double* gd) {
#pragma unroll
    for (int i = 0; i < 12; ++i) gd[i] = 0;
    switch (kind) {
        case 0: case 1:
            dist2_ee_g(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), ld3(x, vid[3]), gd);
            break;
        case 4:
            dist2_pt_g(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), ld3(x, vid[3]), gd);
            break;
        case 2: {   // PE over stencil slots (0, 2, 3)
            double g9[9];
            dist2_pe_g(ld3(x, vid[0]), ld3(x, vid[2]), ld3(x, vid[3]), g9);
#pragma unroll
            for (int k = 0; k < 3; ++k) { gd[k] = g9[k]; gd[6 + k] = g9[3 + k]; gd[9 + k] = g9[6 + k]; }
            break;
        }
        case 3: {   // PP over stencil slots (0, 2)
            double g6[6];
            dist2_pp_g(ld3(x, vid[0]), ld3(x, vid[2]), g6);
#pragma unroll
            for (int k = 0; k < 3; ++k) { gd[k] = g6[k]; gd[6 + k] = g6[3 + k]; }
            break;
        }
        case 5:     // PE, native 3-vertex layout
            dist2_pe_g(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), gd);
            break;
        default:    // PP
            dist2_pp_g(ld3(x, vid[0]), ld3(x, vid[1]), gd);
            break;
    }
}

// local gradients: SoA [3][4 nC] plus the vertex of each slot (-1 when unused or
// when the barrier is not evaluated)
__global__ void k_barrier_grad_local(const double* __restrict__ x, const double* __restrict__ X0, const int* __restrict__ C, int nC,
                                     double kappa, double xi2, double shat, double* __restrict__ gl, int* __restrict__ gv) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nC) return;
    int cc[4], vid[4], kind, nv;
    double mult;
    decode(C, nC, 1, i, cc, kind, vid, nv, mult);
    double d2 = con_dist2(x, kind, vid);
    double s = d2 - xi2;
    long ns = 4l * nC;
    if (!(s > 0)) {
#pragma unroll
        for (int a = 0; a < 4; ++a) gv[4l * i + a] = -1;
        return;
    }
    double gd[12];
    con_dist_grad(x, kind, vid, gd);
    double bg = barrier_g(s, shat, kappa);
    double gout[12];
    if (kind >= 1 && kind <= 3) {
        double eps = ee_mollifier_threshold(ld3(X0, vid[0]), ld3(X0, vid[1]), ld3(X0, vid[2]), ld3(X0, vid[3]));
        double ge[12];
        double m = ee_mollifier_g(ld3(x, vid[0]), ld3(x, vid[1]), ld3(x, vid[2]), ld3(x, vid[3]), eps, ge);
        double b = barrier_e(s, shat, kappa);
#pragma unroll
        for (int k = 0; k < 12; ++k) gout[k] = m * bg * gd[k] + b * ge[k];
    } else {
#pragma unroll
        for (int k = 0; k < 12; ++k) gout[k] = mult * bg * gd[k];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        bool used = a < nv;
        gv[4l * i + a] = used ? vid[a] : -1;
#pragma unroll
        for (int k = 0; k < 3; ++k) gl[k * ns + 4l * i + a] = used ? gout[a * 3 + k] : 0.0;
    }
}

// Local barrier Hessians, projected.  A distance depends on its NV points through NV - 1
// differences only, so the Hessian is formed over those (9 x 9 at most, 45 upper entries)
// and taken to the orthonormal basis of the translation complement by the small constant
// matrix between the two, where the positive part is formed: one constraint per thread,
// in registers from the positions to the blocks.  Point-plane and edge-edge share the form
// (w . (a x b))^2 / |a x b|^2 over (w, a, b); the mollified point-edge and point-point
// cases of an edge pair are functions of the same (w, a, b).
// Bound by the rotations' arithmetic at one wave per SIMD.  12 x 12 Hessians written by one
// kernel (2.3 KB of scratch per thread) and projected by a second took 1,165 + 1,840 us for
// 1.2 million contacts, this 971; 33 + 157 -> 82 us at 20 contacts, the latency of one wave.
//
// Coefficients of the differences over the basis column p: sum_k D[s][k] tr_basis(k, p)
// with w = v2 - v0, a = v1 - v0, b = v3 - v2 (edge-edge) or w = v0 - v1, a = v2 - v1,
// b = v3 - v1 (point-triangle); u = v1 - v0, v = v2 - v0 (point-edge).
template <bool PT>
__device__ __forceinline__ constexpr double diff4(int s, int p) {
    return PT ? (s == 0 ? tr_basis<4>(0, p) - tr_basis<4>(1, p) : s == 1 ? tr_basis<4>(2, p) - tr_basis<4>(1, p) : tr_basis<4>(3, p) - tr_basis<4>(1, p))
              : (s == 0 ? tr_basis<4>(2, p) - tr_basis<4>(0, p) : s == 1 ? tr_basis<4>(1, p) - tr_basis<4>(0, p) : tr_basis<4>(3, p) - tr_basis<4>(2, p));
}
__device__ __forceinline__ constexpr double diff3(int s, int p) { return tr_basis<3>(s + 1, p) - tr_basis<3>(0, p); }
template <int ND, class Coef>
__device__ __forceinline__ void to_reduced(const double* H, double* a, Coef coef) {
#pragma unroll
    for (int p = 0; p < ND; ++p)
#pragma unroll
        for (int q = 0; q < ND; ++q)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    if (q < p || (p == q && j < i)) continue;
                    double v = 0;
#pragma unroll
                    for (int s = 0; s < ND; ++s)
#pragma unroll
                        for (int t = 0; t < ND; ++t) {
                            const double f = coef(s, p) * coef(t, q);
                            if (f != 0.0) v += f * H[upk(9, 3 * s + i, 3 * t + j)];
                        }
                    a[upk(9, 3 * p + i, 3 * q + j)] = v;
                }
}
__global__ void __launch_bounds__(64) k_barrier_hess(const double* __restrict__ x, const double* __restrict__ X0,
                                                     const int* __restrict__ C, int nC, double kappa, double xi2, double shat,
                                                     double* __restrict__ hl) {
    __shared__ double lds[kEmitLds];
    const int i0 = blockIdx.x * 64, i = i0 + threadIdx.x;
    double a[45];
#pragma unroll
    for (int e = 0; e < 45; ++e) a[e] = 0.0;
    int n = 0;
    if (i < nC) {
        int cc[4], vid[4], kind, nv;
        double mult;
        decode(C, nC, 1, i, cc, kind, vid, nv, mult);
        const double s = con_dist2(x, kind, vid) - xi2;
        n = nv;   // blocks of a constraint that is not evaluated are zero
        if (s > 0) {
            const double bg = barrier_g(s, shat, kappa), bh = barrier_h(s, shat, kappa);
            const d3 p0 = ld3(x, vid[0]), p1 = ld3(x, vid[1]);
            if (kind == 6) {
                // 2 I and 2 d over the one difference d; the reduced matrix is
                // 2 mult (4 bh d d^T + 2 bg I), whose positive part is known
                const d3 d = p0 - p1;
                const double across = 4.0 * mult * bg > 0 ? 4.0 * mult * bg : 0.0;
                const double l2 = sq(d), along0 = 2.0 * mult * (4.0 * bh * l2 + 2.0 * bg), along = along0 > 0 ? along0 : 0.0;
                const double f = (along - across) / l2;
                a[upk(9, 0, 0)] = across + f * d.x * d.x; a[upk(9, 0, 1)] = f * d.x * d.y; a[upk(9, 0, 2)] = f * d.x * d.z;
                a[upk(9, 1, 1)] = across + f * d.y * d.y; a[upk(9, 1, 2)] = f * d.y * d.z; a[upk(9, 2, 2)] = across + f * d.z * d.z;
            } else {
                const d3 p2 = ld3(x, vid[2]);
                const d3 p3 = nv == 4 ? ld3(x, vid[3]) : p2;
                double g[9], H[45];   // over (w, a, b), or (u, v) of a point-edge pair
                double fg = mult * bh, fh = mult * bg;
                d3 w, ea, eb;
                if (kind == 4) { w = p0 - p1; ea = p2 - p1; eb = p3 - p1; }
                else { w = p2 - p0; ea = p1 - p0; eb = p3 - p2; }
#pragma unroll
                for (int e = 0; e < 9; ++e) g[e] = 0;
#pragma unroll
                for (int e = 0; e < 45; ++e) H[e] = 0;
                if (kind == 2 || kind == 5) {
                    double gv[6], Hv[36];
                    pe_dist_derivs<true>(kind == 5 ? ea : w, kind == 5 ? w : p3 - p0, gv, Hv);
                    if (kind == 5) {
#pragma unroll
                        for (int r = 0; r < 6; ++r) {
                            g[r] = gv[r];
#pragma unroll
                            for (int c = 0; c < 6; ++c)
                                if (c >= r) H[upk(9, r, c)] = Hv[6 * r + c];
                        }
                    } else {   // u = w, v = w + b
#pragma unroll
                        for (int r = 0; r < 3; ++r) {
                            g[r] = gv[r] + gv[3 + r];
                            g[6 + r] = gv[3 + r];
#pragma unroll
                            for (int c = 0; c < 3; ++c) {
                                const double uv = Hv[6 * r + 3 + c], vv = Hv[6 * (3 + r) + 3 + c];
                                if (c >= r) {
                                    H[upk(9, r, c)] = Hv[6 * r + c] + uv + Hv[6 * (3 + r) + c] + vv;
                                    H[upk(9, 6 + r, 6 + c)] = vv;
                                }
                                H[upk(9, r, 6 + c)] = uv + vv;
                            }
                        }
                    }
                } else if (kind == 3) {
                    put_vec(g, 0, 2.0 * w);
                    H[upk(9, 0, 0)] = H[upk(9, 1, 1)] = H[upk(9, 2, 2)] = 2.0;
                } else {
                    plane_dist_derivs<true>(w, ea, eb, g, H);
                }
                double ge[6], He[36], b = 0, m = 1;
                const bool moll = kind >= 1 && kind <= 3;
                if (moll) {
                    const double eps = ee_mollifier_threshold(ld3(X0, vid[0]), ld3(X0, vid[1]), ld3(X0, vid[2]), ld3(X0, vid[3]));
                    m = ee_mollifier_diff<2>(p0, p1, p2, p3, eps, ge, He);
                    b = barrier_e(s, shat, kappa);
                    fg = m * bh;
                    fh = m * bg;
                }
#pragma unroll
                for (int r = 0; r < 9; ++r)
#pragma unroll
                    for (int c = 0; c < 9; ++c)
                        if (c >= r) H[upk(9, r, c)] = fg * g[r] * g[c] + fh * H[upk(9, r, c)];
                if (moll) {
#pragma unroll
                    for (int r = 0; r < 9; ++r)
#pragma unroll
                        for (int c = 3; c < 9; ++c) {
                            if (c < r) continue;
                            double v = g[r] * ge[c - 3];
                            if (r >= 3) v += ge[r - 3] * g[c];
                            v *= bg;
                            if (r >= 3) v += b * He[6 * (r - 3) + c - 3];
                            H[upk(9, r, c)] += v;
                        }
                }
                if (nv == 3) to_reduced<2>(H, a, [](int sl, int p) { return diff3(sl, p); });
                else if (kind == 4) to_reduced<3>(H, a, [](int sl, int p) { return diff4<true>(sl, p); });
                else to_reduced<3>(H, a, [](int sl, int p) { return diff4<false>(sl, p); });
            }
        }
    }
    const bool any4 = __any(n == 4);
    if (n >= 3) {
        // a positive definite matrix is its own positive part
        bool pd = true;
        double L[45], inv[9];
#pragma unroll
        for (int r = 0; r < 9; ++r)
#pragma unroll
            for (int c = 0; c <= r; ++c) {   // L D L^T, L(r, c) D(c) kept
                double sum = a[upk(9, c, r)];
#pragma unroll
                for (int k = 0; k < c; ++k) sum -= L[upk(9, k, r)] * (L[upk(9, k, c)] * inv[k]);
                L[upk(9, c, r)] = sum;
                if (r == c) {
                    const bool used = r < 6 || n == 4;
                    pd = pd && (sum > 0 || !used);
                    inv[r] = 1.0 / (sum > 0 ? sum : 1.0);
                }
            }
        if (!pd) {
            if (any4) jacobi_psd<9, 9, true>(a);
            else jacobi_psd<6, 9, true>(a);
        }
    }
    emit_blocks(n, nC - i0, lds, hl + 9 * 16l * i0, [&](int k, double* row) {
        if (n == 4) expand_row<4>(a, k, row);
        else if (n == 3 && k < 3) expand_row<3>(a, k, row);
        else if (n == 2 && k < 2) expand_row<2>(a, k, row);
    });
}

__global__ void k_con_dist2(const double* __restrict__ x, const int* __restrict__ C, int nC, double* __restrict__ d2,
                            double* __restrict__ partial) {
    __shared__ double lds[4];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 1e300;
    if (i < nC) {
        int cc[4], vid[4], kind, nv;
        double mult;
        decode(C, nC, 1, i, cc, kind, vid, nv, mult);
        v = con_dist2(x, kind, vid);
        if (d2) d2[i] = v;
    }
    double m = block_min_256(v, lds);
    if (threadIdx.x == 0) partial[blockIdx.x] = m;
}
// one workgroup: a lone thread waited on one load per partial (205 us for the 5000 of a
// 1.2 million contact set)
__global__ void __launch_bounds__(kBlock) k_min_partials(const double* __restrict__ partial, int n, double* __restrict__ out) {
    __shared__ double lds[4];
    double m = 1e300;
    for (int i = threadIdx.x; i < n; i += kBlock) m = partial[i] < m ? partial[i] : m;
    m = block_min_256(m, lds);
    if (threadIdx.x == 0) *out = m;
}

// ------------------------------------------------------------------ host wrappers
double barrier_energy(Ctx& c, const double* x, const int* C, int nC, double kappa, int* bad) {
    if (nC == 0) { if (bad) *bad = 0; return 0.0; }
    const double xi2 = c.P.xi * c.P.xi, shat = c.dHat2 + 2 * std::sqrt(c.dHat2) * c.P.xi;   // IPC.h:756-757
    int nb = nblocks(nC);
    double* part = c.red.ensure(nb);
    CIPC_HIP(hipMemsetAsync(c.counters.p + 12, 0, sizeof(uint32_t), c.s));
    hipLaunchKernelGGL(k_barrier_energy<false>, dim3(nb), dim3(kBlock), 0, c.s, x, c.X0.p, C, nC, kappa, xi2, shat, part, c.counters.p + 12,
                       c.nV);
    CIPC_LAUNCH_CHECK();
    sum_partials(part, nb, c.scal.p + 1, c.s);
    CIPC_HIP(hipMemcpyAsync(c.hScal + 1, c.scal.p + 1, sizeof(double), hipMemcpyDeviceToHost, c.s));
    CIPC_HIP(hipMemcpyAsync(c.hCnt + 12, c.counters.p + 12, sizeof(uint32_t), hipMemcpyDeviceToHost, c.s));
    CIPC_HIP(hipStreamSynchronize(c.s));
    if (bad) *bad = c.hCnt[12] ? 1 : 0;
    return c.hScal[1];
}

__global__ void k_clear_u32(uint32_t* __restrict__ a, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0u;
}
// The same energy over int4 constraint rows (C[4 i + k], the reference's layout) with every
// buffer supplied by the caller: per-block partials part[nblocks(nC)], the sum *out and
// the validity bits *bad (bit 1: a distance at or below the offset, bit 2: an entry
// outside the vertex range), all device memory.  *bad is cleared by a fill kernel.
// Nothing is allocated and nothing is synchronised; the launches go to c.s.
void barrier_energy_rows(Ctx& c, const double* x, const int* Crows, int nC, double kappa, double* part, double* out, uint32_t* bad) {
    const double xi2 = c.P.xi * c.P.xi, shat = c.dHat2 + 2 * std::sqrt(c.dHat2) * c.P.xi;   // IPC.h:756-757
    hipLaunchKernelGGL(k_clear_u32, dim3(1), dim3(64), 0, c.s, bad, 1);
    CIPC_LAUNCH_CHECK();
    if (nC == 0) {
        hipLaunchKernelGGL(k_clear_u32, dim3(1), dim3(64), 0, c.s, reinterpret_cast<uint32_t*>(out), 2);   // +0.0
        CIPC_LAUNCH_CHECK();
        return;
    }
    const int nb = nblocks(nC);
    hipLaunchKernelGGL(k_barrier_energy<true>, dim3(nb), dim3(kBlock), 0, c.s, x, c.X0.p, Crows, nC, kappa, xi2, shat, part, bad, c.nV);
    CIPC_LAUNCH_CHECK();
    sum_partials(part, nb, out, c.s);
}

__global__ void k_vert_bounds(const uint64_t* __restrict__ key, long n, int nV, uint32_t* __restrict__ start, uint32_t* __restrict__ end) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t k = key[i];
    if (k >= (uint64_t)nV) return;
    if (i == 0 || key[i - 1] != k) start[k] = (uint32_t)i;
    if (i == n - 1 || key[i + 1] != k) end[k] = (uint32_t)(i + 1);
}
// slots of vertices flagged in `skip` (rows the caller projects out) are not gathered: a
// static obstacle's vertex (a ground corner) can sit in 10^5 stencils, which one thread
// would otherwise sum serially
__global__ void k_grad_keys(const int* __restrict__ gv, long n, int nV, const uint8_t* __restrict__ skip, uint64_t* __restrict__ key) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int v = gv[i];
    key[i] = (v < 0 || (skip && skip[v])) ? (uint64_t)nV : (uint64_t)v;
}
// Eight lanes per vertex fetch eight slots at a time, the next eight while these are added in
// slot order: a vertex that many stencils touch was one thread's chain of loads.
// Measured: 171 -> 86 us on 4 sheets of 201 x 201 in contact, 46 -> 28 on 101 x 101 (one thread
// with eight slots in flight: 52).
constexpr int kGatherLanes = 8;
__global__ void k_grad_gather(const double* __restrict__ gl, long ns, const uint32_t* __restrict__ slot, const uint32_t* __restrict__ start,
                              const uint32_t* __restrict__ end, int nV, double* __restrict__ g) {
    const int lane = threadIdx.x % kGatherLanes;
    const int v = (int)(((long)blockIdx.x * blockDim.x + threadIdx.x) / kGatherLanes);
    const uint32_t s = v < nV ? start[v] : 0, e = v < nV ? end[v] : 0;
    double sum = 0;   // lanes 0, 1, 2: x, y, z
    double na = 0, nb = 0, nd = 0;
    auto fetch = [&](uint32_t k) {
        const bool on = k + lane < e;
        const long q = on ? slot[k + lane] : 0;
        na = on ? gl[q] : 0.0;
        nb = on ? gl[ns + q] : 0.0;
        nd = on ? gl[2 * ns + q] : 0.0;
    };
    if (s < e) fetch(s);
    for (uint32_t k = s; k < e; k += kGatherLanes) {
        const double a = na, b = nb, d = nd;
        if (k + kGatherLanes < e) fetch(k + kGatherLanes);
#pragma unroll
        for (int u = 0; u < kGatherLanes; ++u) {
            const double x = __shfl(a, u, kGatherLanes), y = __shfl(b, u, kGatherLanes), z = __shfl(d, u, kGatherLanes);
            sum += lane == 0 ? x : lane == 1 ? y : z;   // past the end: + 0
        }
    }
    if (v < nV && lane < 3) g[3 * v + lane] += sum;
}

// g += barrier gradient (deterministic: slots sorted by vertex, summed in slot order)
void barrier_gradient(Ctx& c, const double* x, const int* C, int nC, double kappa, double* g, const uint8_t* skip) {
    if (nC == 0) return;
    const double xi2 = c.P.xi * c.P.xi, shat = c.dHat2 + 2 * std::sqrt(c.dHat2) * c.P.xi;
    long ns = 4l * nC;
    double* gl = c.conGLocal.ensure(3 * ns);
    int* gv = c.conGVert.ensure(ns);
    hipLaunchKernelGGL(k_barrier_grad_local, dim3(nblocks(nC)), dim3(kBlock), 0, c.s, x, c.X0.p, C, nC, kappa, xi2, shat, gl, gv);
    CIPC_LAUNCH_CHECK();
    scatter_local_gradient(c, gl, gv, ns, g, skip);
}

// g += local gradient slots (SoA [3][ns], vertex gv per slot, -1 unused), summed per
// vertex in slot order (radix sort by vertex, stable); vertices flagged in skip keep g
void scatter_local_gradient(Ctx& c, const double* gl, const int* gv, long ns, double* g, const uint8_t* skip) {
    uint64_t* key = c.k64a.ensure(ns);
    uint32_t* slot = c.u32c.ensure(ns);
    hipLaunchKernelGGL(k_grad_keys, dim3(nblocks(ns)), dim3(kBlock), 0, c.s, gv, ns, c.nV, skip, key);
    CIPC_LAUNCH_CHECK();
    const SortedPairs sorted = radix_sort_pairs(key, slot, ns, bits_for((uint64_t)c.nV + 1), c.pw, c.s);
    uint32_t* st = c.u32a.ensure(c.nV);
    uint32_t* en = c.u32b.ensure(c.nV);
    CIPC_HIP(hipMemsetAsync(st, 0, c.nV * sizeof(uint32_t), c.s));
    CIPC_HIP(hipMemsetAsync(en, 0, c.nV * sizeof(uint32_t), c.s));
    hipLaunchKernelGGL(k_vert_bounds, dim3(nblocks(ns)), dim3(kBlock), 0, c.s, (const uint64_t*)sorted.keys, ns, c.nV, st, en);
    CIPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_grad_gather, dim3(nblocks((long)c.nV * kGatherLanes)), dim3(kBlock), 0, c.s, gl, ns, (const uint32_t*)sorted.vals, st, en, c.nV, g);
    CIPC_LAUNCH_CHECK();
}

// Blocks in a Dirichlet row or column are zero after Project_DBC (Math/CSR_MATRIX.h:
// 130-141) and are not stored: a Dirichlet vertex of a static obstacle (a ground corner)
// touches every stencil near it, and its row would otherwise hold a block per contact.
__global__ void k_hess_keys(const int* __restrict__ C, int nC, int nV, const uint8_t* __restrict__ dbc, uint64_t* __restrict__ key) {
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= 16l * nC) return;
    int i = (int)(q / 16), a = (int)((q / 4) % 4), b = (int)(q % 4);
    int cc[4], vid[4], kind, nv;
    double mult;
    decode(C, nC, 1, i, cc, kind, vid, nv, mult);
    const bool keep = a < nv && b < nv && !dbc[vid[a]] && !dbc[vid[b]];
    key[q] = keep ? (uint64_t)vid[a] * (uint64_t)nV + (uint64_t)vid[b] : (uint64_t)nV * (uint64_t)nV;
}
__global__ void k_bsr_from_sorted(const uint64_t* __restrict__ key, long n, int nV, uint32_t* __restrict__ head) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    head[i] = (key[i] < (uint64_t)nV * nV && (i == 0 || key[i] != key[i - 1])) ? 1u : 0u;
}
// Sum the local blocks of each unique (row, col) into the contact BSR; Dirichlet rows and
// columns are zeroed (Project_DBC).  A wave takes 64 sorted entries: their blocks (72 bytes
// each, anywhere) come to LDS by nine independent loads per lane, then the first entry of
// every run sums its run in order.  A run's rest beyond the wave is read directly.
// Bound by the blocks' arrival; one run per thread with nine strided planes took 1,686 us for
// the 19 million slots of 1.2 million contacts, this 827 (14 -> 9.5 us at 20 contacts).
__global__ void __launch_bounds__(kBlock) k_bsr_sum(const uint64_t* __restrict__ key, long n, int nV, const uint32_t* __restrict__ pos,
                                                    const uint32_t* __restrict__ slot, const double* __restrict__ hl,
                                                    const uint8_t* __restrict__ dbc, int nnzb, int* __restrict__ rowOf,
                                                    int* __restrict__ col, double* __restrict__ val) {
    __shared__ double blk[kBlock / 64][64 * 9];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long i0 = (long)blockIdx.x * kBlock + 64 * w, i = i0 + lane;
    const uint64_t none = (uint64_t)nV * nV;
    const uint64_t k = i < n ? key[i] : none;
    const bool used = k < none;
    const uint32_t q = used ? slot[i] : 0;
    const uint64_t before = i > 0 && used ? key[i - 1] : none;
    double v[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) {
        const int o = lane + 64 * m, t = o / 9;
        const uint32_t qt = (uint32_t)__shfl((int)q, t);
        v[m] = __shfl((int)used, t) ? hl[9 * (long)qt + (o - 9 * t)] : 0.0;
    }
#pragma unroll
    for (int m = 0; m < 9; ++m) blk[w][lane + 64 * m] = v[m];
    __syncthreads();
    if (!used || before == k) return;
    double acc[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) acc[m] = blk[w][9 * lane + m];
    long j = i + 1;
    const long end = n < i0 + 64 ? n : i0 + 64;
    for (; j < end && key[j] == k; ++j) {
#pragma unroll
        for (int m = 0; m < 9; ++m) acc[m] += blk[w][9 * (int)(j - i0) + m];
    }
    if (j == end)
        for (; j < n && key[j] == k; ++j) {
            const long qj = slot[j];
#pragma unroll
            for (int m = 0; m < 9; ++m) acc[m] += hl[9 * qj + m];
        }
    int r = (int)(k / (uint64_t)nV), cl = (int)(k % (uint64_t)nV);
    bool z = dbc[r] || dbc[cl];
    int o = (int)pos[i];
    rowOf[o] = r;
    col[o] = cl;
#pragma unroll
    for (int m = 0; m < 9; ++m) val[(long)m * nnzb + o] = z ? 0.0 : acc[m];
}
// rowptr[r] = first block of a row >= r (rowOf sorted): one binary search per row, so
// long runs of empty rows (Dirichlet obstacles) cost no serial loop
__global__ void k_rowptr(const int* __restrict__ rowOf, int nnzb, int nrow, int* __restrict__ rowptr) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nrow) return;
    int lo = 0, hi = nnzb;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (rowOf[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    rowptr[r] = lo;
}

// contact BSR: barrier blocks of C and, when fricXn is given, the friction blocks of the
// lagged friction stencils (slots 16 nC onwards), summed per (row, col)
void barrier_hessian(Ctx& c, const double* x, const int* C, int nC, double kappa, const double* fricXn) {
    BSR& A = c.Acon;
    A.nrow = c.nV;
    const int nF = fricXn ? c.nF : 0;
    if (nC + nF == 0) {
        A.nnzb = 0;
        A.rowptr.ensure(c.nV + 1);
        CIPC_HIP(hipMemsetAsync(A.rowptr.p, 0, (c.nV + 1) * sizeof(int), c.s));
        return;
    }
    const double xi2 = c.P.xi * c.P.xi, shat = c.dHat2 + 2 * std::sqrt(c.dHat2) * c.P.xi;
    long ns = 16l * (nC + nF);
    double* hl = c.conLocal.ensure(9 * ns);
    uint64_t* key = c.k64b.ensure(ns);
    uint32_t* slot = c.u32d.ensure(ns);
    if (nC) {
        hipLaunchKernelGGL(k_barrier_hess, dim3(nblocks(nC, 64)), dim3(64), 0, c.s, x, c.X0.p, C, nC, kappa, xi2, shat, hl);
        CIPC_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_hess_keys, dim3(nblocks(16l * nC)), dim3(kBlock), 0, c.s, C, nC, c.nV, proj_mask(c), key);
        CIPC_LAUNCH_CHECK();
    }
    if (nF) {
        friction_hess_local(c, x, fricXn, hl, 16l * nC);
        friction_hess_keys(c, key + 16l * nC);
    }
    const SortedPairs sorted = radix_sort_pairs(key, slot, ns, bits_for((uint64_t)c.nV * c.nV + 1), c.pw, c.s);
    const uint64_t* skey = sorted.keys;
    uint32_t* head = c.u32a.ensure(ns);
    uint32_t* pos = c.u32b.ensure(ns);
    hipLaunchKernelGGL(k_bsr_from_sorted, dim3(nblocks(ns)), dim3(kBlock), 0, c.s, skey, ns, c.nV, head);
    CIPC_LAUNCH_CHECK();
    scan_exclusive(head, pos, ns, c.counters.p + 5, c.pw, c.s);
    CIPC_HIP(hipMemcpyAsync(c.hCnt + 5, c.counters.p + 5, sizeof(uint32_t), hipMemcpyDeviceToHost, c.s));
    CIPC_HIP(hipStreamSynchronize(c.s));
    int nnzb = (int)c.hCnt[5];
    A.nnzb = nnzb;
    A.rowOf.ensure(std::max(nnzb, 1));
    A.col.ensure(std::max(nnzb, 1));
    A.val.ensure(9l * std::max(nnzb, 1));
    A.rowptr.ensure(c.nV + 1);
    hipLaunchKernelGGL(k_bsr_sum, dim3(nblocks(ns)), dim3(kBlock), 0, c.s, skey, ns, c.nV, pos, (const uint32_t*)sorted.vals, hl, proj_mask(c), nnzb,
                       A.rowOf.p, A.col.p, A.val.p);
    CIPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_rowptr, dim3(nblocks(c.nV + 1)), dim3(kBlock), 0, c.s, A.rowOf.p, nnzb, c.nV, A.rowptr.p);
    CIPC_LAUNCH_CHECK();
}

double min_dist2(Ctx& c, const double* x, const int* C, int nC, double* d2out) {
    if (nC == 0) return 1e300;
    int nb = nblocks(nC);
    double* part = c.red.ensure(nb);
    hipLaunchKernelGGL(k_con_dist2, dim3(nb), dim3(kBlock), 0, c.s, x, C, nC, d2out, part);
    CIPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_min_partials, dim3(1), dim3(kBlock), 0, c.s, part, nb, c.scal.p + 2);
    CIPC_LAUNCH_CHECK();
    CIPC_HIP(hipMemcpyAsync(c.hScal + 2, c.scal.p + 2, sizeof(double), hipMemcpyDeviceToHost, c.s));
    CIPC_HIP(hipStreamSynchronize(c.s));
    return c.hScal[2] - c.P.xi * c.P.xi;
}

}  // namespace cipc
