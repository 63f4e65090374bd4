// Direct solve of the Newton system for small scenes: the reference factorises every
// Newton matrix with CHOLMOD (Math/DIRECT_SOLVER.h:14-66, stype -1) and reports a
// non-positive pivot as CHOLMOD_NOT_POSDEF, after which the step takes a gradient-descent
// direction (IMPLICIT_EULER.h:515-554).  Here: the assembled FP64 matrix (elastic BSR +
// contact BSR, Dirichlet rows already projected) is expanded into a dense row-major array
// padded to whole 64 x 64 tiles (identity on the padding) and factorised by a tiled
// right-looking Cholesky -- one workgroup per tile for the diagonal factor, the panel
// solves and the trailing updates -- then solved by tiled forward and backward
// substitution.  Dense, so limited to kDirectMaxDof unknowns (4.5 GiB of FP64 matrix); it
// is the fallback of the PCG solves for such scenes and a selectable solver.
#include "ctx.hpp"
#include <algorithm>
#include <cmath>

namespace cipc {

constexpr int kDT = 64;          // tile edge
constexpr int kDirectBlock = 256;

__global__ void k_dense_zero(double* __restrict__ a, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) a[i] = 0.0;
}
__global__ void k_dense_pad_identity(double* __restrict__ a, long ld, int n, int npad) {
    const int i = n + blockIdx.x * blockDim.x + threadIdx.x;
    if (i < npad) a[(long)i * ld + i] = 1.0;
}
// one thread per stored block: A[3 r + a][3 c + b] (+)= block; the BSR holds each (r, c)
// once, so a pattern's blocks never collide (the contact BSR is added after the elastic)
__global__ void k_dense_scatter(const int* __restrict__ rowOf, const int* __restrict__ col, const double* __restrict__ val, int nnzb,
                                double* __restrict__ a, long ld, int add) {
    const int blk = blockIdx.x * blockDim.x + threadIdx.x;
    if (blk >= nnzb) return;
    const long r = rowOf[blk], c = col[blk];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double* dst = a + (3 * r + i) * ld + 3 * c + j;
            const double v = val[(long)(3 * i + j) * nnzb + blk];
            *dst = add ? *dst + v : v;
        }
}

__device__ __forceinline__ double lane_read(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane), __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// s / d from the correctly rounded reciprocal r of d: one residual step
__device__ __forceinline__ double div_by(double s, double d, double r) {
    const double q = s * r;
    return fma(fma(-q, d, s), r, q);
}

// sqrt(d) and 1 / sqrt(d) together by Goldschmidt's iteration from the hardware's reciprocal
// square root, with a residual step on the root: a third of the dependent operations of a
// square root followed by a division, which is the tile factor's serial chain.  Pivots near
// the ends of the exponent range take the library functions.
__device__ __forceinline__ void sqrt_and_inverse(double d, double& root, double& inv) {
    if (d > 1e-280 && d < 1e280) {
        const double y = __builtin_amdgcn_rsq(d);
        double g = d * y, h = 0.5 * y;
        double e = fma(-g, h, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
        e = fma(-g, h, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
        root = fma(fma(-g, g, d), h, g);
        inv = 2 * h;
    } else {
        root = sqrt(d);
        inv = 1.0 / root;
    }
}

// A 64 x 64 tile (row-major, leading dimension ld) by 256 threads: 16 entries each as eight
// 16-byte loads, all in flight before the first is stored (a load-store loop waits for each
// in turn, which took longer than the products)
typedef double dt_v2 __attribute__((ext_vector_type(2)));
struct TileRegs {
    dt_v2 v[8];
    __device__ __forceinline__ void load(const double* __restrict__ a, long ld) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = *reinterpret_cast<const dt_v2*>(a + row(q) * ld + col());
    }
    __device__ __forceinline__ static int row(int q) { return 8 * q + (int)(threadIdx.x >> 5); }
    __device__ __forceinline__ static int col() { return 2 * (int)(threadIdx.x & 31); }
    template <int LD>
    __device__ __forceinline__ void put(double (*T)[LD]) const {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            T[row(q)][col()] = v[q].x;
            T[row(q)][col() + 1] = v[q].y;
        }
    }
    template <int LD>
    __device__ __forceinline__ void put_transposed(double (*T)[LD]) const {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            T[col()][row(q)] = v[q].x;
            T[col() + 1][row(q)] = v[q].y;
        }
    }
};

// Cholesky of diagonal tile k (lower, in place) by four waves: wave h keeps columns
// [16h, 16h+16) of every row (lane = row) in registers.  Panel by panel: wave p eliminates
// its own 16 columns without a barrier (pivot and multipliers cross lanes by readlane),
// publishes them in LDS, and after one barrier the later waves apply all 16 columns to
// theirs.  The serial chain is the 64 square roots and divisions; two barriers per column
// (as with the columns published one by one) had cost more than the arithmetic.
// Measured (us per tile without / with the inverse): 40 / 58 -> 26 / 41.
// A non-positive pivot sets *bad and continues with pivot 1 so that the factorisation
// stays finite.  With diag0, a pivot at or below tau x diag0 (the unknown's diagonal
// before elimination: a mode the matrix does not see) is dropped instead: a pivot at the
// unknown's own scale, zero column, dropped[] = 1.  With inv, the inverse of the factored
// tile is written there too.  Every sum runs in a fixed order: trailing updates in
// column order, substitution sums in index order.
static_assert(kDirectBlock == 4 * kDT, "the tile factor runs four waves of one lane per row");
__device__ __forceinline__ void potrf_tile(double* a, long ld, int k, int* __restrict__ bad, const double* __restrict__ diag0,
                                           int* __restrict__ dropped, double tau, double* __restrict__ inv, double (*T)[kDT + 1],
                                           double (*X)[kDT + 1], double* rd) {
    const int tid = threadIdx.x, i = tid & 63, h = tid >> 6;
    const long o = (long)k * kDT;
    const double dg0 = diag0 ? diag0[o + i] : 0.0;
    TileRegs tr;
    tr.load(a + o * ld + o, ld);
    tr.put(T);
    __syncthreads();
    double row[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) row[q] = T[i][16 * h + q];
    for (int p = 0; p < 4; ++p) {
        if (h == p) {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int J = 16 * p + j;
                double d = lane_read(row[j], J);
                int dr = 0;
                bool neg = false;
                if (diag0) {
                    const double d0 = lane_read(dg0, J);
                    if (!(d > tau * d0)) {
                        dr = 1;
                        d = d0 > 0 ? d0 : 1.0;
                    }
                } else if (!(d > 0)) {
                    neg = true;
                    d = 1.0;
                }
                if (i == J) {
                    if (diag0) dropped[o + J] = dr;
                    else if (neg) atomicOr(bad, 1);
                }
                double pv, ri;
                sqrt_and_inverse(d, pv, ri);
                const double lm = i > J && !dr ? div_by(row[j], pv, ri) : 0.0;   // multiplier of this row
                row[j] = i == J ? pv : lm;
#pragma unroll
                for (int q = j + 1; q < 16; ++q) row[q] = fma(-lm, lane_read(lm, 16 * p + q), row[q]);
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) T[i][16 * p + j] = row[j];
        }
        __syncthreads();
        // (entries above the diagonal pick up values that nothing reads)
        if (h > p)
#pragma unroll 4
            for (int j = 0; j < 16; ++j) {
                const double lij = T[i][16 * p + j];
#pragma unroll
                for (int q = 0; q < 16; ++q) row[q] = fma(-lij, T[16 * h + q][16 * p + j], row[q]);
            }
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) a[(o + 4 * q + h) * ld + o + i] = T[4 * q + h][i];
    if (inv) {
        // column i of the inverse, rows [16h, 16h+16) in wave h: X[r] = (delta_ri -
        // sum_{m<r} L[r][m] X[m]) / L[r][r] with the sum taken in m order, quarter by
        // quarter: wave s finishes its rows, then the later waves add their terms
        // from them
        if (h == 0) rd[i] = 1.0 / T[i][i];
        __syncthreads();
        double sacc[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) sacc[q] = 16 * h + q == i ? 1.0 : 0.0;
        for (int st = 0; st < 4; ++st) {
            if (h == st) {
                double xq[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int r = 16 * st + q;
#pragma unroll
                    for (int m = 0; m < q; ++m) sacc[q] = fma(-T[r][16 * st + m], xq[m], sacc[q]);
                    xq[q] = r < i ? 0.0 : div_by(sacc[q], T[r][r], rd[r]);
                    X[r][i] = xq[q];
                }
            }
            __syncthreads();
            if (h > st) {
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int r = 16 * h + q;
#pragma unroll
                    for (int m = 0; m < 16; ++m) sacc[q] = fma(-T[r][16 * st + m], X[16 * st + m][i], sacc[q]);
                }
            }
        }
        double* dst = inv + (long)k * kDT * kDT;
#pragma unroll
        for (int q = 0; q < 16; ++q) dst[(4 * q + h) * kDT + i] = X[4 * q + h][i];
    }
}
__global__ __launch_bounds__(kDirectBlock) void k_potrf_tile(double* __restrict__ a, long ld, int k, int* __restrict__ bad,
                                                             const double* __restrict__ diag0, int* __restrict__ dropped, double tau,
                                                             double* __restrict__ inv) {
    __shared__ double T[kDT][kDT + 1];
    __shared__ double X[kDT][kDT + 1];
    __shared__ double rd[kDT];
    potrf_tile(a, ld, k, bad, diag0, dropped, tau, inv, T, X, rd);
}

// panel: tiles (i, k), i > k, become A_ik L_kk^-T (each row solved forward against L_kk);
// columns of dropped pivots are zero.  Four lanes per row hold every fourth column in
// registers; a finished entry crosses to its row's lanes by a quad permutation, and the
// sums run in column order as in one thread per row, whose 2,016 dependent products took
// 46 us per launch (11 now, at 3,198 unknowns).
template <int SUB>
__device__ __forceinline__ double quad_get(double v) {
    return dpp_move<SUB * 0x55>(v);
}
__global__ __launch_bounds__(kDirectBlock) void k_trsm_tiles(double* __restrict__ a, long ld, int k, const int* __restrict__ dropped) {
    __shared__ double L[kDT][kDT + 1];
    __shared__ double X[kDT][kDT + 1];
    __shared__ double rd[kDT];
    const int i = k + 1 + blockIdx.x, tid = threadIdx.x;
    const long ok = (long)k * kDT, oi = (long)i * kDT;
    {
        TileRegs tl, tx;
        tl.load(a + ok * ld + ok, ld);
        tx.load(a + oi * ld + ok, ld);
        tl.put(L);
        tx.put(X);
    }
    __syncthreads();
    if (tid < kDT) rd[tid] = 1.0 / L[tid][tid];
    __syncthreads();
    const int r = tid >> 2, sub = tid & 3;
    double xr[16];   // columns 4 q + sub
#pragma unroll
    for (int q = 0; q < 16; ++q) xr[q] = X[r][4 * q + sub];
#pragma unroll
    for (int c = 0; c < kDT; ++c) {
        const double mine = xr[c >> 2];
        const double sc = (c & 3) == 0 ? quad_get<0>(mine) : (c & 3) == 1 ? quad_get<1>(mine) : (c & 3) == 2 ? quad_get<2>(mine) : quad_get<3>(mine);
        double x = div_by(sc, L[c][c], rd[c]);
        if (dropped && dropped[ok + c]) x = 0.0;
        if (sub == (c & 3)) xr[c >> 2] = x;
#pragma unroll
        for (int q = c >> 2; q < 16; ++q)
            if (4 * q + sub > c) xr[q] = fma(-x, L[4 * q + sub][c], xr[q]);
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) X[r][4 * q + sub] = xr[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int rr = TileRegs::row(q), c = TileRegs::col();
        *reinterpret_cast<dt_v2*>(a + (oi + rr) * ld + ok + c) = dt_v2{X[rr][c], X[rr][c + 1]};
    }
}

// C (64 x 64 tile, row-major, leading dimension ldc) -= P Q^T  (BT) or P Q  (!BT), P and Q
// 64 x 64 tiles (ldp, ldq); overwrite: C = P Q instead.  On the FP64 matrix cores
// (v_mfma_f64_16x16x4_f64: lane l feeds A row l % 16 and B column l % 16 at k = l / 16 and
// holds D rows 4 t + l / 16, column l % 16): each of the four waves owns a 32 x 32 quarter
// of C.  Both operands are staged in LDS with k contiguous (rows of 66 doubles: 16 rows at
// two neighbouring k's fall on 32 different bank pairs).  The 4 x 4 register blocks on the
// vector units that this replaces read eight LDS words per sixteen products.  Measured (us
// per launch at 3,520 unknowns, with the tiles' loads issued together): trailing update
// 57 -> 35, update of the inverse 71 -> 36, panel 16 -> 6.6.  All reads of P, Q and C precede the
// barrier, so C may be the tile Q.
typedef double dt_v4 __attribute__((ext_vector_type(4)));
constexpr int kDTLd = kDT + 2;
template <bool BT>
__device__ __forceinline__ void tile_update(double* __restrict__ C, long ldc, const double* P, long ldp, const double* Q, long ldq,
                                            double (*Pl)[kDTLd], double (*Ql)[kDTLd], bool overwrite, const int* colMask = nullptr) {
    // colMask (BT only): output columns c with colMask[c] != 0 come out zero
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int r0 = 32 * (tid >> 7), c0 = 32 * ((tid >> 6) & 1);
    double cv[2][2][4];
    if (!overwrite)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 4; ++t) cv[i][j][t] = C[(r0 + 16 * i + 4 * t + g) * ldc + c0 + 16 * j + c];
    TileRegs tp, tq;
    tp.load(P, ldp);
    tq.load(Q, ldq);
    if (BT && colMask)
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (colMask[TileRegs::row(q)]) tq.v[q] = dt_v2{0, 0};
    tp.put(Pl);
    if (BT) tq.put(Ql);
    else tq.put_transposed(Ql);
    __syncthreads();
    dt_v4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = dt_v4{0, 0, 0, 0};
#pragma unroll 4
    for (int l = 0; l < kDT; l += 4) {
        double pv[2], qv[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            pv[i] = Pl[r0 + 16 * i + c][l + g];
            qv[i] = Ql[c0 + 16 * i + c][l + g];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(pv[i], qv[j], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                double* dst = C + (r0 + 16 * i + 4 * t + g) * ldc + c0 + 16 * j + c;
                *dst = overwrite ? acc[i][j][t] : cv[i][j][t] - acc[i][j][t];
            }
}

// One step k of the factorisation, after the diagonal tile, is two launches.
// Panel: tiles (i, k), i > k, by product with the inverted diagonal tile, A_ik <- A_ik
// inv(L_kk)^T, columns of dropped pivots zero.  When the inverse W = L^-1 is wanted (blocked
// forward substitution on the identity, right-looking), the next blocks take its row k at
// the same time: W_kj = inv(L_kk) W_kj, j <= k.
__global__ __launch_bounds__(kDirectBlock) void k_panel_tiles(double* __restrict__ a, long ld, int k, int m, const double* __restrict__ inv,
                                                             const int* __restrict__ dropped, double* __restrict__ W) {
    __shared__ double Pt[kDT][kDTLd];
    __shared__ double Qt[kDT][kDTLd];
    const long ok = (long)k * kDT;
    const double* Ikk = inv + (long)k * kDT * kDT;
    if ((int)blockIdx.x < m) {
        double* Aik = a + (long)(k + 1 + blockIdx.x) * kDT * ld + ok;
        tile_update<true>(Aik, ld, Aik, ld, Ikk, kDT, Pt, Qt, true, dropped ? dropped + ok : nullptr);
    } else {
        double* Wkj = W + ok * ld + (long)((int)blockIdx.x - m) * kDT;
        tile_update<false>(Wkj, ld, Ikk, kDT, Wkj, ld, Pt, Qt, true);
    }
}
// Trailing update of the lower tiles (i, j), k < j <= i: A_ij -= L_ik L_jk^T; block b
// enumerates the lower triangle of the trailing tile matrix row by row.  Block 0 has the next
// diagonal tile and factors it at once: the tile factor is one workgroup's serial chain, and
// as a launch of its own the chip waited for it in every step.  The blocks after the
// triangle update W: W_ij -= L_ik W_kj (i > k, j <= k).  Measured (us per step): at 3,520
// unknowns with the inverse, five launches one after the other 124 (tile factor 41, updates
// 35 and 36), two 80; at 3,198 without, tile factor and update 59 -> 33.
__global__ __launch_bounds__(kDirectBlock) void k_trailing_tiles(double* a, long ld, int k, int nt, int* __restrict__ bad,
                                                                const double* __restrict__ diag0, int* __restrict__ dropped, double tau,
                                                                double* __restrict__ inv, double* __restrict__ W) {
    __shared__ double Pt[kDT][kDTLd];
    __shared__ double Qt[kDT][kDTLd];
    __shared__ double rd[kDT];
    const int m = nt - k - 1, nSyrk = m * (m + 1) / 2;
    const long ok = (long)k * kDT;
    int b = blockIdx.x;
    if (b < nSyrk) {
        int ii = 0;
        while (b >= ii + 1) { b -= ii + 1; ++ii; }   // row ii of the trailing triangle holds ii + 1 tiles
        const long oi = (long)(k + 1 + ii) * kDT, oj = (long)(k + 1 + b) * kDT;
        tile_update<true>(a + oi * ld + oj, ld, a + oi * ld + ok, ld, a + oj * ld + ok, ld, Pt, Qt, false);
        if (blockIdx.x == 0) {
            __syncthreads();   // the tile is in memory for the whole workgroup, the operands' LDS is free
            potrf_tile(a, ld, k + 1, bad, diag0, dropped, tau, inv, reinterpret_cast<double (*)[kDT + 1]>(&Pt[0][0]),
                       reinterpret_cast<double (*)[kDT + 1]>(&Qt[0][0]), rd);
        }
    } else {
        b -= nSyrk;
        const int j = b % (k + 1), i = k + 1 + b / (k + 1);
        const long oi = (long)i * kDT, oj = (long)j * kDT;
        tile_update<false>(W + oi * ld + oj, ld, a + oi * ld + ok, ld, W + ok * ld + oj, ld, Pt, Qt, false);
    }
}

__global__ void k_dense_identity(double* __restrict__ a, long ld, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[(long)i * ld + i] = 1.0;
}

// Factors A = L L^T in place (lower); with W, its inverse L^-1 is built in the same steps,
// tileInv taking the diagonal tiles' inverses, which also turn the panel into a product.
// Without, the panel rows are solved by substitution (the direct solve's exact path).
void dense_cholesky(Ctx& c, double* A, int npad, int* bad, double* tileInv, const double* diag0, int* dropped, double tau, double* W) {
    const int nt = npad / kDT;
    const long ld = npad;
    if (W) {
        hipLaunchKernelGGL(k_dense_zero, dim3(2048), dim3(kBlock), 0, c.s, W, (long)npad * npad);
        hipLaunchKernelGGL(k_dense_identity, dim3(nblocks(npad)), dim3(kBlock), 0, c.s, W, ld, npad);
    }
    hipLaunchKernelGGL(k_potrf_tile, dim3(1), dim3(kDirectBlock), 0, c.s, A, ld, 0, bad, diag0, dropped, tau, tileInv);
    CIPC_LAUNCH_CHECK();
    for (int k = 0; k < nt; ++k) {
        const int m = nt - k - 1;
        if (W) hipLaunchKernelGGL(k_panel_tiles, dim3(m + k + 1), dim3(kDirectBlock), 0, c.s, A, ld, k, m, (const double*)tileInv,
                                  (const int*)dropped, W);
        else if (m > 0) hipLaunchKernelGGL(k_trsm_tiles, dim3(m), dim3(kDirectBlock), 0, c.s, A, ld, k, (const int*)dropped);
        if (m > 0) hipLaunchKernelGGL(k_trailing_tiles, dim3(m * (m + 1) / 2 + (W ? m * (k + 1) : 0)), dim3(kDirectBlock), 0, c.s, A, ld, k,
                                      nt, bad, diag0, dropped, tau, tileInv, W);
        CIPC_LAUNCH_CHECK();
    }
}

// Tile k of the substitutions, one launch: every workgroup solves the diagonal tile itself
// (forward u_k = L_kk^-1 y_k; backward x_k = L_kk^-T u_k), the first writes the result, and
// workgroup b subtracts its tile's product from the right-hand side of tile k + 1 + b
// (forward) or b (backward).  The result goes to another vector than the right-hand side,
// which the other workgroups still read.  The solve runs in one wave, lane = row: a finished
// entry crosses by readlane and every row subtracts its term at once (one thread for the
// whole triangle took 54 us); the tile for the product is loaded meanwhile.
template <bool transposed>
__global__ __launch_bounds__(kDirectBlock) void k_subst_tile(const double* __restrict__ a, long ld, int k, int nRest, double* __restrict__ y,
                                                             double* __restrict__ out) {
    __shared__ double L[kDT][kDT + 1];
    __shared__ double v[kDT];
    __shared__ double part[4][kDT];
    const int tid = threadIdx.x, b = blockIdx.x, ti = transposed ? b : k + 1 + b;
    const long ok = (long)k * kDT, oi = (long)ti * kDT;
    const bool work = b < nRest;
    TileRegs tl;
    tl.load(a + ok * ld + ok, ld);
    double s = tid < kDT ? y[ok + tid] : 0.0;
    // forward: rows 16 q + tid / 16, columns 4 (tid % 16) ..; backward: columns tid % 64,
    // rows 16 (tid / 64) + q
    double m[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const long src = transposed ? (ok + 16 * (tid >> 6) + q) * ld + oi + (tid & 63)
                                    : (oi + 16 * (q >> 2) + (tid >> 4)) * ld + ok + 4 * (tid & 15) + (q & 3);
        m[q] = work ? a[src] : 0.0;
    }
    if (transposed) tl.put_transposed(L);
    else tl.put(L);
    __syncthreads();
    if (tid < kDT) {
        const double d = L[tid][tid], rd = 1.0 / d;
#pragma unroll
        for (int n = 0; n < kDT; ++n) {
            const int c = transposed ? kDT - 1 - n : n;
            const double x = lane_read(div_by(s, d, rd), c);
            s = tid == c ? x : (transposed ? tid < c : tid > c) ? fma(-L[tid][c], x, s) : s;
        }
        v[tid] = s;
        if (b == 0) out[ok + tid] = s;
    }
    __syncthreads();
    if (!work) return;
    if (!transposed) {
        const int c4 = 4 * (tid & 15);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double ps = lane_sum<16>(((m[4 * q] * v[c4] + m[4 * q + 1] * v[c4 + 1]) + m[4 * q + 2] * v[c4 + 2]) + m[4 * q + 3] * v[c4 + 3]);
            if ((tid & 15) == 0) y[oi + 16 * q + (tid >> 4)] -= ps;
        }
    } else {
        double ps = 0;
#pragma unroll
        for (int q = 0; q < 16; ++q) ps = fma(m[q], v[16 * (tid >> 6) + q], ps);
        part[tid >> 6][tid & 63] = ps;
        __syncthreads();
        if (tid < kDT) y[oi + tid] -= ((part[0][tid] + part[1][tid]) + part[2][tid]) + part[3][tid];
    }
}

int direct_solve(Ctx& c, const double* b, double* x) {
    const int n = 3 * c.nV;
    if (n > kDirectMaxDof) return 3;
    const int nt = (n + kDT - 1) / kDT, npad = nt * kDT;
    const long ld = npad;
    double* A = c.denseA.ensure_exact((size_t)npad * npad);
    hipLaunchKernelGGL(k_dense_zero, dim3(2048), dim3(kBlock), 0, c.s, A, (long)npad * npad);
    hipLaunchKernelGGL(k_dense_pad_identity, dim3(1), dim3(kDT), 0, c.s, A, ld, n, npad);
    CIPC_LAUNCH_CHECK();
    BSR* parts[2] = {&c.Ael, &c.Acon};
    for (int q = 0; q < 2; ++q) {
        BSR& M = *parts[q];
        if (M.nnzb == 0) continue;
        hipLaunchKernelGGL(k_dense_scatter, dim3(nblocks(M.nnzb)), dim3(kBlock), 0, c.s, M.rowOf.p, M.col.p, M.val.p, M.nnzb, A, ld, q);
        CIPC_LAUNCH_CHECK();
    }
    int* bad = c.denseBad.ensure(1);
    CIPC_HIP(hipMemsetAsync(bad, 0, sizeof(int), c.s));
    dense_cholesky(c, A, npad, bad, nullptr);
    double* y = c.denseY.ensure(3 * (size_t)npad);
    double *u = y + npad, *xs = u + npad;   // forward and backward results
    CIPC_HIP(hipMemsetAsync(y, 0, npad * sizeof(double), c.s));
    CIPC_HIP(hipMemcpyAsync(y, b, n * sizeof(double), hipMemcpyDeviceToDevice, c.s));
    for (int k = 0; k < nt; ++k)
        hipLaunchKernelGGL(k_subst_tile<false>, dim3(std::max(1, nt - k - 1)), dim3(kDirectBlock), 0, c.s, (const double*)A, ld, k, nt - k - 1, y, u);
    for (int k = nt - 1; k >= 0; --k)
        hipLaunchKernelGGL(k_subst_tile<true>, dim3(std::max(1, k)), dim3(kDirectBlock), 0, c.s, (const double*)A, ld, k, k, u, xs);
    CIPC_LAUNCH_CHECK();
    CIPC_HIP(hipMemcpyAsync(x, xs, n * sizeof(double), hipMemcpyDeviceToDevice, c.s));
    CIPC_HIP(hipMemcpyAsync(c.hCnt + 48, bad, sizeof(int), hipMemcpyDeviceToHost, c.s));
    CIPC_HIP(hipStreamSynchronize(c.s));
    c.directSolves++;
    return c.hCnt[48] ? 1 : 0;
}

}  // namespace cipc
