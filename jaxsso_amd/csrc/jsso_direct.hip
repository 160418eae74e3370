// Sparse direct solve of the batched systems: multifrontal Cholesky of the
// constrained, block-Jacobi-scaled stiffness on a nested-dissection tree, with
// refinement on the FP64 residual (the counterpart of the reference's SuperLU
// solve, JaxSSO/solver.py:176-218).
//
// A front is the dense symmetric matrix of a tree node's pivots (k rows) and its
// border (b rows), k = 6 np, b = 6 nb, held as its lower triangle, row-major:
//   F11 = L L^T,   L21 = F21 L^-T,   C = F22 - L21 L21^T   (passed to the parent)
// and kept for the solves are   S = F11^-1 = L^-T L^-1   and   G = L21 L^-1, so
// that both directions are plain matrix-vector products without a dependence
// inside a panel:
//   forward   r2 -= G r1         (children before parents)
//   backward  x1 = S r1 - G^T x2 (parents before children)
// Every product runs on the FP64 matrix cores (v_mfma_f64_16x16x4): operands from
// LDS as [row][k] with a row stride of 2 (mod 4) doubles, so the 16 rows x 2
// columns a half wavefront reads fall on 32 different bank pairs.
//
// Small fronts (panel rows in LDS) are one workgroup each: gather, factor, panel,
// contribution, all from LDS; only the children's contributions are read and only
// S, G and the own contribution written.  Larger fronts go in panels of <= 96
// pivots whose columns are kept in HBM:
//   k_front_diag   inverse factor of a panel's diagonal block
//   k_front_strip  the rows below a panel's diagonal block: L21 (in place) and G; S
//   k_front_cols   the panel's update of the pivot columns still to come, with the
//                  inverse factor of the next panel's diagonal block
//   k_front_cb     after the last panel: C = gathered children - L21 L21^T over
//                  all pivots at once, so C is written once and never re-read
// The front is never assembled as a whole: each kernel gathers what it is the
// first to touch from the children's contributions and the blocks of K.  All
// fronts of a tree level, over all structures of the plan, go in the same
// launches.
#include <cmath>
#include <cstring>
#include <map>
#include <new>
#include <type_traits>

#include "direct_symbolic.hpp"
#include "solver_common.hpp"
#include "solver_kernels.hpp"

namespace jsso {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int DW = 96;                    // pivots per panel, at most (16 nodes)
constexpr int DROWS = 64;                 // edge of an update tile
constexpr int SROWS = 96;                 // rows of a strip
constexpr int DLEAF = 10;                 // nodes eliminated whole at the tree's leaves (5 to 12: within 3%)
constexpr int DLDS_MAX = 156 * 1024;      // dynamic LDS of a small front
constexpr int DIRECT_MAX_M = 2300;        // largest front (direct_build)
static_assert((DIRECT_MAX_M + 2 * 1024) * 4 * 8 <= DLDS_MAX, "LDS of the backward solve with 4 load cases");
constexpr int DIRECT_STEPS = 6;           // refinement steps, at most
constexpr int DEFECT_STEPS = 40;          // of a K that is not symmetric
constexpr double DIRECT_FLOOR_FACTOR = 16.0;   // attainable accuracy: 16 eps (||A|| ||x|| + ||b||), as the AMG solve
constexpr int HEAD_FRONTS = 64;           // below: k_front_cols factors the next panel's block itself (64
                                          // designs of 100 x 100: 34.3 ms with it, 33.7 without)
constexpr int BWD_PARTS = 8;              // workgroups per panel of the backward solve, at most
constexpr int STRIP_TILES = 3;            // 16x16 tiles of a strip that a wavefront holds
constexpr int DKC = 32;                   // pivot columns staged at a time by the tile kernels

// host: a front of a connectivity pattern; offsets within one structure's storage
struct FrontMeta {
    int32_t np, nb, node0, level;
    int32_t child[2], blk0, nblk;
    int32_t wn, npan;                     // nodes of a panel (the last may have fewer), panels
    bool small;                           // one-workgroup front
    int64_t fac, mat, pan, vec;           // (doubles) S|G panels, contribution (b x b), pivot columns
                                          // (m x k, large fronts), vector (x load cases)
};
// A front of a structure as the kernels take it: everything a workgroup needs in
// one read (following front -> children -> structure by dependent loads cost each of
// the ~100 kernels of a solve 2 us).
struct FrontTask {
    int32_t np, nb, wn, npan;
    int32_t node0, blk0, nblk, kref0;     // first entry in nodes / inv / blkrow, stored blocks, their base in kref
    int32_t sys, gnode0, cb[2];           // structure, its first node, border nodes of the children (0: none)
    int64_t mat, pan, fac, vec;           // offsets (doubles; vec: x load cases)
    int64_t cmat[2], cvec[2];             // the children's contributions and border vectors
};
struct DirectDev {
    const int32_t *nodes, *blk, *blkrow, *kref;
    const int2* inv;                      // per entry of `nodes`: the border node it is in each child, or -1
    const double* A64;
    double *fac, *mat, *vec;
    const double* zero;                   // a zero
    int32_t* bad;                         // per structure: a pivot was not positive
};
struct DirectReport {
    int32_t running, stalled, floor, bad;   // systems; structures with a pivot that is not positive
    double worst;                           // largest relative residual of the best iterates
    int32_t flags;                          // the assembly's (d_status)
    int32_t final;                          // every system done, on a K that this solve is for
    int32_t not_finite;                     // systems whose load is not finite (done: so is u)
};

struct DirectState {
    std::vector<std::vector<FrontTask>> small_tasks, big_tasks;   // per level
    struct Bucket {               // small fronts of a level that need alike much LDS
        size_t lds = 0, off = 0, n = 0;
        int threads = 0;
    };
    std::vector<std::vector<Bucket>> buckets;                        // per level
    std::vector<int> small_m, big_m, big_k, big_b, big_w, big_pan;   // per level: largest fronts, most panels
    std::vector<size_t> small_n, big_n, small_off, big_off;          // tasks of the level, first on the device
    int n_levels = 0, max_m = 0;
    size_t fac_n = 0, mat_n = 0, vec_n = 0;
    double flops = 0.0;
    DirectDev dev{};
    const FrontTask* d_tasks = nullptr;
    double* d_rho = nullptr;
    DirectReport *d_report = nullptr, *h_report = nullptr, *host_report = nullptr;   // host_report: h_report for the device
    size_t vec_bytes = 0;
    std::vector<void*> allocs;
    bool usable = false, factored = false;
    int64_t factorisations = 0, begun = 0, finished = 0;
};

// ---------------------------------------------------------------------------
// device: tiles
// ---------------------------------------------------------------------------
// D = A B + D with A 16x4 (lane: row l % 16, column l / 16), B 4x16 (lane: row
// l / 16, column l % 16), D 16x16 (element i of a lane: row 4 i + l / 16, column
// l % 16): a D tile is, element by element, the B operand of four further steps.
__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ double lane_value(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return join_halves(lo, hi);
}

// 1 / sqrt(d): the hardware estimate and one third-order correction
__device__ __forceinline__ double fast_rsqrt(double d) {
    const double y = __builtin_amdgcn_rsq(d);
    const double e = fma(-d * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// Cholesky factor L of a symmetric 16x16 block A and its inverse, by one wavefront;
// the inverse goes to D (LDS, zeros above the diagonal).
// Lane (r, q) = (l % 16, l / 16) holds A[r][4 i + q], i = 0..3: for a symmetric A
// that is at once the layout of the matrix core's result, of its first operand and,
// read as A[4 i + q][r], of its second.  Per four columns, with T the inverse factor
// of their 4x4 diagonal block (fetched by readlane, factored by all lanes alike),
//   l = A[:, 4 columns] T^T,  A -= l l^T,   x = T W[4 rows, :],  W -= l x   (W <- I)
// are four matrix instructions, x the four rows of the inverse.  Bound by its chain
// of dependent steps (four reciprocal roots per four columns): 4 700 cycles with the
// products by lane-wise arithmetic and readlane, 3 300 so.
__device__ __forceinline__ bool factor16(d4 A, double* D, int ld, int lane) {
    const int r = lane & 15, q = lane >> 4;
    d4 W;
#pragma unroll
    for (int i = 0; i < 4; ++i) W[i] = 4 * i + q == r ? 1.0 : 0.0;
    bool ok = true;
    auto is = [&](int i, int c) { return r == i && q == c ? 1.0 : 0.0; };
    const double m0 = is(0, 0), m10 = is(1, 0), m1 = is(1, 1), m20 = is(2, 0), m21 = is(2, 1), m2 = is(2, 2),
                 m30 = is(3, 0), m31 = is(3, 1), m32 = is(3, 2), m3 = is(3, 3);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const double a = A[b], w = W[b];
        double d[4][4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = c; i < 4; ++i) d[i][c] = lane_value(a, 16 * c + 4 * b + i);
        const double i0 = fast_rsqrt(d[0][0]);
        const double l10 = d[1][0] * i0, l20 = d[2][0] * i0, l30 = d[3][0] * i0;
        const double e1 = fma(-l10, l10, d[1][1]), i1 = fast_rsqrt(e1);
        const double l21 = fma(-l20, l10, d[2][1]) * i1, l31 = fma(-l30, l10, d[3][1]) * i1;
        const double e2 = fma(-l21, l21, fma(-l20, l20, d[2][2])), i2 = fast_rsqrt(e2);
        const double l32 = fma(-l31, l21, fma(-l30, l20, d[3][2])) * i2;
        const double e3 = fma(-l32, l32, fma(-l31, l31, fma(-l30, l30, d[3][3]))), i3 = fast_rsqrt(e3);
        ok &= d[0][0] > 0.0 && e1 > 0.0 && e2 > 0.0 && e3 > 0.0;
        const double t10 = -l10 * i0 * i1, t21 = -l21 * i1 * i2, t32 = -l32 * i2 * i3;
        const double t20 = -fma(l21, t10, l20 * i0) * i2, t31 = -fma(l32, t21, l31 * i1) * i3;
        const double t30 = -fma(l32, t20, fma(l31, t10, l30 * i0)) * i3;
        // T[r][q] for r < 4, zero elsewhere (by masks: selects became branches)
        double T = m0 * i0;
        T = fma(m10, t10, fma(m1, i1, T));
        T = fma(m21, t21, fma(m20, t20, fma(m2, i2, T)));
        T = fma(m3, i3, fma(m32, t32, fma(m31, t31, fma(m30, t30, T))));
        const d4 zero = {0.0, 0.0, 0.0, 0.0};
        const d4 lt = mfma64(T, a, zero), xt = mfma64(T, w, zero);   // element 0: rows q of the 4 x 16 results
        const double l = 4 * b + q > r ? 0.0 : lt[0], x = xt[0];
        D[(4 * b + q) * ld + r] = x;
        if (b < 3) {
            A = mfma64(-l, l, A);
            W = mfma64(-l, x, W);
        }
    }
    return ok;
}

// F11 (kp x kp in LDS, kp a multiple of 16; lower triangle, zeros above it) -> its
// inverse factor (whole workgroup).  Block (I, J) of L^-1, I > J, is left at block
// row J, block column I (as it is, not transposed), the diagonal blocks in place;
// the lower blocks hold L.  Per block column kb two phases with a barrier each:
//   B  wavefront 0 factors the diagonal block; the others take what column kb - 1
//      updates: the rest of the trailing triangle and the sums
//      W_IJ = sum_K L_IK Linv_KJ of the rows below
//   A  wavefront 0: L = A Dinv^T of the next block row and with it the next diagonal
//      block, from its registers; the others: the L below, and row kb of the inverse,
//      -Dinv W_J
// The factorisation of a 16x16 block (one wavefront, ~1.5 us of dependent steps) is
// the chain that bounds this routine (96 columns: 14 us); phase B hides the products
// behind it.  With the next diagonal block updated in a phase of its own, a 200 x 200
// shell took 4.99 ms, so 4.92.
__device__ __forceinline__ bool invert_factor(double* P, int ld, int kp, int wave, int nw, int lane) {
    const int nt = kp >> 4, r = lane & 15, q = lane >> 4;
    bool ok = true;
#pragma unroll 1
    for (int kb = 0; kb < nt; ++kb) {
        // B of block column j = kb - 1: products X Y (Y as it is or transposed) added to C
        const int j = kb - 1, n = nt - kb, ntri = kb ? n * (n + 1) / 2 : 0, all = ntri + n * kb;
#pragma unroll 1
        for (int e = wave ? wave : all; e < all; e += nw - 1) {   // (tile 0 is wavefront 0's)
            const double *X, *Y;
            double* C;
            int ys;
            double sign;
            if (e < ntri) {   // A_IJ -= L_I L_J^T
                int I = 0, J = e;
                while (J > I) {
                    J -= I + 1;
                    ++I;
                }
                I += kb;
                J += kb;
                X = P + (16 * I + r) * ld + 16 * j + q;
                Y = P + (16 * J + r) * ld + 16 * j + q;
                C = P + (16 * I + q) * ld + 16 * J + r;
                ys = 4;
                sign = -1.0;
            } else {   // W_IJ += L_Ij Linv_jJ, kept at block (J, I)
                const int I = kb + (e - ntri) % n, J = (e - ntri) / n;
                X = P + (16 * I + r) * ld + 16 * j + q;
                Y = P + (16 * J + q) * ld + 16 * j + r;
                C = P + (16 * J + q) * ld + 16 * I + r;
                ys = 4 * ld;
                sign = 1.0;
            }
            d4 acc;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = C[4 * i * ld];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc = mfma64(sign * X[4 * t], Y[t * ys], acc);
#pragma unroll
            for (int i = 0; i < 4; ++i) C[4 * i * ld] = acc[i];
        }
        double* D = P + (16 * kb) * ld + 16 * kb;
        auto lower = [&](const double* T) {
            d4 A;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = 4 * i + q;
                A[i] = r >= c ? T[r * ld + c] : T[c * ld + r];
            }
            return A;
        };
        if (wave == 0) ok &= factor16(lower(D), D, ld, lane);
        __syncthreads();
        if (wave == 0) {
            if (kb + 1 < nt) {
                // M = L^T = Dinv A^T: element i of a lane is L[r][4 i + q], both operands of L L^T
                double* N = P + (16 * (kb + 1) + r) * ld + 16 * kb + q;
                double* T = D + 16 * ld + 16;   // the next diagonal block
                d4 A = lower(T);
                d4 M = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int t = 0; t < 4; ++t) M = mfma64(D[r * ld + 4 * t + q], N[4 * t], M);
#pragma unroll
                for (int i = 0; i < 4; ++i) N[4 * i] = M[i];
#pragma unroll
                for (int t = 0; t < 4; ++t) A = mfma64(-M[t], M[t], A);
#pragma unroll
                for (int i = 0; i < 4; ++i) T[r * ld + 4 * i + q] = A[i];   // (held on to, it costs the others registers)
            }
        } else {
#pragma unroll 1
            for (int e0 = wave - 1; e0 < nt - 1 - (kb + 1 < nt); e0 += nw - 1) {
                const int e = e0 + (kb + 1 < nt && e0 >= kb);   // (the next block row is wavefront 0's)
                const bool inv = e < kb;   // row kb of the inverse: -Dinv W; else L_I = A_I Dinv^T
                double* C = P + (inv ? (16 * e + q) * ld + 16 * kb : (16 * (e + 1) + q) * ld + 16 * kb) + r;
                const double* X = inv ? D + r * ld + q : P + (16 * (e + 1) + r) * ld + 16 * kb + q;
                const double* Y = inv ? C : D + r * ld + q;
                const int ys = inv ? 4 * ld : 4;
                const double sign = inv ? -1.0 : 1.0;
                d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int t = 0; t < 4; ++t) acc = mfma64(sign * X[4 * t], Y[t * ys], acc);
#pragma unroll
                for (int i = 0; i < 4; ++i) C[4 * i * ld] = acc[i];
            }
        }
        __syncthreads();
    }
    return ok;
}

// 16 rows X (in LDS, stride ld) times Linv^T, block column J: sum over K <= J
__device__ __forceinline__ d4 strip_L(const double* X, const double* P, int ld, int J, int lane) {
    const int r = lane & 15, q = lane >> 4;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int K = 0; K <= J; ++K) {
        const double* x = X + r * ld + 16 * K + q;
        const double* y = P + (16 * K + r) * ld + 16 * J + q;
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = mfma64(x[4 * t], y[4 * t], acc);
    }
    return acc;
}
// 16 rows of L21 times Linv, block column J: sum over K >= J
__device__ __forceinline__ d4 strip_G(const double* X, const double* P, int ld, int nt, int J, int lane) {
    const int r = lane & 15, q = lane >> 4;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int K = J; K < nt; ++K) {
        const double* x = X + r * ld + 16 * K + q;
        const double* y = P + (16 * J + q) * ld + 16 * K + r;
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = mfma64(x[4 * t], y[4 * t * ld], acc);
    }
    return acc;
}
__device__ __forceinline__ void store_tile(double* G, int64_t ldg, d4 v, int nrow, int ncol, int lane) {
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (4 * i + q < nrow && r < ncol) G[(4 * i + q) * ldg + r] = v[i];
}

// S = Linv^T Linv (k x k, row-major) to global memory
__device__ __forceinline__ void write_S(const double* P, int ld, int kp, int k, double* S, int wave, int nw,
                                        int lane) {
    const int nt = kp >> 4, r = lane & 15, q = lane >> 4;
#pragma unroll 1
    for (int e = wave; e < nt * (nt + 1) / 2; e += nw) {
        int I = 0, J = e;
        while (J > I) {
            J -= I + 1;
            ++I;
        }
        d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
        for (int K = I; K < nt; ++K)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc = mfma64(P[(16 * I + 4 * t + q) * ld + 16 * K + r], P[(16 * J + 4 * t + q) * ld + 16 * K + r], acc);
        store_tile(S + (int64_t)16 * I * k + 16 * J, k, acc, k - 16 * I, k - 16 * J, lane);
        if (I != J) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (16 * I + 4 * i + q < k && 16 * J + r < k)
                    S[(int64_t)(16 * J + r) * k + 16 * I + 4 * i + q] = acc[i];
        }
    }
}

// entry (row, column) of the block that enters a front as F[6 a + row][6 c + col]
__device__ __forceinline__ double stored_entry(const DirectDev& d, int32_t kr, int row, int col) {
    // the triple names the block (column node, row node): kr even, stored as it is
    const int e = (kr & 1) ? row * 6 + col : col * 6 + row;
    const int vp = kr >> 1;
    return d.A64[(int64_t)(vp >> 6) * 36 * ROWS_PER_WG + ((int64_t)(e >> 1) * ROWS_PER_WG + (vp & 63)) * 2 + (e & 1)];
}

// The children's part of a front's entries: where each child keeps its contribution
// C (b x b, row-major, lower triangle)
struct Gather {
    const double *C[2], *zero;
    int ld[2];
    bool any;
};
__device__ __forceinline__ Gather make_gather(const DirectDev& d, const FrontTask& f) {
    Gather g;
    g.zero = d.zero;
    g.any = f.cb[0] > 0 || f.cb[1] > 0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        g.C[c] = d.mat + f.cmat[c];
        g.ld[c] = 6 * f.cb[c];
    }
    return g;
}
// (task, part) of a workgroup of a launch over `parts` parts of n tasks.  Many tasks:
// all parts of a task one after the other on one XCD, whose L2 then holds what they
// share; few: spread over the chip.
struct Where {
    int task, part;
};
__device__ __forceinline__ Where locate(int n, int parts, int b) {
    if (n >= 64) {
        const int q = b >> 3, t = q / parts;
        return {8 * t + (b & 7), q - t * parts};
    }
    return {b % n, b / n};
}
__device__ __forceinline__ Where locate(int n, int parts) { return locate(n, parts, (int)blockIdx.x); }
__host__ __device__ inline int task_slots(int n) { return n >= 64 ? 8 * ((n + 7) / 8) : n; }
static dim3 part_grid(size_t n, int parts) {
    return dim3((unsigned)(task_slots((int)n) * parts));
}
// entry (row, col) of the front, row >= col; a, b: `inv` of their nodes.  Without
// branches, so that a thread's loads are all in flight at once (a wavefront that
// waited for each in turn spent most of its time here): what a child does not hold
// is read from a word that is zero.
__device__ __forceinline__ double gathered(const Gather& g, int2 a, int2 b, int rr, int cc, bool on) {
    const bool x = on && (a.x | b.x) >= 0, y = on && (a.y | b.y) >= 0;
    const double* p = x ? g.C[0] + (int64_t)(6 * a.x + rr) * g.ld[0] + 6 * b.x + cc : g.zero;
    const double* q = y ? g.C[1] + (int64_t)(6 * a.y + rr) * g.ld[1] + 6 * b.y + cc : g.zero;
    return *p + *q;
}
// adds the blocks of K with front rows in [r0, r1) and columns in [c0, c1) to a tile
// in LDS (rows and columns relative to r0, c0; front rows from `split` on are `gap`
// rows further down); four chains of dependent loads per thread in flight
__device__ __forceinline__ void add_stored(const DirectDev& d, const FrontTask& f, int r0,
                                           int r1, int c0, int c1, int split, int gap, double* T, int ld, int tid,
                                           int nth) {
    if (r1 <= r0) return;
    const int n0 = r0 / 6, n1 = (r1 + 5) / 6, m = f.np + f.nb;
    const int32_t* br = d.blkrow + f.node0;
    const int b0 = br[n0], b1 = n1 < m ? br[n1] : f.blk0 + f.nblk;
    const int all = (b1 - b0) * 36;
    for (int e0 = tid; e0 < all; e0 += 4 * nth) {
        double v[4];
        int at[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int e = min(e0 + u * nth, all - 1), blk = e / 36, row = e % 36 / 6, col = e % 6;
            const int32_t* t3 = d.blk + 3 * (b0 + blk);
            const int R = 6 * t3[1] + row, C = 6 * t3[2] + col;
            v[u] = stored_entry(d, d.kref[f.kref0 + t3[0]], row, col);
            at[u] = e0 + u * nth < all && R >= r0 && R < r1 && C >= c0 && C < c1
                        ? (R - r0 + (R >= split ? gap : 0)) * ld + C - c0 : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (at[u] >= 0) T[at[u]] += v[u];
    }
}

// ---------------------------------------------------------------------------
// device: factorisation
// ---------------------------------------------------------------------------
// One small front per workgroup.  Bound by its chain of phases (a leaf of 12 nodes
// on a full chip, us: blocks of K 5, factor 12, strips 9, contribution 7), so every
// phase keeps many loads in flight and spreads over all wavefronts; the children's
// entries of a wavefront's first contribution tile are requested before the
// factorisation and arrive behind it.  Only the panel rows are held in LDS.
template <int NT>
__global__ __launch_bounds__(NT, NT == 1024 ? 4 : NT == 512 ? 4 : 3) void k_front_small(DirectDev d, const FrontTask* __restrict__ tasks) {
    extern __shared__ double P[];
    const FrontTask f = tasks[blockIdx.x];
    constexpr int nw = NT / 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int k = 6 * f.np, b = 6 * f.nb;
    const int kp = (k + 15) & ~15, bp = (b + 15) & ~15, ld = kp + 2;
    const int nt = kp >> 4, bt = bp >> 4, bs = (bt + 1) >> 1, r = lane & 15, q = lane >> 4;
    int2* inv = reinterpret_cast<int2*>(P + (kp + bp) * ld);   // of every node, past the end: none
    const Gather ga = make_gather(d, f);
    auto gather_tile = [&](int I, int J, d4 (&t)[2][2]) {
        const int2* bi = inv + f.np;
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const int col = min(32 * J + 16 * v + r, b - 1), cn = col / 6, cc = col - 6 * cn;
            const int2 ic = bi[cn];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = min(32 * I + 16 * u + 4 * i + q, b - 1), rn = row / 6;
                    t[u][v][i] = gathered(ga, bi[rn], ic, row - 6 * rn, cc, col <= row);
                }
        }
    };
    // contribution: 32x32 tiles of the lower triangle
    int I = 0, J = wave;
    while (J > I) {
        J -= I + 1;
        ++I;
    }
    d4 acc[2][2] = {};
    // panel: what the children pass up, by 4 rows x 16 columns per wavefront, four at a
    // time; the identity on the diagonal
    if (ga.any) {
        for (int e = tid; e < f.np + f.nb + 3; e += NT) inv[e] = e < f.np + f.nb ? d.inv[f.node0 + e] : int2{-1, -1};
        __syncthreads();
        if (I < bs) gather_tile(I, J, acc);
        const int items = ((kp + bp) >> 2) * nt;
        for (int e0 = wave; e0 < items; e0 += 4 * nw) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = min(e0 + u * nw, items - 1), g = e / nt, K = e - g * nt;
                const int row = 4 * g + q, col = 16 * K + r, R = row < kp ? row : row - kp + k;
                const bool on = col < k && (row < kp ? row < k && col <= row : row < kp + b);
                const int rn = on ? R / 6 : 0, cn = on ? col / 6 : 0;
                v[u] = gathered(ga, inv[rn], inv[cn], R - 6 * rn, col - 6 * cn, on) + (row == col ? 1.0 : 0.0);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {   // (the last item again where there are fewer)
                const int e = min(e0 + u * nw, items - 1), g = e / nt, K = e - g * nt;
                P[(4 * g + q) * ld + 16 * K + r] = v[u];
            }
        }
    } else {
        for (int e = 2 * tid; e < (kp + bp) * ld; e += 2 * NT)
            *reinterpret_cast<double2*>(P + e) = double2{0.0, 0.0};
        __syncthreads();
        for (int e = tid; e < kp; e += NT) P[e * ld + e] = 1.0;
    }
    __syncthreads();
    add_stored(d, f, 0, k + b, 0, k, k, kp - k, P, ld, tid, NT);
    __syncthreads();
    const bool ok = invert_factor(P, ld, kp, wave, nw, lane);
    if (!ok && tid == 0) atomicOr(d.bad + f.sys, 1);
    double* S = d.fac + f.fac;
    double* G = S + (int64_t)k * k;
    // strips, tile by tile: L21 (kept in registers until every wavefront has read F21),
    // then G = L21 L^-1; as many rounds as 16 x 16 tiles per wavefront need
    for (int e0 = 0; e0 < bt * nt; e0 += STRIP_TILES * nw) {
        // (rows of one round are whole: a round takes all columns of its row tiles)
        const int rows = min(bt - e0 / nt, STRIP_TILES * nw / nt), n = rows * nt, row0 = e0 / nt;
        d4 v[STRIP_TILES];
#pragma unroll
        for (int u = 0; u < STRIP_TILES; ++u) {
            const int e = wave + nw * u;
            if (e < n) v[u] = strip_L(P + (kp + 16 * (row0 + e % rows)) * ld, P, ld, nt - 1 - e / rows, lane);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < STRIP_TILES; ++u) {
            const int e = wave + nw * u, B = row0 + e % rows, K = nt - 1 - e / rows;
            if (e < n) {
#pragma unroll
                for (int i = 0; i < 4; ++i) P[(kp + 16 * B + 4 * i + q) * ld + 16 * K + r] = v[u][i];
            }
        }
        __syncthreads();
        for (int e = wave; e < n; e += nw) {
            const int B = row0 + e % rows, K = e / rows;
            store_tile(G + (int64_t)16 * B * k + 16 * K, k, strip_G(P + (kp + 16 * B) * ld, P, ld, nt, K, lane),
                       b - 16 * B, k - 16 * K, lane);
        }
        e0 += n - STRIP_TILES * nw;
    }
    write_S(P, ld, kp, k, S, nw - 1 - wave, nw, lane);
    double* Cout = d.mat + f.mat;
    const int k4 = (k + 3) >> 2;
    while (I < bs) {
        // (rows past the last tile read the tile before: their products are not stored)
        const int i1 = 2 * I + 1 < bt ? 16 : 0, j1 = 2 * J + 1 < bt ? 16 : 0;
        const double* x = P + (kp + 32 * I + r) * ld + q;
        const double* y = P + (kp + 32 * J + r) * ld + q;
#pragma unroll 4
        for (int t = 0; t < k4; ++t) {
            const double a0 = -x[4 * t], a1 = -x[i1 * ld + 4 * t], b0 = y[4 * t], b1 = y[j1 * ld + 4 * t];
            acc[0][0] = mfma64(a0, b0, acc[0][0]);
            acc[0][1] = mfma64(a0, b1, acc[0][1]);
            acc[1][0] = mfma64(a1, b0, acc[1][0]);
            acc[1][1] = mfma64(a1, b1, acc[1][1]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = 32 * I + 16 * u + 4 * i + q, col = 32 * J + 16 * v + r;
                    if (row < b && col <= row) Cout[(int64_t)row * b + col] = acc[u][v][i];
                }
        J += nw;
        while (J > I) {
            J -= I + 1;
            ++I;
        }
        if (I < bs) {
            if (ga.any)
                gather_tile(I, J, acc);
            else
                acc[0][0] = acc[0][1] = acc[1][0] = acc[1][1] = d4{0.0, 0.0, 0.0, 0.0};
        }
    }
}

// offset of panel p's S (w x w, then its G) in a front's factor
__device__ __forceinline__ int64_t panel_offset(int m, int w, int p) {
    return (int64_t)p * w * w + (int64_t)p * m * w - (int64_t)w * w * p * (p + 1) / 2;
}

// The inverse factor of a diagonal block: from the block in P (whole workgroup) to the
// block's place in the pivot columns.
__device__ __forceinline__ void factor_block(const DirectDev& d, const FrontTask& f, double* P, int ld, int kp, int w,
                                             double* F, int k, int wave, int lane) {
    const bool ok = invert_factor(P, ld, kp, wave, 8, lane);
    if (!ok && wave == 0 && lane == 0) atomicOr(d.bad + f.sys, 1);
    for (int row = wave; row < w; row += 8)
        for (int col = lane; col <= row; col += 64)
            F[(int64_t)row * k + col] = P[(16 * (col >> 4) + (row & 15)) * ld + 16 * (row >> 4) + (col & 15)];
}

// diagonal block of panel p (gathered for the first panel), factored
__global__ __launch_bounds__(512) void k_front_diag(DirectDev d, const FrontTask* __restrict__ tasks, int p) {
    extern __shared__ double P[];
    const FrontTask f = tasks[blockIdx.x];
    if (p >= f.npan) return;
    const int k = 6 * f.np, c0 = 6 * p * f.wn, w = min(6 * f.wn, k - c0);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kp = (w + 15) & ~15, ld = kp + 2;
    double* F = d.mat + f.pan + (int64_t)c0 * k + c0;
    const Gather ga = make_gather(d, f);
    __shared__ int2 inv[DW / 6 + 1];
    if (tid < w / 6) inv[tid] = d.inv[f.node0 + tid];
    __syncthreads();
    for (int c1 = 0; c1 < kp; c1 += 64) {
        const int col = c1 + lane, cn = min(col, w - 1) / 6, cc = col - 6 * cn;
        const int2 ic = inv[cn];
        for (int row0 = wave; row0 < kp; row0 += 32) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int row = row0 + 8 * u, rn = min(row, w - 1) / 6;
                const bool on = row < w && col <= row;
                if (p > 0)
                    v[u] = *(on ? F + (int64_t)row * k + col : d.zero) + (row == col && row >= w ? 1.0 : 0.0);
                else
                    v[u] = (row == col ? 1.0 : 0.0) + gathered(ga, inv[rn], ic, row - 6 * rn, cc, on);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (row0 + 8 * u < kp && col < kp) P[(row0 + 8 * u) * ld + col] = v[u];
        }
    }
    __syncthreads();
    if (p == 0) add_stored(d, f, 0, w, 0, w, w, 0, P, ld, tid, 512);
    __syncthreads();
    factor_block(d, f, P, ld, kp, w, F, k, wave, lane);
}

// `rows` (<= 96) rows below panel p's diagonal block: L21 = F21 L^-T (in place) and G = L21 L^-1;
// the last part: S = L^-T L^-1, which nothing waits for
__global__ __launch_bounds__(1024) void k_front_strip(DirectDev d, const FrontTask* __restrict__ tasks, int p, int n, int parts, int rows) {
    extern __shared__ double P[];
    const Where at = locate(n, parts);
    if (at.task >= n) return;
    const FrontTask f = tasks[at.task];
    if (p >= f.npan) return;
    const int k = 6 * f.np, m = k + 6 * f.nb, c0 = 6 * p * f.wn, w = min(6 * f.wn, k - c0);
    const int r0 = c0 + w + rows * at.part;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kp = (w + 15) & ~15, ld = kp + 2, nt = kp >> 4;
    double* F = d.mat + f.pan + c0;   // column c0 of the pivot columns
    if (at.part == parts - 1) {
        static_assert(DW <= 96, "six rows a wavefront");
        for (int col = lane; col < kp; col += 64) {
            double y[6];
#pragma unroll
            for (int u = 0; u < 6; ++u) {
                const int row = wave + 16 * u;
                y[u] = *(row < w && col <= row ? F + (int64_t)(c0 + row) * k + col : d.zero) +
                       (row == col && row >= w ? 1.0 : 0.0);
            }
#pragma unroll
            for (int u = 0; u < 6; ++u) {
                const int row = wave + 16 * u;
                if (row < kp && col >> 4 <= row >> 4)
                    P[(16 * (col >> 4) + (row & 15)) * ld + 16 * (row >> 4) + (col & 15)] = y[u];
            }
        }
        __syncthreads();
        write_S(P, ld, kp, w, d.fac + f.fac + panel_offset(m, 6 * f.wn, p), wave, 16, lane);
        return;
    }
    if (r0 >= m) return;
    double* X = P + kp * ld;
    const int nr = min(rows, m - r0), rt = rows >> 4;
    const Gather ga = make_gather(d, f);
    __shared__ int2 ir[SROWS / 6 + 2], icol[DW / 6 + 1];
    const int rn0 = r0 / 6;
    if (p == 0) {
        if (tid < SROWS / 6 + 2) ir[tid] = rn0 + tid < f.np + f.nb ? d.inv[f.node0 + rn0 + tid] : int2{-1, -1};
        if (tid >= 64 && tid < 64 + w / 6) icol[tid - 64] = d.inv[f.node0 + tid - 64];
        __syncthreads();
    }
    // lane: two columns; wavefront: rows wave, wave + 16, ..; U of them in flight
    const int col = 2 * lane, cn = min(col, w - 1) / 6, cc = col - 6 * cn;
    auto load = [&](auto count, int u0, auto entry) {
        constexpr int U = decltype(count)::value;
        double2 v[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int row = wave + 16 * (u0 + u);
            v[u] = entry(min(r0 + row, m - 1), row < nr && col < w);
            y[u] = *reinterpret_cast<const double2*>(row < w && col <= row ? F + (int64_t)(c0 + row) * k + col : d.zero);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int row = wave + 16 * (u0 + u);
            if (col < kp && row < rows) *reinterpret_cast<double2*>(X + row * ld + col) = v[u];
            // block (I, J) of the inverse factor goes to block row J, block column I; zeros
            // above its diagonal, ones on the padding's
            if (row < kp && col >> 4 <= row >> 4) {
                double2 z;
                z.x = col <= row && row < w ? y[u].x : row == col ? 1.0 : 0.0;
                z.y = col + 1 <= row && row < w ? y[u].y : row == col + 1 && row >= w ? 1.0 : 0.0;
                *reinterpret_cast<double2*>(P + (16 * (col >> 4) + (row & 15)) * ld + 16 * (row >> 4) + (col & 15)) = z;
            }
        }
    };
    static_assert(DW <= 96 && SROWS <= 96, "six rows a wavefront, 48 pairs of columns");
    if (p > 0) {
        load(std::integral_constant<int, 6>(), 0, [&](int R, bool on) {
            return *reinterpret_cast<const double2*>(on ? F + (int64_t)R * k + col : d.zero);
        });
    } else {
        const int2 ic = icol[cn];
        auto entry = [&](int R, bool on) {
            const int rn = R / 6;
            const int2 jr = ir[rn - rn0];
            return make_double2(gathered(ga, jr, ic, R - 6 * rn, cc, on), gathered(ga, jr, ic, R - 6 * rn, cc + 1, on));
        };
        load(std::integral_constant<int, 3>(), 0, entry);
        load(std::integral_constant<int, 3>(), 3, entry);
    }
    __syncthreads();
    if (p == 0) {
        add_stored(d, f, r0, r0 + nr, 0, w, m, 0, X, ld, tid, 1024);
        __syncthreads();
    }
    // rt row tiles x nt block columns over 16 wavefronts
    d4 v[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int e = wave + 16 * u;
        if (e < rt * nt) v[u] = strip_L(X + 16 * (e % rt) * ld, P, ld, e / rt, lane);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int e = wave + 16 * u, I = e % rt, J = e / rt;
        if (e < rt * nt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) X[(16 * I + 4 * i + q) * ld + 16 * J + r] = v[u][i];
            store_tile(F + (int64_t)(r0 + 16 * I) * k + 16 * J, k, v[u], nr - 16 * I, w - 16 * J, lane);
        }
    }
    __syncthreads();
    double* G = d.fac + f.fac + panel_offset(m, 6 * f.wn, p) + (int64_t)w * w + (int64_t)(r0 - c0 - w) * w;
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int e = wave + 16 * u, I = e % rt, J = e / rt;
        if (e < rt * nt)
            store_tile(G + (int64_t)16 * I * w + 16 * J, w, strip_G(X + 16 * I * ld, P, ld, nt, J, lane), nr - 16 * I,
                       w - 16 * J, lane);
    }
}

// acc += X_I Y_J^T of a 64x64 tile (wavefront: 32x32 of it) over the pivot columns
// [c0, c0 + w): rows i0.. and j0.. of the pivot columns F (m rows, row stride k)
struct TileAcc {
    d4 a[2][2];
};
__device__ __forceinline__ void tile_product(const double* __restrict__ F, int k, int m, int i0, int j0, int c0, int w,
                                             double* X, double* Y, int tid, TileAcc& t) {
    constexpr int LD = DKC + 2;
    const int lane = tid & 63, wave = tid >> 6;
    const int wi = 32 * (wave >> 1), wj = 32 * (wave & 1);
    // thread: pairs of columns; 16 pairs of a row, 16 rows at a time
    const int pc = 2 * (tid & 15), pr = tid >> 4;
    double2 xv[4], yv[4];
    auto fetch = [&](int k0) {
        const bool on = k0 + pc < w;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int ri = i0 + pr + 16 * u, rj = j0 + pr + 16 * u;
            xv[u] = on && ri < m ? *reinterpret_cast<const double2*>(F + (int64_t)ri * k + c0 + k0 + pc)
                                 : double2{0.0, 0.0};
            yv[u] = on && rj < m ? *reinterpret_cast<const double2*>(F + (int64_t)rj * k + c0 + k0 + pc)
                                 : double2{0.0, 0.0};
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < w; k0 += DKC) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            *reinterpret_cast<double2*>(X + (pr + 16 * u) * LD + pc) = xv[u];
            *reinterpret_cast<double2*>(Y + (pr + 16 * u) * LD + pc) = yv[u];
        }
        __syncthreads();
        if (k0 + DKC < w) fetch(k0 + DKC);   // the next chunk is on its way during this one's products
        const double* x = X + (wi + (lane & 15)) * LD + (lane >> 4);
        const double* y = Y + (wj + (lane & 15)) * LD + (lane >> 4);
        auto step = [&](int s) {
            const double a0 = x[4 * s], a1 = x[16 * LD + 4 * s], b0 = y[4 * s], b1 = y[16 * LD + 4 * s];
            t.a[0][0] = mfma64(a0, b0, t.a[0][0]);
            t.a[0][1] = mfma64(a0, b1, t.a[0][1]);
            t.a[1][0] = mfma64(a1, b0, t.a[1][0]);
            t.a[1][1] = mfma64(a1, b1, t.a[1][1]);
        };
        if (k0 + DKC <= w) {
#pragma unroll
            for (int s = 0; s < DKC / 4; ++s) step(s);
        } else {
#pragma unroll 2
            for (int s = 0; s < (w - k0 + 3) >> 2; ++s) step(s);
        }
    }
}

// The next panel's diagonal block: panel p's update of it (gathered here for p = 0) and
// its inverse factor, by one workgroup of 512 threads.
__device__ __forceinline__ void next_block(const DirectDev& d, const FrontTask& f, int p, double* P, int tid) {
    const int k = 6 * f.np, c0 = 6 * p * f.wn, w = 6 * f.wn, c1 = c0 + w, w1 = min(w, k - c1);
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, q = lane >> 4;
    const int ldx = ((w + 15) & ~15) + 2, kp = (w1 + 15) & ~15, ld = kp + 2, nt = kp >> 4;
    double* F = d.mat + f.pan + (int64_t)c1 * k;   // rows of the next panel
    __shared__ int2 inv[DW / 6 + 1];
    if (p == 0) {
        if (tid < w1 / 6) inv[tid] = d.inv[f.node0 + c1 / 6 + tid];
        __syncthreads();
    }
    // a wavefront's tiles of the lower triangle in the matrix core's layout, and the
    // panel's columns of these rows: all on their way together
    constexpr int MT = (DW / 16 * (DW / 16 + 1) / 2 + 7) / 8;
    const Gather ga = make_gather(d, f);
    d4 t[MT];
    int ti[MT], tj[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        int I = 0, J = wave + 8 * u;
        while (J > I) {
            J -= I + 1;
            ++I;
        }
        ti[u] = I;
        tj[u] = J;
    }
    if (p > 0) {
#pragma unroll
        for (int u = 0; u < MT; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 16 * ti[u] + 4 * i + q, col = 16 * tj[u] + r;
                t[u][i] = *(row < w1 && col <= row ? F + (int64_t)row * k + c1 + col : d.zero);
            }
    } else {
#pragma unroll
        for (int u = 0; u < MT; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 16 * ti[u] + 4 * i + q, col = 16 * tj[u] + r;
                const int rn = min(row, w1 - 1) / 6, cn = min(col, w1 - 1) / 6;
                t[u][i] = gathered(ga, inv[rn], inv[cn], row - 6 * rn, col - 6 * cn, row < w1 && col <= row);
            }
    }
    static_assert(DW <= 96, "12 rows a wavefront, 48 pairs of columns");
#pragma unroll
    for (int u0 = 0; u0 < 12; u0 += 6) {
        double2 x[6];
#pragma unroll
        for (int u = 0; u < 6; ++u) {
            const int row = wave + 8 * (u0 + u);
            x[u] = *reinterpret_cast<const double2*>(row < w1 && 2 * lane < w ? F + (int64_t)row * k + c0 + 2 * lane
                                                                              : d.zero);
        }
#pragma unroll
        for (int u = 0; u < 6; ++u)
            if (wave + 8 * (u0 + u) < kp && 2 * lane < ldx - 2)
                *reinterpret_cast<double2*>(P + (wave + 8 * (u0 + u)) * ldx + 2 * lane) = x[u];
    }
    __syncthreads();
    const double *X[MT], *Y[MT];   // (a tile past the last: any, unused)
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        X[u] = P + (16 * min(ti[u], nt - 1) + r) * ldx + q;
        Y[u] = P + (16 * min(tj[u], nt - 1) + r) * ldx + q;
    }
#pragma unroll 2
    for (int c = 0; c < (w + 3) >> 2; ++c)   // the tiles in turn: their chains overlap
#pragma unroll
        for (int u = 0; u < MT; ++u) t[u] = mfma64(-X[u][4 * c], Y[u][4 * c], t[u]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        if (ti[u] >= nt) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 16 * ti[u] + 4 * i + q, col = 16 * tj[u] + r;
            P[row * ld + col] = t[u][i] + (row == col && (p == 0 || row >= w1) ? 1.0 : 0.0);
            if (ti[u] != tj[u]) P[(16 * tj[u] + 4 * i + q) * ld + 16 * ti[u] + r] = 0.0;
        }
    }
    __syncthreads();
    if (p == 0) {
        add_stored(d, f, c1, c1 + w1, c1, c1 + w1, 6 * (f.np + f.nb) + k, 0, P, ld, tid, 512);
        __syncthreads();
    }
    factor_block(d, f, P, ld, kp, w1, F + c1, k, wave, lane);
}

// Panel p's update of the pivot columns after it.  The first workgroups take the next
// panel's diagonal block, one per front, and factor it: the chain of the panels, which
// the update of the rest (`parts` pairs of 64x64 tiles a front; gathered here for
// p = 0) runs beside.  Factored in a
// launch of its own after the update, a panel took 65 us, so 57 (200 x 200 shell, 58
// panels in sequence).  Launches of many fronts fill the chip without it, and do so
// better with a tile per workgroup (HEAD_FRONTS).
template <bool HEAD>
__global__ __launch_bounds__(HEAD ? 512 : 256, HEAD ? 4 : 1) void k_front_cols(DirectDev d, const FrontTask* __restrict__ tasks, int p, int n, int parts) {
    extern __shared__ double P[];
    const int heads = HEAD ? task_slots(n) : 0, b = blockIdx.x;
    const Where at = b < heads ? Where{b, 0} : locate(n, parts, b - heads);
    if (at.task >= n) return;
    const FrontTask f = tasks[at.task];
    if (p + 1 >= f.npan) return;
    if (b < heads) {
        next_block(d, f, p, P, threadIdx.x);
        return;
    }
    const int k = 6 * f.np, m = k + 6 * f.nb, c0 = 6 * p * f.wn, w = 6 * f.wn, t0 = c0 + w;
    const int w1 = HEAD ? min(w, k - t0) : 0;      // rows and columns that the head takes
    const int nc = (k - t0 + DROWS - 1) / DROWS;   // tile columns; tile -> (row, column), columns of a row together
    const int half = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    const int first = (HEAD ? 2 : 1) * at.part;
    if (t0 + DROWS * (first / nc) >= m) return;
    const int i0 = t0 + DROWS * ((first + half) / nc), j0 = t0 + DROWS * ((first + half) % nc);
    const bool on = i0 < m && j0 <= i0 && (i0 - t0 + DROWS > w1 || j0 - t0 + DROWS > w1);
    if (!HEAD && !on) return;
    double* sh = P + half * 2 * DROWS * (DKC + 2);
    double* F = d.mat + f.pan;
    TileAcc t = {};
    tile_product(F, k, on ? m : 0, i0, j0, c0, w, sh, sh + DROWS * (DKC + 2), tid, t);
    const int wi = 32 * (wave >> 1), wj = 32 * (wave & 1);
    const Gather ga = make_gather(d, f);
    const int2* inv = d.inv + f.node0;
    const int i1 = on ? min(m, i0 + DROWS) : i0, j1 = min(k, j0 + DROWS);
    constexpr int LDT = DROWS + 2;
    static_assert(LDT * DROWS <= 2 * DROWS * (DKC + 2), "tile fits the staging buffers");
    if (p == 0) {   // the blocks of K that enter this tile
        __syncthreads();
        for (int e = tid; e < LDT * DROWS; e += 256) sh[e] = 0.0;
        __syncthreads();
        add_stored(d, f, i0, i1, j0, j1, m + k, 0, sh, LDT, tid, 256);
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = i0 + wi + 16 * a + 4 * i + (lane >> 4), col = j0 + wj + 16 * b + (lane & 15);
                if (row >= i1 || col >= j1 || col > row || (row - t0 < w1 && col - t0 < w1)) continue;
                double v;
                if (p > 0)
                    v = F[(int64_t)row * k + col];
                else
                    v = (row == col ? 1.0 : 0.0) + gathered(ga, inv[row / 6], inv[col / 6], row % 6, col % 6, true) +
                        sh[(row - i0) * LDT + col - j0];
                F[(int64_t)row * k + col] = v - t.a[a][b][i];
            }
}

// contribution of a large front, 64x64 tiles of the lower triangle; bound by the FP64
// matrix cores' rate and by the latency of the gathers before them, which three waves a
// SIMD cover best (64 designs of 100 x 100: 32.4 ms an evaluation with the two that
// unbounded registers leave, 31.7 with three, 33.3 with four, which spill)
__global__ __launch_bounds__(256, 3) void k_front_cb(DirectDev d, const FrontTask* __restrict__ tasks, int n, int parts) {
    __shared__ double sh[2 * DROWS * (DKC + 2)];
    __shared__ int2 ir[DROWS / 6 + 3], ic[DROWS / 6 + 3];
    const Where at = locate(n, parts);
    if (at.task >= n) return;
    const FrontTask f = tasks[at.task];
    const int k = 6 * f.np, b = 6 * f.nb, m = k + b, nt = (b + DROWS - 1) / DROWS;
    const int e = at.part;
    if (e >= nt * (nt + 1) / 2) return;
    int I = (int)((sqrtf(8.0f * e + 1.0f) - 1.0f) * 0.5f);
    while (I * (I + 1) / 2 > e) --I;
    while ((I + 1) * (I + 2) / 2 <= e) ++I;
    const int J = e - I * (I + 1) / 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4;
    const int rn0 = DROWS * I / 6, cn0 = DROWS * J / 6;
    if (tid < DROWS / 6 + 3) {
        ir[tid] = rn0 + tid < f.nb ? d.inv[f.node0 + f.np + rn0 + tid] : int2{-1, -1};
        ic[tid] = cn0 + tid < f.nb ? d.inv[f.node0 + f.np + cn0 + tid] : int2{-1, -1};
    }
    __syncthreads();
    const int wi = DROWS * I + 32 * (wave >> 1), wj = DROWS * J + 32 * (wave & 1);
    const Gather ga = make_gather(d, f);
    TileAcc t;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
        const int col = wj + 16 * v + r, cn = col / 6;
        const int2 jc = ic[cn - cn0];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wi + 16 * u + 4 * i + q, rn = row / 6;
                t.a[u][v][i] = -gathered(ga, ir[rn - rn0], jc, row - 6 * rn, col - 6 * cn, row < b && col <= row);
            }
    }
    tile_product(d.mat + f.pan, k, m, k + DROWS * I, k + DROWS * J, 0, k, sh, sh + DROWS * (DKC + 2), tid, t);
    double* C = d.mat + f.mat;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wi + 16 * u + 4 * i + q, col = wj + 16 * v + r;
                if (row < b && col <= row) C[(int64_t)row * b + col] = -t.a[u][v][i];
            }
}

// ---------------------------------------------------------------------------
// device: solves
// ---------------------------------------------------------------------------
// a front's vector v (pivots, then border; [..][NR]): right-hand side of the
// pivots plus what its children pass up; nodes l0 <= l < l1
template <int NR>
__device__ __forceinline__ void gather_rhs(const DirectDev& d, const FrontTask& f, const double* __restrict__ r,
                                           int l0, int l1, double* dst, int tid, int nth) {
    const double *v0 = d.vec + f.cvec[0] * NR, *v1 = d.vec + f.cvec[1] * NR;
    for (int e = tid; e < (l1 - l0) * 6 * NR; e += nth) {
        const int l = l0 + e / (6 * NR), q = e % (6 * NR);
        const int2 a = d.inv[f.node0 + l];
        const double* pr = l < f.np ? r + ((int64_t)f.gnode0 + d.nodes[f.node0 + l]) * 6 * NR + q : d.zero;
        const double* p0 = a.x >= 0 ? v0 + a.x * 6 * NR + q : d.zero;
        const double* p1 = a.y >= 0 ? v1 + a.y * 6 * NR + q : d.zero;
        dst[e] = *pr + *p0 + *p1;
    }
}
template <int NR>
__device__ __forceinline__ bool any_active(const int32_t* __restrict__ active, int sys) {
    bool any = false;
#pragma unroll
    for (int h = 0; h < NR; ++h) any |= active[sys * NR + h] != 0;
    return any;
}

// r2 -= G r1 for one panel of every front, `rows` rows below it per workgroup; the
// first panel gathers the vector.  Bound by the reads of G (each once).
template <int NR>
__global__ __launch_bounds__(256) void k_solve_fwd(DirectDev d, const FrontTask* __restrict__ tasks,
                                                   const int32_t* __restrict__ active,
                                                   const double* __restrict__ r, int p, int n, int parts, int rows) {
    __shared__ double r1[DW * NR];
    const Where at = locate(n, parts);
    if (at.task >= n) return;
    const FrontTask f = tasks[at.task];
    if (p >= f.npan || !any_active<NR>(active, f.sys)) return;
    const int mn = f.np + f.nb, m = 6 * mn, p0 = p * f.wn, wn = min(f.wn, f.np - p0), w = 6 * wn, c0 = 6 * p0;
    const int r0 = c0 + w + rows * at.part;
    if (at.part > 0 && r0 >= m) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double* v = d.vec + f.vec * NR;
    const int r1end = min(m, r0 + rows);
    if (p == 0) {
        gather_rhs<NR>(d, f, r, 0, wn, r1, tid, 256);
        gather_rhs<NR>(d, f, r, r0 / 6, r1end / 6, v + (int64_t)r0 * NR, tid, 256);
    } else {
        for (int e = tid; e < w * NR; e += 256) r1[e] = v[(int64_t)c0 * NR + e];
    }
    __threadfence_block();
    __syncthreads();
    if (p == 0 && at.part == 0)
        for (int e = tid; e < w * NR; e += 256) v[e] = r1[e];
    const double* G = d.fac + f.fac + panel_offset(m, 6 * f.wn, p) + (int64_t)w * w;
    // 16 rows per wavefront; lane: row l % 16, columns 4 (l / 16) .. + 3 of every 16, all
    // loads of a row in flight
    for (int row0 = r0 + 16 * wave; row0 < r1end; row0 += 64) {
        const int row = row0 + (lane & 15), j0 = 4 * (lane >> 4);
        const bool on = row < r1end;
        const double* g = G + (int64_t)((on ? row : r0) - c0 - w) * w;
        double acc[NR];
#pragma unroll
        for (int h = 0; h < NR; ++h) acc[h] = 0.0;
        constexpr int T = NR == 1 ? DW / 16 : 2;   // (more load cases: fewer loads ahead, or registers run out)
#pragma unroll 1
        for (int t0 = 0; 16 * t0 < w; t0 += T) {
            double2 a[T][2];
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int j = j0 + 16 * (t0 + t) + 2 * u;
                    a[t][u] = *reinterpret_cast<const double2*>(j < w ? g + j : d.zero);
                }
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int j = min(j0 + 16 * (t0 + t) + 2 * u, w - 2);
#pragma unroll
                    for (int h = 0; h < NR; ++h)
                        acc[h] += a[t][u].x * r1[j * NR + h] + a[t][u].y * r1[(j + 1) * NR + h];
                }
        }
#pragma unroll
        for (int h = 0; h < NR; ++h) {
            acc[h] += __shfl_xor(acc[h], 16);
            acc[h] += __shfl_xor(acc[h], 32);
        }
        if (on && lane < 16) {
#pragma unroll
            for (int h = 0; h < NR; ++h) v[(int64_t)row * NR + h] -= acc[h];
        }
    }
}

// x1 = S r1 - G^T x2 for one panel of every front, its columns over `parts` workgroups;
// x in node order.  Bound by the reads of S and G, each once: a workgroup alone with the
// panel of a large front (2 300 rows of 96) took 13 us, eight take 8.
template <int NR, int NT>
__global__ __launch_bounds__(NT) void k_solve_bwd(DirectDev d, const FrontTask* __restrict__ tasks,
                                                  const int32_t* __restrict__ active, double* __restrict__ x, int p,
                                                  int n, int parts) {
    extern __shared__ double P[];
    const Where at = locate(n, parts);
    if (at.task >= n) return;
    const FrontTask f = tasks[at.task];
    if (p >= f.npan || f.np == 0 || !any_active<NR>(active, f.sys)) return;
    const int mn = f.np + f.nb, m = 6 * mn, p0 = p * f.wn, wn = min(f.wn, f.np - p0), w = 6 * wn, c0 = 6 * p0;
    const int tid = threadIdx.x, nb = m - c0 - w;
    double* r1 = P;                          // [w][NR], then x2 [nb][NR]: one vector for the rows of S and -G
    const double* v = d.vec + f.vec * NR + (int64_t)c0 * NR;
    for (int e = tid; e < (w + nb) * NR; e += NT) {
        const int l = p0 + e / (6 * NR), q = e % (6 * NR);
        r1[e] = e < w * NR ? v[e] : -x[((int64_t)f.gnode0 + d.nodes[f.node0 + l]) * 6 * NR + q];
    }
    __syncthreads();
    const double* S = d.fac + f.fac + panel_offset(m, 6 * f.wn, p);   // w rows of S (symmetric), then G's
    // lane pairs of columns, this part's from j0 on; groups of hw threads share the rows, eight in flight
    const int h0 = w / 2 * at.part / parts, hw = w / 2 * (at.part + 1) / parts - h0, j0 = 2 * h0, wj = 2 * hw;
    if (hw == 0) return;
    const int ng = NT / hw, g = tid / hw, j = 2 * (tid - g * hw);
    double acc[2][NR];
#pragma unroll
    for (int h = 0; h < NR; ++h) acc[0][h] = acc[1][h] = 0.0;
    if (g < ng) {
        for (int i0 = g; i0 < w + nb; i0 += 8 * ng) {
            double2 a[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = i0 + u * ng;
                a[u] = *reinterpret_cast<const double2*>(i < w + nb ? S + (int64_t)i * w + j0 + j : d.zero);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = min(i0 + u * ng, w + nb - 1);
#pragma unroll
                for (int h = 0; h < NR; ++h) {
                    acc[0][h] += a[u].x * r1[i * NR + h];
                    acc[1][h] += a[u].y * r1[i * NR + h];
                }
            }
        }
    }
    double* red = r1 + (w + nb) * NR;        // [ng][wj][NR]
    if (g < ng) {
#pragma unroll
        for (int h = 0; h < NR; ++h) {
            red[(g * wj + j) * NR + h] = acc[0][h];
            red[(g * wj + j + 1) * NR + h] = acc[1][h];
        }
    }
    __syncthreads();
    // sums over the groups: eight partial sums each, then those
    for (int e = tid; e < 8 * wj * NR; e += NT) {
        const int c = e % (wj * NR), q0 = e / (wj * NR);
        double s = 0.0;
        for (int q = q0; q < ng; q += 8) s += red[q * wj * NR + c];
        if (q0 < ng) red[e] = s;   // (its own first term's place)
    }
    __syncthreads();
    for (int e = tid; e < wj * NR; e += NT) {
        double s = 0.0;
        for (int q = 0; q < min(8, ng); ++q) s += red[q * wj * NR + e];
        const int c = j0 * NR + e, l = p0 + c / (6 * NR), q = c % (6 * NR);
        x[((int64_t)f.gnode0 + d.nodes[f.node0 + l]) * 6 * NR + q] = s;
    }
}

// x64 += z for the systems still running
template <int NR>
__global__ __launch_bounds__(SOLVER_WG) void k_direct_add(Slices sl, const int32_t* __restrict__ slice_act,
                                                          const double* __restrict__ z, double* __restrict__ x) {
    const int w = slice_of_block(sl);
    if (w < 0) return;
    const int mask = slice_act[w];
    const int64_t R = 6 * (int64_t)sl.row0[w] + threadIdx.x;
    if (mask == 0 || R >= 6 * (int64_t)sl.row1[w]) return;
#pragma unroll
    for (int h = 0; h < NR; ++h)
        if ((mask >> h) & 1) x[R * NR + h] += z[R * NR + h];
}

// what the host needs to know after a refinement step
__global__ __launch_bounds__(256) void k_direct_report(int nsys, int n_struct, const int32_t* __restrict__ status,
                                                       const double* __restrict__ best,
                                                       const int32_t* __restrict__ bad,
                                                       const int32_t* __restrict__ flags, DirectReport* out,
                                                       DirectReport* host) {
    __shared__ int cnt[5];
    __shared__ double worst[4];
    const int tid = threadIdx.x;
    if (tid < 5) cnt[tid] = 0;
    __syncthreads();
    int run = 0, stall = 0, floor = 0, nb = 0, load = 0;
    double w = 0.0;
    for (int k = tid; k < nsys; k += 256) {
        run += status[k] == SYS_RUNNING;
        stall += status[k] == SYS_STALLED;
        floor += status[k] == SYS_FLOOR;
        load += status[k] == SYS_LOAD;
        w = fmax(w, best[k]);
    }
    for (int k = tid; k < n_struct; k += 256) nb += bad[k] != 0;
    if (run) atomicAdd(&cnt[0], run);
    if (stall) atomicAdd(&cnt[1], stall);
    if (floor) atomicAdd(&cnt[2], floor);
    if (nb) atomicAdd(&cnt[3], nb);
    if (load) atomicAdd(&cnt[4], load);
    for (int o = 32; o > 0; o >>= 1) w = fmax(w, __shfl_xor(w, o));
    if ((tid & 63) == 0) worst[tid >> 6] = w;
    __syncthreads();
    if (tid == 0) {
        DirectReport v;
        v.running = cnt[0];
        v.stalled = cnt[1];
        v.floor = cnt[2];
        v.bad = cnt[3];
        v.not_finite = cnt[4];
        v.worst = fmax(fmax(worst[0], worst[1]), fmax(worst[2], worst[3]));
        v.flags = *flags;
        v.final = !(v.running | v.stalled | v.bad | (v.flags & (STATUS_NONSYM | 1)));
        *out = v;
        *host = v;   // pinned: no copy of its own
    }
}

// After a step's report: u = L^-T x of the best iterates where that is the end (u is
// not touched before: it may be f itself, which another route then still needs), NaN
// for a load that is not finite; else the iterates that have become the best are kept.
template <int NR>
__global__ __launch_bounds__(SOLVER_WG) void k_direct_finish(Slices sl, const int32_t* __restrict__ save,
                                                             const int32_t* __restrict__ status,
                                                             const DirectReport* __restrict__ report,
                                                             const double* __restrict__ Linv,
                                                             const double* __restrict__ x64,
                                                             double* __restrict__ xbest, double* __restrict__ u) {
    const int w = slice_of_block(sl);
    if (w < 0) return;
    const int sys = sl.sys[w];
    const int64_t R = 6 * (int64_t)sl.row0[w] + threadIdx.x;
    const bool end = report->final != 0;
    if (R >= 6 * (int64_t)sl.row1[w] || (!end && report->running == 0)) return;
    const int64_t i = R / 6;
    const int r = (int)(R % 6);
#pragma unroll
    for (int h = 0; h < NR; ++h) {
        const bool now = save[sys * NR + h] != 0;
        if (end) {
            const double* x = now ? x64 : xbest;
            double v = 0.0;
#pragma unroll
            for (int c = 0; c < 6; ++c) v += Linv[i * 36 + c * 6 + r] * x[(6 * i + c) * NR + h];
            u[R * NR + h] = status[sys * NR + h] == SYS_LOAD ? __builtin_nan("") : v;
        } else if (now) {
            xbest[R * NR + h] = x64[R * NR + h];
        }
    }
}

__global__ __launch_bounds__(256) void k_direct_clear(int n, int32_t* __restrict__ bad) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i < n) bad[i] = 0;
}

// ---------------------------------------------------------------------------
// device: refinement with a K that is not symmetric (the factorisation is of its
// symmetric part)
// ---------------------------------------------------------------------------
// r = f - op(K) u on the free DOFs, scaled to L^-1 r for the factorisation; per-slice
// partial sums of <r, r>.  Thread = scalar row of the slice, a row's blocks in column
// order; op(K) = K^T reads column rr of the block at the transposed position.
template <int NR>
__global__ __launch_bounds__(SOLVER_WG) void k_defect(Slices sl, Partials P, SysState st,
                                                      const int32_t* __restrict__ rowptr,
                                                      const int32_t* __restrict__ colind,
                                                      const int32_t* __restrict__ tpos,
                                                      const uint8_t* __restrict__ fixed,
                                                      const double* __restrict__ K, const double* __restrict__ Linv,
                                                      const double* __restrict__ f, const double* __restrict__ u,
                                                      double* __restrict__ rs) {
    __shared__ double lds[NWAVES * NR], rl[SOLVER_WG][NR];
    const int w = slice_of_block(sl);
    if (w < 0 || st.slice_act[w] == 0) return;
    const int tid = threadIdx.x;
    const int64_t R = 6 * (int64_t)sl.row0[w] + tid;
    const bool on = R < 6 * (int64_t)sl.row1[w];
    double v[NR];
#pragma unroll
    for (int h = 0; h < NR; ++h) v[h] = 0.0;
    const int i = (int)(R / 6), rr = (int)(R % 6);
    if (on && !fixed[R]) {
        double acc[NR];
#pragma unroll
        for (int h = 0; h < NR; ++h) acc[h] = 0.0;
        for (int k = rowptr[i]; k < rowptr[i + 1]; ++k) {
            const int64_t j = colind[k];
            const double* b = tpos ? K + (int64_t)tpos[k] * 36 + rr : K + (int64_t)k * 36 + rr * 6;
            const int step = tpos ? 6 : 1;
#pragma unroll
            for (int c = 0; c < 6; ++c)
#pragma unroll
                for (int h = 0; h < NR; ++h) acc[h] += b[c * step] * u[(6 * j + c) * NR + h];
        }
#pragma unroll
        for (int h = 0; h < NR; ++h) v[h] = f[R * NR + h] - acc[h];
    }
#pragma unroll
    for (int h = 0; h < NR; ++h) rl[tid][h] = v[h];
    __syncthreads();
    if (on) {
#pragma unroll
        for (int h = 0; h < NR; ++h) {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < 6; ++c) s += Linv[(int64_t)i * 36 + rr * 6 + c] * rl[tid - rr + c][h];
            rs[R * NR + h] = s;
            v[h] *= v[h];
        }
    }
    write_partials<NR, NWAVES>(v, lds, P.t, w);
}

// A system ends where its residual ||r|| / ||f|| no longer halves: at its attainable
// accuracy if that is within tol, else without convergence, as does a load whose squares
// leave the range of FP64.  One wavefront per structure; step 0 takes ||f|| from u = 0.
template <int NR>
__global__ __launch_bounds__(64) void k_defect_decide(Slices sl, Partials P, SysState st, int step, double tol) {
    const int sys = blockIdx.x, lane = threadIdx.x;
    const int s0 = sl.sys_off[sys], s1 = sl.sys_off[sys + 1];
    double t[NR];
#pragma unroll
    for (int h = 0; h < NR; ++h) t[h] = 0.0;
    for (int w = s0 + lane; w < s1; w += 64)
#pragma unroll
        for (int h = 0; h < NR; ++h) t[h] += P.t[(int64_t)w * NR + h];
    int mask = 0;
#pragma unroll
    for (int h = 0; h < NR; ++h) {
        const double rr = wave_sum(t[h]);
        const int k = sys * NR + h;
        if (!st.active[k]) continue;
        const double ff = step == 0 ? rr : st.bnorm2[k], prev = st.relres[k];
        const double rel = step == 0 ? 1.0 : sqrt(rr / ff);
        int active = 1, status = SYS_RUNNING;
        if (step == 0 ? !(rr >= LOAD2_MIN && rr <= LOAD2_MAX) : rel == 0.0 || !(rel <= 0.5 * prev)) {
            active = 0;
            status = rel <= tol ? SYS_CONVERGED : SYS_STALLED;
        }
        if (lane == 0) {
            if (step == 0) st.bnorm2[k] = ff;
            st.relres[k] = rel;
            st.best[k] = rel;
            st.active[k] = active;
            st.status[k] = status;
        }
        mask |= active << h;
    }
    for (int w = s0 + lane; w < s1; w += 64) st.slice_act[w] = mask;
}

// u = 0, NaN for a load that is not finite
template <int NR>
__global__ __launch_bounds__(SOLVER_WG) void k_defect_start(Slices sl, const int32_t* __restrict__ status,
                                                            double* __restrict__ u) {
    const int w = slice_of_block(sl);
    if (w < 0) return;
    const int sys = sl.sys[w];
    const int64_t R = 6 * (int64_t)sl.row0[w] + threadIdx.x;
    if (R >= 6 * (int64_t)sl.row1[w]) return;
#pragma unroll
    for (int h = 0; h < NR; ++h) u[R * NR + h] = status[sys * NR + h] == SYS_LOAD ? __builtin_nan("") : 0.0;
}

// u += L^-T z for the systems still running
template <int NR>
__global__ __launch_bounds__(SOLVER_WG) void k_defect_add(Slices sl, const int32_t* __restrict__ slice_act,
                                                          const double* __restrict__ Linv,
                                                          const double* __restrict__ z, double* __restrict__ u) {
    const int w = slice_of_block(sl);
    if (w < 0) return;
    const int mask = slice_act[w];
    const int64_t R = 6 * (int64_t)sl.row0[w] + threadIdx.x;
    if (mask == 0 || R >= 6 * (int64_t)sl.row1[w]) return;
    const int64_t i = R / 6;
    const int r = (int)(R % 6);
#pragma unroll
    for (int h = 0; h < NR; ++h) {
        if (!((mask >> h) & 1)) continue;
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < 6; ++c) s += Linv[i * 36 + c * 6 + r] * z[(6 * i + c) * NR + h];
        u[R * NR + h] += s;
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
static size_t small_front_lds(int np, int nb) {
    const int kp = (6 * np + 15) & ~15, bp = (6 * nb + 15) & ~15;
    return (size_t)(kp + bp) * (kp + 2) * 8 + (size_t)(np + nb + 3) * 8;
}

// first-fit allocation of the stored fronts of one structure: a front's matrix
// lives from its own level to its parent's
struct Arena {
    std::vector<std::pair<int64_t, int64_t>> holes;   // (offset, size), by offset
    int64_t top = 0;
    int64_t take(int64_t n) {
        if (n == 0) return 0;
        n = (n + 1) & ~(int64_t)1;
        for (size_t i = 0; i < holes.size(); ++i)
            if (holes[i].second >= n) {
                const int64_t at = holes[i].first;
                holes[i].first += n;
                holes[i].second -= n;
                if (holes[i].second == 0) holes.erase(holes.begin() + i);
                return at;
            }
        const int64_t at = top;
        top += n;
        return at;
    }
    void give(int64_t at, int64_t n) {
        n = (n + 1) & ~(int64_t)1;
        if (n == 0) return;
        auto it = std::lower_bound(holes.begin(), holes.end(), std::make_pair(at, (int64_t)0));
        it = holes.insert(it, {at, n});
        if (it + 1 != holes.end() && it->first + it->second == (it + 1)->first) {
            it->second += (it + 1)->second;
            holes.erase(it + 1);
        }
        if (it != holes.begin() && (it - 1)->first + (it - 1)->second == it->first) {
            (it - 1)->second += it->second;
            holes.erase(it);
        }
    }
};

// false where the fronts, or the storage of the structures so far, are past the limits
static bool direct_build_host(Plan* pl, DirectState& D, size_t most_bytes, std::vector<int32_t>& nodes,
                              std::vector<int32_t>& blk, std::vector<int32_t>& blkrow, std::vector<int2>& inv) {
    const auto& off = pl->h_node_off;
    struct Cls {
        int32_t fr0, n_fr, sys;
        int64_t fac, mat, vec;
    };
    std::vector<Cls> cls;
    std::map<uint64_t, std::vector<int>> by_hash;
    std::vector<FrontMeta> fr;
    struct Base {
        int64_t fac, mat, vec;
    };
    std::vector<Base> base(pl->n_sys);
    std::vector<int32_t> lrp, lci, cls_of(pl->n_sys);
    for (int s = 0; s < pl->n_sys; ++s) {
        const int32_t n0 = off[s], n = off[s + 1] - n0, b0 = pl->h_rowptr[n0];
        const int32_t nb = pl->h_rowptr[n0 + n] - b0;
        uint64_t h = 1469598103934665603ull ^ (uint64_t)n;
        for (int i = 0; i <= n; ++i) h = (h ^ (uint32_t)(pl->h_rowptr[n0 + i] - b0)) * 1099511628211ull;
        for (int k = 0; k < nb; ++k) h = (h ^ (uint32_t)(pl->h_colind[b0 + k] - n0)) * 1099511628211ull;
        int found = -1;
        for (int c : by_hash[h]) {
            const int t = cls[c].sys;
            const int32_t m0 = off[t], c0 = pl->h_rowptr[m0];
            if (off[t + 1] - m0 != n || pl->h_rowptr[m0 + n] - c0 != nb) continue;
            bool same = true;
            for (int i = 0; i <= n && same; ++i) same = pl->h_rowptr[n0 + i] - b0 == pl->h_rowptr[m0 + i] - c0;
            for (int k = 0; k < nb && same; ++k) same = pl->h_colind[b0 + k] - n0 == pl->h_colind[c0 + k] - m0;
            if (same) {
                found = c;
                break;
            }
        }
        if (found < 0) {
            lrp.resize(n + 1);
            lci.resize(nb);
            for (int i = 0; i <= n; ++i) lrp[i] = pl->h_rowptr[n0 + i] - b0;
            for (int k = 0; k < nb; ++k) lci[k] = pl->h_colind[b0 + k] - n0;
            FrontTree T;
            int32_t largest = 0;
            const bool fits = build_fronts(n, lrp.data(), lci.data(), DLEAF, T, DIRECT_MAX_M / 6, &largest);
            D.max_m = std::max(D.max_m, 6 * largest);
            if (!fits) return false;
            Cls C{(int32_t)fr.size(), (int32_t)T.fronts.size(), s, 0, 0, 0};
            const int32_t node_base = (int32_t)nodes.size(), blk_base = (int32_t)(blk.size() / 3);
            for (size_t t = 0; t < T.fronts.size(); ++t) {
                const auto& F = T.fronts[t];
                FrontMeta M{};
                M.np = F.np;
                M.nb = F.nb;
                M.node0 = node_base + F.node0;
                M.level = F.level;
                M.child[0] = M.child[1] = -1;
                for (int q = T.child_ptr[t]; q < T.child_ptr[t + 1]; ++q) {
                    if (q - T.child_ptr[t] >= 2) return false;
                    M.child[q - T.child_ptr[t]] = C.fr0 + T.child[q];
                }
                M.blk0 = blk_base + F.blk0;
                M.nblk = F.nblk;
                const int k = 6 * F.np, b = 6 * F.nb, m = k + b;
                M.small = k <= DW && small_front_lds(F.np, F.nb) <= DLDS_MAX;
                M.npan = M.small ? 1 : std::max(1, (k + DW - 1) / DW);
                M.wn = std::max(1, (F.np + M.npan - 1) / M.npan);
                M.npan = std::max(1, (F.np + M.wn - 1) / M.wn);
                M.fac = C.fac;
                M.vec = C.vec;
                for (int p = 0, c0 = 0; p < M.npan; ++p) {
                    const int w = std::min(6 * M.wn, k - c0);
                    C.fac += (int64_t)w * w + (int64_t)(m - c0 - w) * w;
                    c0 += w;
                }
                C.fac = (C.fac + 1) & ~(int64_t)1;
                C.vec += m;
                const double kd = k, bd = b;
                D.flops += kd * kd * kd + 2 * bd * kd * kd + bd * bd * kd;
                D.n_levels = std::max(D.n_levels, F.level + 1);
                fr.push_back(M);
            }
            // storage: level by level, a child's matrix is free once its parent's level is done
            std::vector<std::vector<int32_t>> lev;
            for (int t = 0; t < C.n_fr; ++t) {
                const int L = fr[C.fr0 + t].level;
                if ((int)lev.size() <= L) lev.resize(L + 1);
                lev[L].push_back(C.fr0 + t);
            }
            Arena A;
            auto cb = [](const FrontMeta& M) { return (int64_t)36 * M.nb * M.nb; };
            auto cols = [](const FrontMeta& M) { return M.small ? 0 : (int64_t)36 * (M.np + M.nb) * M.np; };
            for (auto& L : lev) {
                for (int t : L) {
                    fr[t].mat = A.take(cb(fr[t]));
                    fr[t].pan = A.take(cols(fr[t]));
                }
                for (int t : L) {
                    A.give(fr[t].pan, cols(fr[t]));
                    for (int c : fr[t].child)
                        if (c >= 0) A.give(fr[c].mat, cb(fr[c]));
                }
            }
            C.mat = A.top;
            inv.resize(inv.size() + T.nodes.size(), int2{-1, -1});
            for (size_t t = 0; t < T.fronts.size(); ++t)
                for (int c = 0; c < 2; ++c) {
                    const int ch = fr[C.fr0 + t].child[c];
                    if (ch < 0) continue;
                    const FrontMeta& G = fr[ch];
                    const int32_t* rl = T.rel.data() + T.fronts[ch - C.fr0].node0 + G.np;
                    for (int l = 0; l < G.nb; ++l) {
                        int2& a = inv[fr[C.fr0 + t].node0 + rl[l]];
                        (c ? a.y : a.x) = l;
                    }
                }
            nodes.insert(nodes.end(), T.nodes.begin(), T.nodes.end());
            blk.insert(blk.end(), T.blk.begin(), T.blk.end());
            for (int32_t q : T.blkrow) blkrow.push_back(blk_base + q);
            found = (int)cls.size();
            cls.push_back(C);
            by_hash[h].push_back(found);
        } else {
            const Cls& C = cls[found];
            for (int t = 0; t < C.n_fr; ++t) {
                const double kd = 6 * fr[C.fr0 + t].np, bd = 6 * fr[C.fr0 + t].nb;
                D.flops += kd * kd * kd + 2 * bd * kd * kd + bd * bd * kd;
            }
        }
        cls_of[s] = found;
        const Cls& C = cls[found];
        base[s] = Base{(int64_t)D.fac_n, (int64_t)D.mat_n, (int64_t)D.vec_n};
        D.fac_n += C.fac;
        D.mat_n += C.mat;
        D.vec_n += C.vec;
        if ((D.fac_n + D.mat_n) * 8 > most_bytes) return false;
    }
    D.small_tasks.resize(D.n_levels);
    D.big_tasks.resize(D.n_levels);
    D.small_m.assign(D.n_levels, 0);
    D.big_m.assign(D.n_levels, 0);
    D.big_k.assign(D.n_levels, 0);
    D.big_b.assign(D.n_levels, 0);
    D.big_w.assign(D.n_levels, 0);
    D.big_pan.assign(D.n_levels, 0);
    for (int s = 0; s < pl->n_sys; ++s) {
        const Cls& C = cls[cls_of[s]];
        for (int t = C.fr0; t < C.fr0 + C.n_fr; ++t) {
            const FrontMeta& M = fr[t];
            if (M.np == 0 && M.nb == 0) continue;   // (joins components: nothing to do)
            const Base& B = base[s];
            FrontTask T{M.np, M.nb, M.wn, M.npan, M.node0, M.blk0, M.nblk, pl->h_rowptr[off[s]], s, off[s], {0, 0},
                        B.mat + M.mat, B.mat + M.pan, B.fac + M.fac, B.vec + M.vec, {0, 0}, {0, 0}};
            for (int c = 0; c < 2; ++c)
                if (M.child[c] >= 0) {
                    const FrontMeta& G = fr[M.child[c]];
                    T.cb[c] = G.nb;
                    T.cmat[c] = B.mat + G.mat;
                    T.cvec[c] = B.vec + G.vec + 6 * G.np;
                }
            if (M.small) {
                D.small_tasks[M.level].push_back(T);
                if (M.np) D.small_m[M.level] = std::max(D.small_m[M.level], 6 * (M.np + M.nb));
            } else {
                D.big_tasks[M.level].push_back(T);
                D.big_m[M.level] = std::max(D.big_m[M.level], 6 * (M.np + M.nb));
                D.big_k[M.level] = std::max(D.big_k[M.level], 6 * M.np);
                D.big_b[M.level] = std::max(D.big_b[M.level], 6 * M.nb);
                D.big_w[M.level] = std::max(D.big_w[M.level], 6 * M.wn);
                D.big_pan[M.level] = std::max(D.big_pan[M.level], M.npan);
            }
        }
    }
    return true;
}

template <typename T>
static int direct_alloc(DirectState& D, T** dst, size_t count) {
    *dst = nullptr;
    void* q = nullptr;
    if (hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) {
        (void)hipGetLastError();
        return JSSO_ENOMEM;
    }
    D.allocs.push_back(q);
    *dst = (T*)q;
    return JSSO_OK;
}
template <typename T>
static int direct_upload(DirectState& D, const T** dst, const std::vector<T>& src) {
    T* p = nullptr;
    int rc = direct_alloc(D, &p, src.size());
    if (rc) return rc;
    if (!src.empty()) JSSO_HIP(hipMemcpy(p, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    *dst = p;
    return JSSO_OK;
}

void direct_destroy(Plan* pl) {
    DirectState* D = pl->direct;
    if (!D) return;
    for (void* a : D->allocs) (void)hipFree(a);
    if (D->dev.vec) (void)hipFree(D->dev.vec);
    if (D->h_report) (void)hipHostFree(D->h_report);
    delete D;
    pl->direct = nullptr;
}

// Builds the analysis and its storage; leaves D.usable false where the direct solve is
// not the better choice or does not fit.
//
// The direct solve is taken where its fronts stay small: fill and operations grow
// with the largest front (m rows: m^2 storage, m^3 operations), while the
// AMG-preconditioned CG grows with the number of nodes.  One shell of n x n quads
// has m ~ 9 n: assembly and solve of one smooth shell, ms direct / AMG: 40x40
// (m = 366) 0.79 / 1.9, 100x100 1.8 / 3.2, 200x200 4.8 / 6.7, 250x250 (m = 2256)
// 6.7 / 8.4, 300x300 10.2 / 9.4.  Designs that take the CG more iterations gain more,
// and so do batches, which fill the chip on every tree level (64 SIMP shells of
// 100x100, with gradients: 31.6 / 62).  It needs its storage too: up to an eighth of
// the card, and half of what is free.
static int direct_build(Plan* pl, DirectState& D) {
    std::vector<int32_t> nodes, blk, blkrow;
    std::vector<int2> inv;
    size_t free_b = 0, total_b = 0;
    JSSO_HIP(hipMemGetInfo(&free_b, &total_b));
    if (!direct_build_host(pl, D, std::min(total_b / 8, free_b / 2), nodes, blk, blkrow, inv)) return JSSO_OK;
    int rc = 0;
    std::vector<FrontTask> tasks;
    D.buckets.resize(D.n_levels);
    for (int L = 0; L < D.n_levels; ++L) {
        // small fronts by the LDS they need: 3, 2 or 1 workgroups per CU, of as many
        // threads as then fill it.  Fewer fronts than CUs go in one launch.
        auto& st = D.small_tasks[L];
        auto lds = [](const FrontTask& t) { return small_front_lds(t.np, t.nb); };
        std::stable_sort(st.begin(), st.end(),
                         [&](const FrontTask& x, const FrontTask& y) { return lds(x) > lds(y); });
        constexpr size_t limit[3] = {78 * 1024, 52 * 1024, 0};
        for (size_t i = 0; i < st.size();) {
            const size_t need = lds(st[i]);
            const int c = need > limit[0] ? 0 : need > limit[1] ? 1 : 2;
            size_t j = st.size();
            if (st.size() > 512)
                for (j = i; j < st.size() && lds(st[j]) > limit[c];) ++j;
            D.buckets[L].push_back({need, tasks.size() + i, j - i, 1024 >> c});
            i = j;
        }
        D.small_off.push_back(tasks.size());
        D.small_n.push_back(D.small_tasks[L].size());
        tasks.insert(tasks.end(), D.small_tasks[L].begin(), D.small_tasks[L].end());
        D.big_off.push_back(tasks.size());
        D.big_n.push_back(D.big_tasks[L].size());
        tasks.insert(tasks.end(), D.big_tasks[L].begin(), D.big_tasks[L].end());
    }
    std::vector<std::vector<FrontTask>>().swap(D.small_tasks);
    std::vector<std::vector<FrontTask>>().swap(D.big_tasks);
    // ||A||_2 <= 4: with identity diagonal blocks, x^T A x = sum_e x_e^T A_e x_e is at most
    // (nodes of an element) x sum_e x_e^T diag(A_e) x_e = (nodes of an element) ||x||^2
    std::vector<double> rho(pl->n_sys, 4.0);
    const double* dr = nullptr;
    if ((rc = direct_upload(D, &D.dev.nodes, nodes)) || (rc = direct_upload(D, &D.dev.inv, inv)) ||
        (rc = direct_upload(D, &D.dev.blk, blk)) || (rc = direct_upload(D, &D.dev.blkrow, blkrow)) ||
        (rc = direct_upload(D, &D.dev.kref, pl->h_kref)) || (rc = direct_upload(D, &D.d_tasks, tasks)) ||
        (rc = direct_upload(D, &dr, rho)) || (rc = direct_alloc(D, &D.d_report, 1)) ||
        (rc = direct_alloc(D, &D.dev.fac, D.fac_n)) || (rc = direct_alloc(D, &D.dev.mat, D.mat_n)) ||
        (rc = direct_alloc(D, &D.dev.bad, pl->n_sys)) ||
        (rc = direct_upload(D, &D.dev.zero, std::vector<double>(2, 0.0)))) {
        for (void* a : D.allocs) (void)hipFree(a);
        D.allocs.clear();
        return rc == JSSO_ENOMEM ? JSSO_OK : rc;
    }
    JSSO_HIP(hipHostMalloc((void**)&D.h_report, sizeof(DirectReport), hipHostMallocDefault));
    JSSO_HIP(hipHostGetDevicePointer((void**)&D.host_report, D.h_report, 0));
    D.d_rho = const_cast<double*>(dr);
    D.dev.A64 = pl->d_Ke64;
    const std::pair<const void*, size_t> lds[] = {
        {(const void*)k_front_small<1024>, DLDS_MAX}, {(const void*)k_front_small<512>, DLDS_MAX},
        {(const void*)k_front_small<256>, DLDS_MAX},  {(const void*)k_front_diag, DW * (DW + 2) * 8},
        {(const void*)k_front_strip, (DW + SROWS) * (DW + 2) * 8}, {(const void*)k_front_cols<true>, DW * (DW + 2) * 8},
        {(const void*)k_solve_bwd<1, 256>, DLDS_MAX}, {(const void*)k_solve_bwd<1, 1024>, DLDS_MAX},
        {(const void*)k_solve_bwd<2, 256>, DLDS_MAX}, {(const void*)k_solve_bwd<2, 1024>, DLDS_MAX},
        {(const void*)k_solve_bwd<3, 256>, DLDS_MAX}, {(const void*)k_solve_bwd<3, 1024>, DLDS_MAX},
        {(const void*)k_solve_bwd<4, 256>, DLDS_MAX}, {(const void*)k_solve_bwd<4, 1024>, DLDS_MAX}};
    for (const auto& l : lds)
        JSSO_HIP(hipFuncSetAttribute(l.first, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.second));
    D.usable = true;
    return JSSO_OK;
}

static int direct_factor(Plan* pl, DirectState& D, hipStream_t s) {
    hipLaunchKernelGGL(k_direct_clear, dim3((unsigned)((pl->n_sys + 255) / 256)), dim3(256), 0, s, pl->n_sys, D.dev.bad);
    static_assert((DW + SROWS) * (DW + 2) * 8 <= DLDS_MAX, "panel LDS");
    for (int L = 0; L < D.n_levels; ++L) {
        for (const auto& B : D.buckets[L]) {
            const FrontTask* t = D.d_tasks + B.off;
            const dim3 g((unsigned)B.n);
            if (B.threads == 1024)
                hipLaunchKernelGGL(k_front_small<1024>, g, dim3(1024), B.lds, s, D.dev, t);
            else if (B.threads == 512)
                hipLaunchKernelGGL(k_front_small<512>, g, dim3(512), B.lds, s, D.dev, t);
            else
                hipLaunchKernelGGL(k_front_small<256>, g, dim3(256), B.lds, s, D.dev, t);
        }
        const int nb = (int)D.big_n[L];
        if (nb) {
            const FrontTask* t = D.d_tasks + D.big_off[L];
            const int m = D.big_m[L], kw = (D.big_w[L] + 15) & ~15;   // largest front, widest panel
            // strips of 96 rows, or of 32 while that leaves CUs without work
            const int rows = (int64_t)nb * ((m + SROWS - 1) / SROWS) >= 512 ? SROWS : 32;
            const bool head = nb < HEAD_FRONTS;
            const size_t block = (size_t)kw * (kw + 2) * 8, tile = (size_t)2 * DROWS * (DKC + 2) * 8;
            for (int p = 0; p < D.big_pan[L]; ++p) {
                if (p == 0 || !head) hipLaunchKernelGGL(k_front_diag, dim3(nb), dim3(512), block, s, D.dev, t, p);
                const int strips = (m + rows - 1) / rows + 1;
                hipLaunchKernelGGL(k_front_strip, part_grid(nb, strips), dim3(1024),
                                   (size_t)(kw + rows) * (kw + 2) * 8, s, D.dev, t, p, nb, strips, rows);
                if (p + 1 < D.big_pan[L]) {
                    const int tiles = ((m + DROWS - 1) / DROWS) * ((D.big_k[L] + DROWS - 1) / DROWS);
                    const int parts = (tiles + 1) / 2;
                    if (head)
                        hipLaunchKernelGGL(k_front_cols<true>, part_grid(nb, parts + 1), dim3(512),
                                           std::max(block, 2 * tile), s, D.dev, t, p, nb, parts);
                    else
                        hipLaunchKernelGGL(k_front_cols<false>, part_grid(nb, tiles), dim3(256), tile, s, D.dev, t, p,
                                           nb, tiles);
                }
            }
            const int bt = (D.big_b[L] + DROWS - 1) / DROWS, tiles = bt * (bt + 1) / 2;
            if (bt)
                hipLaunchKernelGGL(k_front_cb, part_grid(nb, tiles), dim3(256), 0, s, D.dev, t, nb, tiles);
        }
    }
    JSSO_HIP(hipGetLastError());
    D.factored = true;
    ++D.factorisations;
    return JSSO_OK;
}

// z = M^-1 r (both in node order, [dof][NR])
template <int NR>
static void direct_apply(DirectState& D, const int32_t* active, const double* r, double* z, hipStream_t s) {
    for (int L = 0; L < D.n_levels; ++L) {
        if (D.small_n[L])
            hipLaunchKernelGGL((k_solve_fwd<NR>), part_grid(D.small_n[L], 1), dim3(256), 0, s, D.dev,
                               D.d_tasks + D.small_off[L], active, r, 0, (int)D.small_n[L], 1, 1 << 20);
        const int nb = (int)D.big_n[L];
        if (!nb) continue;
        const int rows = nb * ((D.big_m[L] + 191) / 192) >= 512 ? 192 : 48;   // (multiples of 6)
        const int parts = (D.big_m[L] + rows - 1) / rows;
        for (int p = 0; p < D.big_pan[L]; ++p)
            hipLaunchKernelGGL((k_solve_fwd<NR>), part_grid(nb, parts), dim3(256), 0, s, D.dev,
                               D.d_tasks + D.big_off[L], active, r, p, nb, parts, rows);
    }
    for (int L = D.n_levels - 1; L >= 0; --L) {
        const int nb = (int)D.big_n[L];
        // columns in parts while that leaves CUs without work
        const int cols = nb ? std::max(1, std::min(BWD_PARTS, 256 / nb)) : 1;
        for (int p = D.big_pan[L] - 1; nb && p >= 0; --p)
            hipLaunchKernelGGL((k_solve_bwd<NR, 1024>), part_grid(nb, cols), dim3(1024),
                               ((size_t)D.big_m[L] + 2 * 1024) * NR * 8, s, D.dev, D.d_tasks + D.big_off[L], active, z,
                               p, nb, cols);
        if (D.small_n[L])
            hipLaunchKernelGGL((k_solve_bwd<NR, 256>), part_grid(D.small_n[L], 1), dim3(256),
                               ((size_t)D.small_m[L] + 2 * 256) * NR * 8, s, D.dev, D.d_tasks + D.small_off[L], active,
                               z, 0, (int)D.small_n[L], 1);
    }
}

static int direct_vectors(DirectState& D, int nrhs, bool& have) {
    const size_t need = D.vec_n * nrhs * 8;
    have = true;
    if (D.vec_bytes >= need) return JSSO_OK;
    if (D.dev.vec) JSSO_HIP(hipFree(D.dev.vec));
    D.dev.vec = nullptr;
    D.vec_bytes = 0;
    if (hipMalloc((void**)&D.dev.vec, need) != hipSuccess) {
        (void)hipGetLastError();
        have = false;
        return JSSO_OK;
    }
    D.vec_bytes = need;
    return JSSO_OK;
}

static int ensure_factor(Plan* pl, DirectState& D, hipStream_t s) {
    if (D.factored) return JSSO_OK;
    std::pair<hipEvent_t, hipEvent_t>* ev = nullptr;
    timing_begin_slot(s, ev, JSSO_TIMING_SETUP);
    const int rc = direct_factor(pl, D, s);
    timing_end(s, ev);
    return rc;
}

// Waves per slice of the residual kernel, unless jsso_plan_cg_tuning has set them: as many
// as fit its registers, 4 with up to two load cases.  A rule and not a timing, so that two
// plans of one pattern sum in the same order.  Medians in us with 1 / 2 / 4 waves: gridshell
// of 121 nodes 4.1 / 3.9 / 3.7, 40 x 40 shell 7.3 / 6.1 / 5.6 (two load cases 8.0 / 6.7 /
// 6.7), 200 x 200 shell 15.5 / 15.9 / 15.3, 64 shells of 100 x 100 237 / 212 / 178.
template <int NR>
constexpr int residual_waves() {
    return WpsFits<double, NR, 4>::value ? 4 : WpsFits<double, NR, 2>::value ? 2 : 1;
}

// u = K^-1 f by the factorisation and refinement; done = false (and nothing said
// about u) where a pivot is not positive or a system does not reach its tolerance
// or its attainable accuracy (strict: or whose load's squares leave the range of FP64).
// A structure and load case whose load is not finite gets NaN and is not counted as
// converged (JSSO_NOT_CONVERGED).
template <int NR>
static int run_direct(Plan* pl, DirectState& D, const double* f, double* u, double tol, int maxit, int slot,
                      bool strict, jsso_info* info, hipStream_t s, bool& done) {
    Workspace w;
    int rc = get_workspace(pl, NR, w);
    if (rc) return rc;
    bool have = false;
    if ((rc = direct_vectors(D, NR, have)) || !have) return rc;
    const int nsys = pl->n_sys * NR;
    const Slices sl = make_slices(pl, 0, pl->n_wg);
    const dim3 g = slice_grid(sl);
    double* r = (double*)w.r[0];
    double* z = (double*)w.p;
    hipLaunchKernelGGL((k_init<double, NR, true>), g, dim3(SOLVER_WG), 0, s, sl, w.P, pl->d_fixed, pl->d_Linv, f,
                       w.b64, w.x64, w.xbest, (double*)w.xlo, r, z);
    hipLaunchKernelGGL((k_decide<NR>), dim3(pl->n_sys), dim3(64), 0, s, sl, w.P, w.st, pl->n_sys,
                       strict ? DECIDE_START_STRICT : DECIDE_START, tol, 0, 0, (const double*)nullptr, 0.0, 0);
    int32_t& wps = pl->direct_wps[slot][NR];
    if (wps <= 0) wps = residual_waves<NR>();
    if ((rc = ensure_factor(pl, D, s))) return rc;
    for (int it = 1; it <= std::min(maxit, DIRECT_STEPS); ++it) {
        direct_apply<NR>(D, w.st.active, r, it == 1 ? w.x64 : z, s);   // (x is zero before)
        if (it > 1)
            hipLaunchKernelGGL((k_direct_add<NR>), g, dim3(SOLVER_WG), 0, s, sl, (const int32_t*)w.st.slice_act,
                               (const double*)z, w.x64);
        auto residual = [&](auto W) {
            constexpr int WP = decltype(W)::value;
            hipLaunchKernelGGL((k_replace<double, NR, WP>), g, dim3(64 * WP), 0, s, sl, w.P, w.st,
                               (const double*)pl->d_Ke64, (const double*)w.b64, (const double*)w.x64, r);
        };
        if (WpsFits<double, NR, 4>::value && wps >= 4)
            residual(std::integral_constant<int, WpsFits<double, NR, 4>::value ? 4 : 1>());
        else if (WpsFits<double, NR, 2>::value && wps >= 2)
            residual(std::integral_constant<int, WpsFits<double, NR, 2>::value ? 2 : 1>());
        else
            residual(std::integral_constant<int, 1>());
        // (a step that gains less than 10% ends a system at its attainable accuracy as
        // converged there; off it, three steps in a row that gain less end it as stalled)
        hipLaunchKernelGGL((k_decide<NR>), dim3(pl->n_sys), dim3(64), 0, s, sl, w.P, w.st, pl->n_sys, DECIDE_STEP, tol,
                           1, 2, (const double*)D.d_rho, DIRECT_FLOOR_FACTOR, 0);
        hipLaunchKernelGGL(k_direct_report, dim3(1), dim3(256), 0, s, nsys, pl->n_sys, (const int32_t*)w.st.status,
                           (const double*)w.st.best, (const int32_t*)D.dev.bad, (const int32_t*)pl->d_status,
                           D.d_report, D.host_report);
        hipLaunchKernelGGL((k_direct_finish<NR>), g, dim3(SOLVER_WG), 0, s, sl, (const int32_t*)w.st.save,
                           (const int32_t*)w.st.status, (const DirectReport*)D.d_report, pl->d_Linv, (const double*)w.x64, w.xbest, u);
        JSSO_HIP(hipGetLastError());
        JSSO_HIP(hipStreamSynchronize(s));
        const DirectReport& R = *D.h_report;
        pl->status_cache = pl->status_last = R.flags;
        if (R.running && !R.bad && !R.stalled && !(R.flags & (STATUS_NONSYM | 1))) continue;
        if (!R.final) return JSSO_OK;
        done = true;
        ++D.finished;
        if (info) {
            *info = jsso_info{};
            info->iterations = info->replacements = it;
            info->converged = nsys - R.not_finite;
            info->n_systems = nsys;
            info->rel_residual = R.worst;
            info->at_floor = R.floor;
            info->waves_per_slice = wps;
        }
        timing_collect();
        return R.not_finite ? JSSO_NOT_CONVERGED : JSSO_OK;
    }
    return JSSO_OK;
}

// the plan's analysis, built at its first use; nullptr where the direct solve is not taken
static int direct_state(Plan* pl, int nrhs, DirectState** out) {
    *out = nullptr;
    if (!(nrhs >= 1 && nrhs <= 4)) return JSSO_OK;
    if (!pl->direct) {
        pl->direct = new (std::nothrow) DirectState();
        if (!pl->direct) return JSSO_OK;
        int rc = JSSO_OK;
        try {
            rc = direct_build(pl, *pl->direct);
        } catch (const std::bad_alloc&) {   // (host memory: the iterative solve needs less)
            pl->direct->usable = false;
        }
        if (rc) {
            direct_destroy(pl);
            return rc;
        }
    }
    DirectState& D = *pl->direct;
    if (!D.usable) return JSSO_OK;
    if (!pl->direct_valid) D.factored = false;
    pl->direct_valid = true;
    *out = &D;
    ++D.begun;
    return JSSO_OK;
}

void direct_info(const Plan* pl, int64_t* out) {
    const DirectState* D = pl->direct;
    out[0] = D ? D->usable : -1;
    out[1] = D ? D->max_m : 0;
    out[2] = D ? (int64_t)((D->fac_n + D->mat_n) * 8 + D->vec_bytes) : 0;
    out[3] = D ? (int64_t)D->flops : 0;
    out[4] = D ? D->factorisations : 0;
    out[5] = D ? D->begun : 0;
    out[6] = D ? D->finished : 0;
}

int direct_solve(Plan* pl, const double* f, double* u, int nrhs, int slot, double tol, int maxit, bool strict,
                 jsso_info* info, hipStream_t s, bool& done) {
    done = false;
    DirectState* D = nullptr;
    int rc = direct_state(pl, nrhs, &D);
    if (rc || !D) return rc;
    switch (nrhs) {
        case 1: return run_direct<1>(pl, *D, f, u, tol, maxit, slot, strict, info, s, done);
        case 2: return run_direct<2>(pl, *D, f, u, tol, maxit, slot, strict, info, s, done);
        case 3: return run_direct<3>(pl, *D, f, u, tol, maxit, slot, strict, info, s, done);
        default: return run_direct<4>(pl, *D, f, u, tol, maxit, slot, strict, info, s, done);
    }
}

template <int NR>
static int run_defect(Plan* pl, DirectState& D, const double* K, const double* f, double* u, bool transpose,
                      double tol, int maxit, jsso_info* info, hipStream_t s, bool& done) {
    Workspace w;
    int rc = get_workspace(pl, NR, w);
    if (rc) return rc;
    bool have = false;
    if ((rc = direct_vectors(D, NR, have)) || !have) return rc;
    const int nsys = pl->n_sys * NR;
    const Slices sl = make_slices(pl, 0, pl->n_wg);
    const dim3 g = slice_grid(sl);
    double *r = (double*)w.r[0], *z = (double*)w.p;
    // activity from L^-1 f
    hipLaunchKernelGGL((k_init<double, NR, true>), g, dim3(SOLVER_WG), 0, s, sl, w.P, pl->d_fixed, pl->d_Linv, f,
                       w.b64, w.x64, w.xbest, (double*)w.xlo, r, z);
    hipLaunchKernelGGL((k_decide<NR>), dim3(pl->n_sys), dim3(64), 0, s, sl, w.P, w.st, pl->n_sys,
                       DECIDE_START_STRICT, tol, 0, 0, (const double*)nullptr, 0.0, 0);
    hipLaunchKernelGGL((k_defect_start<NR>), g, dim3(SOLVER_WG), 0, s, sl, (const int32_t*)w.st.status, u);
    if ((rc = ensure_factor(pl, D, s))) return rc;
    const int most = std::min(maxit, DEFECT_STEPS);
    for (int it = 0; it <= most; ++it) {
        hipLaunchKernelGGL((k_defect<NR>), g, dim3(SOLVER_WG), 0, s, sl, w.P, w.st, pl->d_rowptr, pl->d_colind,
                           transpose ? (const int32_t*)pl->d_tpos : (const int32_t*)nullptr, pl->d_fixed, K,
                           pl->d_Linv, f, (const double*)u, r);
        hipLaunchKernelGGL((k_defect_decide<NR>), dim3(pl->n_sys), dim3(64), 0, s, sl, w.P, w.st, it, tol);
        // (the host looks from the fourth step on, at every second one: a gain of 30 a
        // step, the best seen, needs five)
        if (it == most || (it >= 4 && it % 2 == 0)) {
            hipLaunchKernelGGL(k_direct_report, dim3(1), dim3(256), 0, s, nsys, pl->n_sys,
                               (const int32_t*)w.st.status, (const double*)w.st.best, (const int32_t*)D.dev.bad,
                               (const int32_t*)pl->d_status, D.d_report, D.host_report);
            JSSO_HIP(hipGetLastError());
            JSSO_HIP(hipStreamSynchronize(s));
            const DirectReport& R = *D.h_report;
            if (R.bad || R.stalled) return JSSO_OK;
            if (!R.running) {
                done = true;
                ++D.finished;
                if (info) {
                    *info = jsso_info{};
                    info->iterations = info->replacements = it;
                    info->converged = nsys - R.not_finite;
                    info->n_systems = nsys;
                    info->rel_residual = R.worst;
                }
                return R.not_finite ? JSSO_NOT_CONVERGED : JSSO_OK;
            }
        }
        direct_apply<NR>(D, w.st.active, r, z, s);
        hipLaunchKernelGGL((k_defect_add<NR>), g, dim3(SOLVER_WG), 0, s, sl, (const int32_t*)w.st.slice_act,
                           pl->d_Linv, (const double*)z, u);
    }
    return JSSO_OK;
}

// op(K) u = f for a K that is not symmetric (block CSR values K), by refinement with
// the factorisation of S = (K + K^T) / 2; done = false where it does not converge
int direct_defect(Plan* pl, const double* K, const double* f, double* u, int nrhs, bool transpose, double tol,
                  int maxit, jsso_info* info, hipStream_t s, bool& done) {
    done = false;
    DirectState* D = nullptr;
    int rc = direct_state(pl, nrhs, &D);
    if (rc || !D) return rc;
    switch (nrhs) {
        case 1: return run_defect<1>(pl, *D, K, f, u, transpose, tol, maxit, info, s, done);
        case 2: return run_defect<2>(pl, *D, K, f, u, transpose, tol, maxit, info, s, done);
        case 3: return run_defect<3>(pl, *D, K, f, u, transpose, tol, maxit, info, s, done);
        default: return run_defect<4>(pl, *D, K, f, u, transpose, tol, maxit, info, s, done);
    }
}

}  // namespace jsso
