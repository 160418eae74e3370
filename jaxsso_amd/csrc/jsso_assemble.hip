// Numeric assembly on the 6x6 block pattern (gathers over the element blocks,
// fixed summation order, no atomics), constraint masking and the block-Jacobi
// scaling the solver uses.  The solver needs only the factors of the diagonal
// blocks and the scaled off-diagonal blocks in sliced ELL; both are gathered
// straight from the element blocks.  K and Kc in block CSR (export, y = K x,
// the plain path) are gathered on demand.
//
//   K_ij       = sum over contributions (element e, local a, b) of Ke_e[a][b]
//   Kc         = K with rows/columns of constrained DOFs replaced by identity
//   Kc_ii      = L_i L_i^T (Cholesky), Linv_i = L_i^-1
//   Ks_ij      = Linv_i Kc_ij Linv_j^T   (i != j; Ks_ii = I implicitly)
//
// The Lagrange-multiplier system of the reference (assemblemodel.py:111-163)
// and this constrained system have the same u: every prescribed displacement
// is zero, so u_c = 0 and K_ff u_f = f_f.
#include "jsso_internal.hpp"

namespace jsso {

// Block-CSR K, 128 blocks per workgroup.  Each value is the sum of its element
// contributions in element order (beams, then quads, element index, a, b).  Bound by
// memory: the element blocks are read once or twice and K is written; a thread reads
// W entries of up to MAX_CONTRIB contributions of three blocks before the first sum,
// entries fastest, so that every access is whole lines.  W = 2 needs 16-byte aligned
// K.  KC: also the constrained Kc (plain path).  A 200 x 200 shell (361k blocks,
// 104 MB of K) took 151 us with a thread per entry and both outputs, and 40 us more to
// copy K to the caller; this takes 62 us, straight into the caller's buffer.
constexpr int GATHER_BLOCKS = 128;
constexpr int MAX_CONTRIB = 2;   // element blocks per off-diagonal block read without a loop (2 on a quad mesh)

template <int W, bool KC>
__global__ __launch_bounds__(256) void gather_blocks_kernel(int64_t nnzb, const int32_t* __restrict__ cptr,
                                                            const int32_t* __restrict__ csrc,
                                                            const int32_t* __restrict__ browof,
                                                            const int32_t* __restrict__ colind,
                                                            const uint8_t* __restrict__ fixed,
                                                            const double* __restrict__ ke,
                                                            double* __restrict__ K, double* __restrict__ Kc) {
    struct alignas(8 * W) Vec {
        double v[W];
    };
    constexpr int G = 36 / W, ITEMS = GATHER_BLOCKS * G / 256, AHEAD = 3;
    static_assert(GATHER_BLOCKS * G % 256 == 0 && ITEMS % AHEAD == 0, "whole rounds");
    __shared__ int32_t src[GATHER_BLOCKS][MAX_CONTRIB], start[GATHER_BLOCKS], count[GATHER_BLOCKS];
    __shared__ uint8_t rfix[GATHER_BLOCKS], cfix[GATHER_BLOCKS], diag[GATHER_BLOCKS];
    const int64_t k0 = xcd_wg() * GATHER_BLOCKS;
    if (k0 >= nnzb) return;
    const int t = threadIdx.x;
    if (t < GATHER_BLOCKS) {
        int c0 = 0, n = 0;
        int32_t e[MAX_CONTRIB] = {};   // 0 (a valid block) when unused
        if (k0 + t < nnzb) {
            c0 = cptr[k0 + t];
            n = cptr[k0 + t + 1] - c0;
            for (int c = 0; c < n && c < MAX_CONTRIB; ++c) e[c] = csrc[c0 + c];
            if (KC) {
                const int64_t i = browof[k0 + t], j = colind[k0 + t];
                int fr = 0, fc = 0;
                for (int r = 0; r < 6; ++r) {
                    fr |= (fixed[6 * i + r] != 0) << r;
                    fc |= (fixed[6 * j + r] != 0) << r;
                }
                rfix[t] = (uint8_t)fr;
                cfix[t] = (uint8_t)fc;
                diag[t] = i == j;
            }
        }
        for (int c = 0; c < MAX_CONTRIB; ++c) src[t][c] = e[c];
        start[t] = c0;
        count[t] = n;
    }
    __syncthreads();
    const Vec* kv = (const Vec*)ke;
#pragma unroll 1
    for (int r = 0; r < ITEMS; r += AHEAD) {
        Vec v[AHEAD][MAX_CONTRIB];
#pragma unroll
        for (int h = 0; h < AHEAD; ++h) {
            const int it = t + (r + h) * 256, b = it / G, q = it % G;
#pragma unroll
            for (int c = 0; c < MAX_CONTRIB; ++c) v[h][c] = kv[(int64_t)src[b][c] * G + q];
        }
#pragma unroll
        for (int h = 0; h < AHEAD; ++h) {
            const int it = t + (r + h) * 256, b = it / G, q = it % G, n = count[b];
            Vec sum = {};
#pragma unroll
            for (int c = 0; c < MAX_CONTRIB; ++c)
#pragma unroll
                for (int w = 0; w < W; ++w)
                    if (c < n) sum.v[w] += v[h][c].v[w];
            for (int c = MAX_CONTRIB; c < n; ++c) {   // the diagonal, and nodes of many members
                const Vec x = kv[(int64_t)csrc[start[b] + c] * G + q];
#pragma unroll
                for (int w = 0; w < W; ++w) sum.v[w] += x.v[w];
            }
            if (k0 + b >= nnzb) break;
            ((Vec*)K)[k0 * G + it] = sum;
            if (KC) {
                Vec x;
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const int row = (q * W + w) / 6, col = (q * W + w) % 6;
                    const bool held = ((rfix[b] >> row) | (cfix[b] >> col)) & 1;
                    x.v[w] = !held ? sum.v[w] : (diag[b] && row == col) ? 1.0 : 0.0;
                }
                ((Vec*)Kc)[k0 * G + it] = x;
            }
        }
    }
}

// Per node: the constrained diagonal block, summed from its element blocks in
// the same order as K, its Cholesky factor, the inverse factor and the
// block-Jacobi inverse Minv_i = Linv_i^T Linv_i.  status[0] |= 1 when a block
// is not positive definite.  64 nodes per workgroup: all threads gather the blocks
// (entry fastest) into LDS, the first wave factorises a node per lane, all threads
// write.  A lane per node reading and writing its own 36-value rows took 37 us for
// 40k nodes (a 200 x 200 shell); this takes 20 us, bound by the chain of one
// factorisation and by two rounds of memory latency.  The coordinates that the plan
// keeps are copied here as well: a copy of its own costs a launch.
constexpr int DIAG_NODES = 64;
constexpr int DIAG_CONTRIB = 4;   // element blocks of a node read without a loop (4 on a quad mesh)

__global__ __launch_bounds__(256) void diag_factor_kernel(int32_t n_nodes, const int32_t* __restrict__ diag,
                                                          const int32_t* __restrict__ cptr,
                                                          const int32_t* __restrict__ csrc,
                                                          const uint8_t* __restrict__ fixed,
                                                          const double* __restrict__ ke,
                                                          double* __restrict__ Linv, double* __restrict__ Minv,
                                                          int32_t* status, const double* __restrict__ crds,
                                                          double* __restrict__ crds_kept) {
    __shared__ double tile[DIAG_NODES][37], minv[DIAG_NODES][37];
    __shared__ int32_t src[DIAG_NODES][DIAG_CONTRIB], start[DIAG_NODES], count[DIAG_NODES];
    const int64_t i0 = xcd_wg() * DIAG_NODES;
    if (i0 >= n_nodes) return;
    const int t = threadIdx.x, nn = (int)(n_nodes - i0 < DIAG_NODES ? n_nodes - i0 : DIAG_NODES);
    if (t < DIAG_NODES) {
        int c0 = 0, n = 0;
        int32_t e[DIAG_CONTRIB] = {};
        if (t < nn) {
            const int k = diag[i0 + t];
            c0 = cptr[k];
            n = cptr[k + 1] - c0;
            for (int c = 0; c < n && c < DIAG_CONTRIB; ++c) e[c] = csrc[c0 + c];
        }
        for (int c = 0; c < DIAG_CONTRIB; ++c) src[t][c] = e[c];
        start[t] = c0;
        count[t] = n;
    } else if (t - DIAG_NODES < 3 * nn) {   // 192 threads, 3 x 64 coordinates
        crds_kept[3 * i0 + t - DIAG_NODES] = crds[3 * i0 + t - DIAG_NODES];
    }
    __syncthreads();
    constexpr int ITEMS = DIAG_NODES * 36 / 256, AHEAD = 3;   // 9
#pragma unroll
    for (int r = 0; r < ITEMS; r += AHEAD) {
        double v[AHEAD][DIAG_CONTRIB];
#pragma unroll
        for (int h = 0; h < AHEAD; ++h) {
            const int it = t + (r + h) * 256, b = it / 36, q = it % 36;
#pragma unroll
            for (int c = 0; c < DIAG_CONTRIB; ++c) v[h][c] = ke[(int64_t)src[b][c] * 36 + q];
        }
#pragma unroll
        for (int h = 0; h < AHEAD; ++h) {
            const int it = t + (r + h) * 256, b = it / 36, q = it % 36, n = count[b];
            double sum = 0.0;
#pragma unroll
            for (int c = 0; c < DIAG_CONTRIB; ++c)
                if (c < n) sum += v[h][c];
            for (int c = DIAG_CONTRIB; c < n; ++c) sum += ke[(int64_t)csrc[start[b] + c] * 36 + q];
            tile[b][q] = sum;
        }
    }
    __syncthreads();
    if (t < nn) {
        const int64_t i = i0 + t;
        double A[6][6], L[6][6], Li[6][6], B[36];
#pragma unroll
        for (int q = 0; q < 36; ++q) B[q] = tile[t][q];
        bool fx[6];
#pragma unroll
        for (int r = 0; r < 6; ++r) fx[r] = fixed[6 * i + r] != 0;
#pragma unroll
        for (int r = 0; r < 6; ++r)
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                const double brc = (fx[r] | fx[c]) ? (r == c ? 1.0 : 0.0) : B[r * 6 + c];
                const double bcr = (fx[r] | fx[c]) ? (r == c ? 1.0 : 0.0) : B[c * 6 + r];
                A[r][c] = 0.5 * (brc + bcr);
                L[r][c] = 0.0;
                Li[r][c] = 0.0;
            }
        bool ok = true;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            double d = A[j][j];
#pragma unroll
            for (int k = 0; k < j; ++k) d -= L[j][k] * L[j][k];
            if (!(d > 0.0)) { ok = false; d = 1.0; }
            const double ljj = sqrt(d);
            L[j][j] = ljj;
#pragma unroll
            for (int r = j + 1; r < 6; ++r) {
                double s = A[r][j];
#pragma unroll
                for (int k = 0; k < j; ++k) s -= L[r][k] * L[j][k];
                L[r][j] = s / ljj;
            }
        }
        // inverse of the lower-triangular factor
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            Li[j][j] = 1.0 / L[j][j];
#pragma unroll
            for (int r = j + 1; r < 6; ++r) {
                double s = 0.0;
#pragma unroll
                for (int k = j; k < r; ++k) s -= L[r][k] * Li[k][j];
                Li[r][j] = s / L[r][r];
            }
        }
#pragma unroll
        for (int r = 0; r < 6; ++r)
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                tile[t][r * 6 + c] = Li[r][c];
                double s = 0.0;
#pragma unroll
                for (int k = 0; k < 6; ++k) s += Li[k][r] * Li[k][c];
                minv[t][r * 6 + c] = s;
            }
        if (!ok) atomicOr(status, 1);
    }
    __syncthreads();
    for (int it = t; it < nn * 36; it += 256) {
        Linv[i0 * 36 + it] = tile[it / 36][it % 36];
        Minv[i0 * 36 + it] = minv[it / 36][it % 36];
    }
}

// One workgroup per sliced-ELL slot (64 positions, one per block row of the
// slice): the slot's off-diagonal blocks are summed from their element blocks
// (same order as K), masked (a constrained row or column of an off-diagonal
// block is zero), scaled Ks_ij = Linv_i Kc_ij Linv_j^T and written to the FP64,
// FP32 and FP16 ELL copies (the solver's residual replacement, its iterations,
// and the AMG smoothing products).  Padding positions (src < 0) keep their zeros.
//   phase 1: all 256 threads read the element blocks as (position, entry) pairs,
//            entry fastest (consecutive threads, consecutive values; every load
//            of a thread issued before the first sum), and stage the blocks, the
//            row factors L_i^-1 (64 consecutive rows: contiguous) and the column
//            factors L_j^-1 in LDS;
//   phase 2: wave w computes columns c = w, w + 4 of every position's Ks (lane =
//            position);
//   phase 3: Ks goes back through LDS and out in the value-slot layout (16-byte
//            groups of entries, lanes interleaved per group), whole lines at a time.
//            Stored from phase 2 entry by entry, 160k blocks (a 200 x 200 shell) took
//            71 us; this takes 62 us.
constexpr int ASM_WG = 256;

struct alignas(8) Half4 {
    _Float16 v[4];
};

__global__ __launch_bounds__(ASM_WG) void ell_assemble_kernel(
    int64_t n_slots, const int32_t* __restrict__ ell_src, const int32_t* __restrict__ browof,
    const int32_t* __restrict__ colind, const int32_t* __restrict__ cptr, const int32_t* __restrict__ csrc,
    const uint8_t* __restrict__ fixed, const double* __restrict__ ke, const double* __restrict__ Linv,
    double* __restrict__ Ke64, float* __restrict__ Ke32, _Float16* __restrict__ Ke16, int32_t n_beam,
    const int32_t* __restrict__ status) {
    constexpr int P = ROWS_PER_WG;
    // K not symmetric (set by this assembly's element kernels): the solver copies
    // hold the symmetric part (K_ij + K_ji^T) / 2, the preconditioning operator of
    // the defect correction; the element blocks of (j, i) are the swapped
    // element-local blocks of the same elements
    const bool sym_part = (*status & STATUS_NONSYM) != 0;
    __shared__ double tile[P][37];
    __shared__ double li[P][21], lj[P][21];   // lower triangles, row by row
    __shared__ int32_t cidx[P][MAX_CONTRIB], cstart[P], ccount[P], rowi[P], colj[P];
    __shared__ uint8_t rfix[P][6], cfix[P][6];
    const int64_t slot = blockIdx.x;
    if (slot >= n_slots) return;
    const int t = threadIdx.x;
    if (t < P) {
        const int32_t src = ell_src[slot * P + t];
        int n = 0, c0 = 0, i = 0, j = 0;
        int32_t e[MAX_CONTRIB] = {};
        if (src >= 0) {
            c0 = cptr[src];
            n = cptr[src + 1] - c0;
            for (int c = 0; c < n && c < MAX_CONTRIB; ++c) e[c] = csrc[c0 + c];
            i = browof[src];
            j = colind[src];
#pragma unroll
            for (int r = 0; r < 6; ++r) {
                rfix[t][r] = fixed[6 * (int64_t)i + r];
                cfix[t][r] = fixed[6 * (int64_t)j + r];
            }
        }
#pragma unroll
        for (int c = 0; c < MAX_CONTRIB; ++c) cidx[t][c] = e[c];   // 0 (a valid block) when unused
        cstart[t] = c0;
        ccount[t] = n;
        rowi[t] = i;
        colj[t] = j;
    }
    __syncthreads();
    constexpr int NPAIR = P * 36 / ASM_WG;   // 9
    double v[NPAIR][MAX_CONTRIB];
#pragma unroll
    for (int it = 0; it < NPAIR; ++it) {
        const int u = t + it * ASM_WG;
        const int p = u / 36, q = u % 36;
#pragma unroll
        for (int c = 0; c < MAX_CONTRIB; ++c) v[it][c] = ke[(int64_t)cidx[p][c] * 36 + q];
    }
    for (int u = t; u < P * 21; u += ASM_WG) {
        const int p = u / 21, q = u % 21;
        const int r = (q >= 1) + (q >= 3) + (q >= 6) + (q >= 10) + (q >= 15), at = 6 * r + q - r * (r + 1) / 2;
        li[p][q] = Linv[(int64_t)rowi[p] * 36 + at];
        lj[p][q] = Linv[(int64_t)colj[p] * 36 + at];
    }
#pragma unroll
    for (int it = 0; it < NPAIR; ++it) {
        const int u = t + it * ASM_WG;
        const int p = u / 36, q = u % 36;
        const int n = ccount[p];
        double sum = 0.0;
#pragma unroll
        for (int c = 0; c < MAX_CONTRIB; ++c)
            if (c < n) sum += v[it][c];
        for (int c = MAX_CONTRIB; c < n; ++c) sum += ke[(int64_t)csrc[cstart[p] + c] * 36 + q];   // rare meshes
        if (sym_part) {
            const int qt = (q % 6) * 6 + q / 6;
            double st = 0.0;
            for (int c = 0; c < n; ++c) {
                const int32_t src = c < MAX_CONTRIB ? cidx[p][c] : csrc[cstart[p] + c];
                int64_t sw;
                if (src < 4 * n_beam) {
                    const int l = src & 3;
                    sw = (src & ~3) | ((l & 1) << 1) | (l >> 1);
                } else {
                    const int64_t qq = src - 4 * (int64_t)n_beam;
                    const int l = (int)(qq & 15);
                    sw = 4 * (int64_t)n_beam + (qq & ~(int64_t)15) + ((l & 3) << 2) + (l >> 2);
                }
                st += ke[sw * 36 + qt];
            }
            sum = 0.5 * (sum + st);
        }
        tile[p][q] = (n > 0 && !(rfix[p][q / 6] | cfix[p][q % 6])) ? sum : 0.0;
    }
    __syncthreads();
    const int wave = t >> 6, lane = t & 63;
    double Ks[2][6];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int c = wave + 4 * h;
        if (c >= 6) break;
        // column c of T = B Lj^T, then column c of Ks = Li T (both factors lower triangular)
        double Tc[6];
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            double s = 0.0;
#pragma unroll
            for (int k2 = 0; k2 < 6; ++k2)
                if (k2 <= c) s += tile[lane][r * 6 + k2] * lj[lane][c * (c + 1) / 2 + k2];
            Tc[r] = s;
        }
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            double s = 0.0;
#pragma unroll
            for (int k2 = 0; k2 <= r; ++k2) s += li[lane][r * (r + 1) / 2 + k2] * Tc[k2];
            Ks[h][r] = ccount[lane] ? s : 0.0;   // padding (or an empty block): zero
        }
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int c = wave + 4 * h;
        if (c >= 6) break;
#pragma unroll
        for (int r = 0; r < 6; ++r) tile[lane][r * 6 + c] = Ks[h][r];
    }
    __syncthreads();
    // value-slot layout: 16-byte groups of entries, lanes interleaved per group
    // (2 doubles / 4 floats per group)
    const int64_t base = slot * 36 * P;
    double2* out64 = (double2*)(Ke64 + base);
    float4* out32 = (float4*)(Ke32 + base);
    Half4* out16 = (Half4*)(Ke16 + base);
    for (int g = t; g < 18 * P; g += ASM_WG) {
        const double* v = &tile[g % P][2 * (g / P)];
        out64[g] = make_double2(v[0], v[1]);
    }
    for (int g = t; g < 9 * P; g += ASM_WG) {
        const double* v = &tile[g % P][4 * (g / P)];
        out32[g] = make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
        out16[g] = Half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
    }
}

// K and Kc in block CSR, for callers that need them (export, y = K x, the plain path).
int launch_full_blocks(Plan* p, hipStream_t s) {
    if (p->full_valid || p->nnzb == 0) return JSSO_OK;
    const dim3 grid = xcd_grid((p->nnzb + GATHER_BLOCKS - 1) / GATHER_BLOCKS);
    hipLaunchKernelGGL((gather_blocks_kernel<2, true>), grid, dim3(256), 0, s, p->nnzb, p->d_cptr, p->d_csrc,
                       p->d_browof, p->d_colind, p->d_fixed, p->d_ke, p->d_K, p->d_Kc);
    JSSO_HIP(hipGetLastError());
    p->full_valid = true;
    return JSSO_OK;
}

// K alone into the caller's buffer (which may be 8-byte aligned only).
int launch_export_blocks(Plan* p, double* K, hipStream_t s) {
    if (p->nnzb == 0) return JSSO_OK;
    const dim3 grid = xcd_grid((p->nnzb + GATHER_BLOCKS - 1) / GATHER_BLOCKS);
    if (((uintptr_t)K & 15) == 0)
        hipLaunchKernelGGL((gather_blocks_kernel<2, false>), grid, dim3(256), 0, s, p->nnzb, p->d_cptr, p->d_csrc,
                           p->d_browof, p->d_colind, p->d_fixed, p->d_ke, K, (double*)nullptr);
    else
        hipLaunchKernelGGL((gather_blocks_kernel<1, false>), grid, dim3(256), 0, s, p->nnzb, p->d_cptr, p->d_csrc,
                           p->d_browof, p->d_colind, p->d_fixed, p->d_ke, K, (double*)nullptr);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

__global__ void clear_status_kernel(int32_t* status) { *status = 0; }

int launch_clear_status(Plan* p, hipStream_t s) {
    hipLaunchKernelGGL(clear_status_kernel, dim3(1), dim3(1), 0, s, p->d_status);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

int launch_assemble(Plan* p, const double* crds, hipStream_t s) {
    JSSO_REQUIRE(p->on_device, JSSO_EINVAL, "plan not uploaded to the device");
    p->full_valid = false;
    if (p->n_nodes > 0) {
        hipLaunchKernelGGL(diag_factor_kernel, xcd_grid((p->n_nodes + DIAG_NODES - 1) / DIAG_NODES), dim3(256), 0, s,
                           p->n_nodes, p->d_diag, p->d_cptr, p->d_csrc, p->d_fixed, p->d_ke, p->d_Linv, p->d_Minv,
                           p->d_status, crds, p->d_crds);
        JSSO_HIP(hipGetLastError());
    }
    const int64_t n_slots = p->ell_slots / ROWS_PER_WG - 1;   // value slots, without the zero slot
    if (n_slots > 0) {
        hipLaunchKernelGGL(ell_assemble_kernel, dim3((unsigned)n_slots), dim3(ASM_WG), 0, s, n_slots, p->d_ell_src,
                           p->d_browof, p->d_colind, p->d_cptr, p->d_csrc, p->d_fixed, p->d_ke, p->d_Linv,
                           p->d_Ke64, p->d_Ke32, (_Float16*)p->d_Ke16, p->n_beam, p->d_status);
        JSSO_HIP(hipGetLastError());
    }
    return JSSO_OK;
}

// y = K x on the full (unconstrained) block-CSR matrix, one thread per scalar row.
__global__ __launch_bounds__(256) void spmv_full_kernel(int32_t n_nodes, const int32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ colind,
                                                        const double* __restrict__ K,
                                                        const double* __restrict__ x, double* __restrict__ y) {
    const int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (R >= 6 * (int64_t)n_nodes) return;
    const int i = (int)(R / 6), r = (int)(R % 6);
    double acc = 0.0;
    for (int k = rowptr[i]; k < rowptr[i + 1]; ++k) {
        const double* b = K + (int64_t)k * 36 + r * 6;
        const double* xj = x + 6 * (int64_t)colind[k];
#pragma unroll
        for (int c = 0; c < 6; ++c) acc += b[c] * xj[c];
    }
    y[R] = acc;
}

// r = f - op(K) u with op(K) = K or K^T (the unconstrained block CSR; u is zero
// at constrained DOFs) and r zero at constrained DOFs; vectors [6 n][nrhs].
// Thread per (scalar row, load case); a row's blocks in column order.
__global__ __launch_bounds__(256) void defect_residual_kernel(int32_t n_nodes, int nrhs,
                                                              const int32_t* __restrict__ rowptr,
                                                              const int32_t* __restrict__ colind,
                                                              const int32_t* __restrict__ tpos,
                                                              const uint8_t* __restrict__ fixed,
                                                              const double* __restrict__ K,
                                                              const double* __restrict__ f,
                                                              const double* __restrict__ u, double* __restrict__ r) {
    const int64_t t = xcd_wg() * blockDim.x + threadIdx.x;
    if (t >= 6 * (int64_t)n_nodes * nrhs) return;
    const int h = (int)(t % nrhs);
    const int64_t R = t / nrhs;
    if (fixed[R]) {
        r[t] = 0.0;
        return;
    }
    const int i = (int)(R / 6), rr = (int)(R % 6);
    double acc = 0.0;
    for (int k = rowptr[i]; k < rowptr[i + 1]; ++k) {
        const int64_t j = colind[k];
        // (K^T)_ij = (K_ji)^T: row rr of it is column rr of the block at the transposed position
        const double* b = tpos ? K + (int64_t)tpos[k] * 36 + rr : K + (int64_t)k * 36 + rr * 6;
        const int st = tpos ? 6 : 1;
#pragma unroll
        for (int c = 0; c < 6; ++c) acc += b[c * st] * u[(6 * j + c) * nrhs + h];
    }
    r[t] = f[t] - acc;
}

__global__ __launch_bounds__(256) void axpy_kernel(int64_t n, const double* __restrict__ x, double* __restrict__ y) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) y[t] += x[t];
}

int launch_defect_residual(Plan* p, const double* K, const double* f, const double* u, int nrhs, bool transpose,
                           double* r, hipStream_t s) {
    JSSO_REQUIRE(p->on_device, JSSO_EINVAL, "plan not uploaded to the device");
    const int64_t n = 6 * (int64_t)p->n_nodes * nrhs;
    if (n == 0) return JSSO_OK;
    hipLaunchKernelGGL(defect_residual_kernel, xcd_grid((n + 255) / 256), dim3(256), 0, s, p->n_nodes, nrhs,
                       p->d_rowptr, p->d_colind, transpose ? (const int32_t*)p->d_tpos : (const int32_t*)nullptr,
                       p->d_fixed, K, f, u, r);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

int launch_axpy(int64_t n, const double* x, double* y, hipStream_t s) {
    if (n <= 0) return JSSO_OK;
    hipLaunchKernelGGL(axpy_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, x, y);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

int launch_spmv_full(Plan* p, const double* K, const double* x, double* y, hipStream_t s) {
    JSSO_REQUIRE(p->on_device, JSSO_EINVAL, "plan not uploaded to the device");
    const int64_t n = 6 * (int64_t)p->n_nodes;
    if (n == 0) return JSSO_OK;
    hipLaunchKernelGGL(spmv_full_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p->n_nodes,
                       p->d_rowptr, p->d_colind, K, x, y);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

}  // namespace jsso
