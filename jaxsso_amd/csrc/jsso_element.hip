// Element stiffness kernels (beam-column, MITC-4) and the adjoint
// kernels.  Element math lives in element_math.hpp.
#include <mutex>

#include "quad_adjoint.hpp"
#include "jsso_internal.hpp"

namespace jsso {

// A wavefront's 64 element blocks (a lane's 6x6 each, consecutive in memory from dst on;
// the first n of them are stored) through LDS in whole lines, a half of each block at a
// time; st: 64 * OUT doubles of the wavefront, free once the workgroup gets here.
constexpr int OUT = 19;   // odd: the lanes' values start in different banks
__device__ __forceinline__ void store_blocks(const double (&out)[6][6], double* st, double* dst, int n) {
    const int wl = threadIdx.x & 63;
    double2* to = (double2*)dst;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 18; ++q) st[wl * OUT + q] = out[3 * half + q / 6][q % 6];
        __syncthreads();
#pragma unroll 3
        for (int i = wl; i < 9 * n; i += 64) {
            const int blk = i / 9, k = i % 9;
            const double* v = st + blk * OUT + 2 * k;
            to[blk * 18 + 9 * half + k] = make_double2(v[0], v[1]);
        }
    }
}

// ---------------------------------------------------------------------------
// Beam-column stiffness: one thread per (element, node pair a, b).
// Ke_ab = blockdiag(D^-1, D^-1) K_loc,ab blockdiag(D, D)  (solve(T,K)@T,
// element.py:130-139); D^-1 = D^T for the orthogonal general branch.
// BLOCKS: output [e][a][b][6x6] (assembly), else row-major 12x12 per element.
// The entries of K_loc are formed once and placed by the signs of their node pair:
// looked up entry by entry (36 switches with their divisions) and stored by lane, 220
// beams took 19 us; this takes 5 us, and 62 us for 228k (256 gridshells, 263 MB), bound
// by its stores.
// ---------------------------------------------------------------------------
template <bool BLOCKS>
__global__ __launch_bounds__(256) void ke_beam_kernel(int32_t n, const double* __restrict__ crds_e,
                                                      const int32_t* __restrict__ cnct,
                                                      const double* __restrict__ crds_nodes,
                                                      const double* __restrict__ props,
                                                      double* __restrict__ ke, int32_t* flags,
                                                      int32_t* status) {
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    const int e = BLOCKS ? min(tid >> 2, n - 1) : tid >> 2;   // (there the wave stores together)
    if (e >= n) return;
    const int a = (tid >> 1) & 1, b = tid & 1;
    double c[6];
    if (cnct) {
        const int n0 = cnct[2 * e], n1 = cnct[2 * e + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            c[k] = crds_nodes[3 * n0 + k];
            c[3 + k] = crds_nodes[3 * n1 + k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 6; ++k) c[k] = crds_e[6 * e + k];
    }
    const double E = props[6 * e + 0], G = props[6 * e + 1], Iy = props[6 * e + 2],
                 Iz = props[6 * e + 3], Jt = props[6 * e + 4], A = props[6 * e + 5];
    double D[3][3], Di[3][3], L;
    const bool special = beam_dircos<double>(c, D, L);
    if (special) {
        inv3(D, Di);
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) Di[i][j] = D[j][i];
    }
    if (flags && a == 0 && b == 0) flags[e] = special ? 1 : 0;
    if (status && special && a == 0 && b == 0) atomicOr(status, STATUS_NONSYM | STATUS_Y_BEAM);
    // K_loc (beam_kloc's entries): axial, torsion; per bending plane the coefficients of
    // w w, w theta, theta theta of one node, theta theta of two
    const double ax = A * E / L, to = G * Jt / L;
    const double z12 = 12.0 * E * Iz / (L * L * L), z6 = 6.0 * E * Iz / (L * L), zr = (a == b ? 4.0 : 2.0) * E * Iz / L;
    const double y12 = 12.0 * E * Iy / (L * L * L), y6 = 6.0 * E * Iy / (L * L), yr = (a == b ? 4.0 : 2.0) * E * Iy / L;
    const bool same = a == b;
    double out[6][6];
#pragma unroll
    for (int pq = 0; pq < 4; ++pq) {
        const int p = pq >> 1, q = pq & 1;  // translation / rotation sub-blocks
        double S[3][3] = {}, tmp[3][3];
        if (p == q) {
            S[0][0] = p ? (same ? to : -to) : (same ? ax : -ax);
            S[1][1] = p ? yr : (same ? z12 : -z12);
            S[2][2] = p ? zr : (same ? y12 : -y12);
        } else {
            const bool first = (p ? b : a) == 0;   // the translation's node
            const double sz = first ? z6 : -z6, sy = first ? -y6 : y6;
            S[1][2] = p ? sy : sz;
            S[2][1] = p ? sz : sy;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                tmp[i][j] = S[i][0] * D[0][j] + S[i][1] * D[1][j] + S[i][2] * D[2][j];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                out[3 * p + i][3 * q + j] = Di[i][0] * tmp[0][j] + Di[i][1] * tmp[1][j] + Di[i][2] * tmp[2][j];
    }
    if (BLOCKS) {
        __shared__ double lds[4][64 * OUT];
        const int b0 = blockIdx.x * 256 + (threadIdx.x & ~63);   // the wave's first block
        store_blocks(out, lds[threadIdx.x >> 6], ke + (int64_t)b0 * 36, min(64, 4 * n - b0));
        return;
    }
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) ke[(int64_t)e * 144 + (6 * a + i) * 12 + 6 * b + j] = out[i][j];
}

// ---------------------------------------------------------------------------
// MITC-4 stiffness: 16 lanes per element (one per node pair), 16 elements per
// 256-thread workgroup.  Lanes 0-3 stage the per-Gauss-point tiles (det J, dH,
// shear B) in LDS, lanes 0-7 the drilling candidates; then every lane forms
// its 6x6 block of T^T (k_m + k_b) T (element.py:1073-1084).
// MODE: QK_BLOCKS output [e][a][b][6x6] (assembly), QK_GLOBAL row-major 24x24
// per element, QK_LOCAL row-major 24x24 of k_m + k_b before the rotation
// (Quad.element_K_quad_local, element.py:1086-1095).  EPW elements per
// workgroup (4, 8 or 16: 64, 128 or 256 threads), chosen per plan by timing on
// the live assembly (tune_ke_quad).  QK_BLOCKS is bound by its stores: a wave's 64
// blocks are one contiguous 18 KB, which go out through LDS in whole lines.  A lane
// storing its own 288 bytes took 79 us for 40k elements (184 MB); this takes 53 us.
// ---------------------------------------------------------------------------
enum { QK_BLOCKS = 0, QK_GLOBAL = 1, QK_LOCAL = 2 };

struct QuadTile {
    double R[9];
    double t, E, nu, kx, ky;
    double detJ[4];
    double dH[4][8];
    double Bg[4][24];
    double diag[8];
};

template <int MODE, int EPW = 16>
__global__ __launch_bounds__(16 * EPW) void ke_quad_kernel(int32_t n, const double* __restrict__ crds_e,
                                                           const int32_t* __restrict__ cnct,
                                                           const double* __restrict__ crds_nodes,
                                                           const double* __restrict__ props,
                                                           double* __restrict__ ke, int32_t* status = nullptr) {
    // one wave's part: the tiles of its four elements, then (QK_BLOCKS) its 64 blocks on
    // their way out, a lane's 36 values an odd stride apart
    constexpr int TILE = sizeof(QuadTile) / sizeof(double);
    constexpr int WAVE_LDS = MODE == QK_BLOCKS ? 64 * OUT : 4 * TILE;
    __shared__ double lds[EPW / 4][WAVE_LDS];
    const int le = threadIdx.x >> 4, lane = threadIdx.x & 15;
    const int e = blockIdx.x * EPW + le;
    const bool valid = e < n;
    QuadTile& T = *(QuadTile*)&lds[le >> 2][(le & 3) * TILE];
    if (valid && lane < 4) {
        double c[12];
        if (cnct) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const int nd = cnct[4 * e + a];
#pragma unroll
                for (int k = 0; k < 3; ++k) c[3 * a + k] = crds_nodes[3 * nd + k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 12; ++k) c[k] = crds_e[12 * e + k];
        }
        V3<double> R[3];
        double xy[8];
        quad_frame<double>(c, R, xy);
        QuadGP<double> G;
        quad_gp<double>(xy, lane, G);
        T.detJ[lane] = G.detJ;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            T.dH[lane][k] = G.dH[0][k];
            T.dH[lane][4 + k] = G.dH[1][k];
        }
#pragma unroll
        for (int k = 0; k < 12; ++k) quad_bgamma_col<double>(xy, G, k, T.Bg[lane][k], T.Bg[lane][12 + k]);
        if (lane == 0) {
            T.R[0] = R[0].x; T.R[1] = R[0].y; T.R[2] = R[0].z;
            T.R[3] = R[1].x; T.R[4] = R[1].y; T.R[5] = R[1].z;
            T.R[6] = R[2].x; T.R[7] = R[2].y; T.R[8] = R[2].z;
            T.t = props[5 * e + 0];
            T.E = props[5 * e + 1];
            T.nu = props[5 * e + 2];
            T.kx = props[5 * e + 3];
            T.ky = props[5 * e + 4];
            // Cm of element.py:852-875 is [[Ex, nu Ex, 0], [nu Ey, Ey, 0], ...]: not
            // symmetric when kx_mod != ky_mod (and nu != 0), so neither is this Ke
            if (status && T.nu != 0.0 && T.kx != T.ky) atomicOr(status, STATUS_NONSYM | STATUS_ORTHO_QUAD);
        }
    }
    __syncthreads();
    if (valid && lane < 8) {
        double cb, cs;
        quad_plate_consts<double>(T.t, T.E, T.nu, cb, cs);
        const int d = (lane / 2) * 3 + 1 + (lane & 1);
        const int a = d / 3, comp = d % 3;
        double acc = 0.0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            double k0 = 0, k1 = 0, k2 = 0;
            if (comp == 1) { k1 = T.dH[g][4 + a]; k2 = T.dH[g][a]; }
            else { k0 = -T.dH[g][a]; k2 = -T.dH[g][4 + a]; }
            const double b0 = T.Bg[g][d], b1 = T.Bg[g][12 + d];
            acc += (cb_form<double>(cb, T.nu, k0, k1, k2, k0, k1, k2) + cs * (b0 * b0 + b1 * b1)) * T.detJ[g];
        }
        T.diag[lane] = acc;
    }
    __syncthreads();
    if (MODE != QK_BLOCKS && !valid) return;   // (there the wave stores together)
    const int a = lane >> 2, b = lane & 3;
    double cb, cs, Cm[3][3];
    quad_plate_consts<double>(T.t, T.E, T.nu, cb, cs);
    quad_cm<double>(T.E, T.nu, T.kx, T.ky, Cm);
    double mem[2][2] = {{0, 0}, {0, 0}}, ben[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll 1
    for (int g = 0; g < 4; ++g) {
        const double dJ = T.detJ[g];
        const double ha0 = T.dH[g][a], ha1 = T.dH[g][4 + a], hb0 = T.dH[g][b], hb1 = T.dH[g][4 + b];
        // membrane columns: u -> (h0, 0, h1), v -> (0, h1, h0)
        const double Ba[2][3] = {{ha0, 0.0, ha1}, {0.0, ha1, ha0}};
        const double Bb[2][3] = {{hb0, 0.0, hb1}, {0.0, hb1, hb0}};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                double s = 0.0;
#pragma unroll
                for (int r = 0; r < 3; ++r)
                    s += Ba[i][r] * (Cm[r][0] * Bb[j][0] + Cm[r][1] * Bb[j][1] + Cm[r][2] * Bb[j][2]);
                mem[i][j] += s * dJ;
            }
        // bending columns w, theta_x, theta_y
        const double Ka[3][3] = {{0, 0, 0}, {0, ha1, ha0}, {-ha0, 0, -ha1}};
        const double Kb[3][3] = {{0, 0, 0}, {0, hb1, hb0}, {-hb0, 0, -hb1}};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const double kb_ = cb_form<double>(cb, T.nu, Ka[i][0], Ka[i][1], Ka[i][2], Kb[j][0], Kb[j][1], Kb[j][2]);
                const double sh_ = cs * (T.Bg[g][3 * a + i] * T.Bg[g][3 * b + j] +
                                         T.Bg[g][12 + 3 * a + i] * T.Bg[g][12 + 3 * b + j]);
                ben[i][j] += (kb_ + sh_) * dJ;
            }
    }
    // local 6x6 block, DOFs [u, v, w, rx, ry, rz]
    double Lb[6][6];
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) Lb[i][j] = 0.0;
    Lb[0][0] = T.t * mem[0][0]; Lb[0][1] = T.t * mem[0][1];
    Lb[1][0] = T.t * mem[1][0]; Lb[1][1] = T.t * mem[1][1];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Lb[2 + i][2 + j] = ben[i][j];
    if (a == b) {
        double m = fabs(T.diag[0]);
#pragma unroll
        for (int i = 1; i < 8; ++i) m = fmin(m, fabs(T.diag[i]));
        Lb[5][5] = m / 1000.0;
    }
    if (MODE == QK_LOCAL) {
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int j = 0; j < 6; ++j) ke[(int64_t)e * 576 + (6 * a + i) * 24 + 6 * b + j] = Lb[i][j];
        return;
    }
    double R[3][3];
#pragma unroll
    for (int i = 0; i < 9; ++i) R[i / 3][i % 3] = T.R[i];
    double out[6][6];
#pragma unroll
    for (int pq = 0; pq < 4; ++pq) {
        const int p = pq >> 1, q = pq & 1;
        double tmp[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                tmp[i][j] = Lb[3 * p + i][3 * q + 0] * R[0][j] + Lb[3 * p + i][3 * q + 1] * R[1][j] +
                            Lb[3 * p + i][3 * q + 2] * R[2][j];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                out[3 * p + i][3 * q + j] = R[0][i] * tmp[0][j] + R[1][i] * tmp[1][j] + R[2][i] * tmp[2][j];
    }
    if (MODE == QK_BLOCKS) {
        const int64_t e0 = (int64_t)blockIdx.x * EPW + (threadIdx.x >> 6) * 4;
        store_blocks(out, lds[le >> 2], ke + e0 * 16 * 36, (int)(n - e0 < 4 ? n - e0 : 4) * 16);
        return;
    }
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) ke[(int64_t)e * 576 + (6 * a + i) * 24 + 6 * b + j] = out[i][j];
}

int launch_ke_beam(int32_t n, const double* crds_e, const int32_t* cnct, const double* crds_nodes,
                   const double* props, double* ke, int32_t* flags, int32_t* status, hipStream_t s) {
    if (n <= 0) return JSSO_OK;
    const int threads = 256;
    const int64_t total = (int64_t)n * 4;
    const int grid = (int)((total + threads - 1) / threads);
    if (cnct)
        hipLaunchKernelGGL(ke_beam_kernel<true>, dim3(grid), dim3(threads), 0, s, n, crds_e, cnct,
                           crds_nodes, props, ke, flags, status);
    else
        hipLaunchKernelGGL(ke_beam_kernel<false>, dim3(grid), dim3(threads), 0, s, n, crds_e, cnct,
                           crds_nodes, props, ke, flags, status);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

int launch_ke_quad(int32_t n, const double* crds_e, const int32_t* cnct, const double* crds_nodes,
                   const double* props, double* ke, hipStream_t s, int epw, int32_t* status) {
    if (n <= 0) return JSSO_OK;
    const int grid = (n + 15) / 16;
    if (cnct) {
        switch (epw) {
            case 4:
                hipLaunchKernelGGL((ke_quad_kernel<QK_BLOCKS, 4>), dim3((n + 3) / 4), dim3(64), 0, s, n, crds_e, cnct,
                                   crds_nodes, props, ke, status);
                break;
            case 8:
                hipLaunchKernelGGL((ke_quad_kernel<QK_BLOCKS, 8>), dim3((n + 7) / 8), dim3(128), 0, s, n, crds_e,
                                   cnct, crds_nodes, props, ke, status);
                break;
            default:
                hipLaunchKernelGGL((ke_quad_kernel<QK_BLOCKS, 16>), dim3(grid), dim3(256), 0, s, n, crds_e, cnct,
                                   crds_nodes, props, ke, status);
        }
    } else
        hipLaunchKernelGGL((ke_quad_kernel<QK_GLOBAL, 16>), dim3(grid), dim3(256), 0, s, n, crds_e, cnct,
                           crds_nodes, props, ke, status);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

// ---------------------------------------------------------------------------
// Element-level parts of the reference's element API, one thread per element.
// ---------------------------------------------------------------------------

// BeamCol.T (12x12 = blockdiag of the direction cosines, element.py:66-105) and
// BeamCol.K_local (element.py:107-128), row-major; either output may be NULL.
__global__ __launch_bounds__(256) void beam_local_kernel(int32_t n, const double* __restrict__ crds,
                                                         const double* __restrict__ props, double* __restrict__ T,
                                                         double* __restrict__ kl) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    double c[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) c[k] = crds[6 * e + k];
    double D[3][3], L;
    beam_dircos<double>(c, D, L);
    if (T) {
        double* t = T + (int64_t)e * 144;
        for (int i = 0; i < 12; ++i)
            for (int j = 0; j < 12; ++j) t[i * 12 + j] = (i / 3 == j / 3) ? D[i % 3][j % 3] : 0.0;
    }
    if (kl) {
        const double E = props[6 * e + 0], G = props[6 * e + 1], Iy = props[6 * e + 2], Iz = props[6 * e + 3],
                     Jt = props[6 * e + 4], A = props[6 * e + 5];
        double* k = kl + (int64_t)e * 144;
        for (int i = 0; i < 12; ++i)
            for (int j = 0; j < 12; ++j) k[i * 12 + j] = beam_kloc<double>(i, j, L, E, G, Iy, Iz, Jt, A);
    }
}

// Quad.loc_crds (in-plane coordinates, the normal of the element's plane and of
// the triangles 1-2-3 and 1-3-4, element.py:488-539) and Quad.T (24x24 =
// blockdiag of the frame, element.py:643-696); each output may be NULL.
__global__ __launch_bounds__(256) void quad_frame_kernel(int32_t n, const double* __restrict__ crds,
                                                         double* __restrict__ xy_out, double* __restrict__ normals,
                                                         double* __restrict__ T) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    double c[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) c[k] = crds[12 * e + k];
    V3<double> R[3];
    double xy[8];
    quad_frame<double>(c, R, xy);
    if (xy_out)
#pragma unroll
        for (int k = 0; k < 8; ++k) xy_out[8 * e + k] = xy[k];
    if (normals) {
        const V3<double> X0{c[0], c[1], c[2]}, X1{c[3], c[4], c[5]}, X2{c[6], c[7], c[8]}, X3{c[9], c[10], c[11]};
        const V3<double> v31 = sub(X0, X2), v32 = sub(X1, X2), v34 = sub(X3, X2);
        V3<double> t1 = cross(v31, v32), t2 = cross(v34, v31);
        t1 = scale(t1, norm(t1));
        t2 = scale(t2, norm(t2));
        const double nv[9] = {R[2].x, R[2].y, R[2].z, t1.x, t1.y, t1.z, t2.x, t2.y, t2.z};
#pragma unroll
        for (int k = 0; k < 9; ++k) normals[9 * e + k] = nv[k];
    }
    if (T) {
        const double D[3][3] = {{R[0].x, R[0].y, R[0].z}, {R[1].x, R[1].y, R[1].z}, {R[2].x, R[2].y, R[2].z}};
        double* t = T + (int64_t)e * 576;
        for (int i = 0; i < 24; ++i)
            for (int j = 0; j < 24; ++j) t[i * 24 + j] = (i / 3 == j / 3) ? D[i % 3][j % 3] : 0.0;
    }
}

// At natural coordinates (r, s): Quad.J (2x2), B_kappa (3x12), B_gamma_MITC4
// (2x12), B_m (3x8) from the in-plane coordinates (element.py:698-818), and the
// constitutive Cb (3x3), Cs (2x2), Cm (3x3) from [t, E, nu, kx_mod, ky_mod]
// (element.py:820-875); row-major, each output may be NULL.
__global__ __launch_bounds__(256) void quad_gauss_kernel(int32_t n, const double* __restrict__ xy_in,
                                                         const double* __restrict__ props, double r, double s,
                                                         double* __restrict__ Jo, double* __restrict__ Bk,
                                                         double* __restrict__ Bg, double* __restrict__ Bm,
                                                         double* __restrict__ Cb, double* __restrict__ Cs,
                                                         double* __restrict__ Cm) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    if (xy_in) {
        double xy[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) xy[k] = xy_in[8 * e + k];
        QuadGP<double> G;
        double Jm[2][2];
        quad_gp_rs<double>(xy, r, s, G, Jm);
        if (Jo)
#pragma unroll
            for (int k = 0; k < 4; ++k) Jo[4 * e + k] = Jm[k / 2][k % 2];
        if (Bk) {
            double* b = Bk + (int64_t)e * 36;
            for (int a = 0; a < 4; ++a)
                for (int c = 0; c < 3; ++c) {
                    double k0, k1, k2;
                    quad_bkappa_col<double>(G, a, c, k0, k1, k2);
                    b[0 * 12 + 3 * a + c] = k0;
                    b[1 * 12 + 3 * a + c] = k1;
                    b[2 * 12 + 3 * a + c] = k2;
                }
        }
        if (Bg) {
            double* b = Bg + (int64_t)e * 24;
            for (int k = 0; k < 12; ++k) quad_bgamma_col<double>(xy, G, k, b[k], b[12 + k]);
        }
        if (Bm) {
            double* b = Bm + (int64_t)e * 24;
            for (int a = 0; a < 4; ++a) {
                b[0 * 8 + 2 * a] = G.dH[0][a];
                b[0 * 8 + 2 * a + 1] = 0.0;
                b[1 * 8 + 2 * a] = 0.0;
                b[1 * 8 + 2 * a + 1] = G.dH[1][a];
                b[2 * 8 + 2 * a] = G.dH[1][a];
                b[2 * 8 + 2 * a + 1] = G.dH[0][a];
            }
        }
    }
    if (props) {
        const double t = props[5 * e + 0], E = props[5 * e + 1], nu = props[5 * e + 2], kx = props[5 * e + 3],
                     ky = props[5 * e + 4];
        double cb, cs, M[3][3];
        quad_plate_consts<double>(t, E, nu, cb, cs);
        if (Cb) {
            const double v[9] = {cb, cb * nu, 0.0, cb * nu, cb, 0.0, 0.0, 0.0, cb * (1.0 - nu) / 2.0};
#pragma unroll
            for (int k = 0; k < 9; ++k) Cb[9 * e + k] = v[k];
        }
        if (Cs) {
            Cs[4 * e + 0] = cs;
            Cs[4 * e + 1] = 0.0;
            Cs[4 * e + 2] = 0.0;
            Cs[4 * e + 3] = cs;
        }
        if (Cm) {
            quad_cm<double>(E, nu, kx, ky, M);
#pragma unroll
            for (int k = 0; k < 9; ++k) Cm[9 * e + k] = M[k / 3][k % 3];
        }
    }
}

// Elements per workgroup of the assembly's MITC-4 kernel, timed on the live
// plan at its first assembly (every variant writes the same element blocks,
// bit for bit): 4, 8 and 16 elements (64, 128, 256 threads) per workgroup.
int tune_ke_quad(Plan* p, const double* crds, const double* props, double* ke, hipStream_t s, int32_t& out) {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    JSSO_HIP(hipEventCreate(&e0));
    JSSO_HIP(hipEventCreate(&e1));
    float best = 0.f;
    int pick = 16;
    for (int epw : {16, 8, 4}) {
        int rc = launch_ke_quad(p->n_quad, nullptr, p->d_cnct_quad, crds, props, ke, s, epw, p->d_status);   // warm
        if (rc) return rc;
        JSSO_HIP(hipEventRecord(e0, s));
        for (int rep = 0; rep < 2; ++rep)
            if ((rc = launch_ke_quad(p->n_quad, nullptr, p->d_cnct_quad, crds, props, ke, s, epw, p->d_status)))
                return rc;
        JSSO_HIP(hipEventRecord(e1, s));
        JSSO_HIP(hipEventSynchronize(e1));
        float ms = 0.f;
        JSSO_HIP(hipEventElapsedTime(&ms, e0, e1));
        if (epw == 16 || ms < best) {
            best = ms;
            pick = epw;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    out = pick;
    return JSSO_OK;
}

int launch_beam_local(int32_t n, const double* crds, const double* props, double* T, double* kl, hipStream_t s) {
    if (n <= 0) return JSSO_OK;
    hipLaunchKernelGGL(beam_local_kernel, dim3((n + 255) / 256), dim3(256), 0, s, n, crds, props, T, kl);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

int launch_quad_local(int32_t n, const double* crds, const double* props, double* xy, double* normals, double* T,
                      double* kl, hipStream_t s) {
    if (n <= 0) return JSSO_OK;
    if (xy || normals || T)
        hipLaunchKernelGGL(quad_frame_kernel, dim3((n + 255) / 256), dim3(256), 0, s, n, crds, xy, normals, T);
    if (kl)
        hipLaunchKernelGGL((ke_quad_kernel<QK_LOCAL, 16>), dim3((n + 15) / 16), dim3(256), 0, s, n, crds,
                           (const int32_t*)nullptr, (const double*)nullptr, props, kl, (int32_t*)nullptr);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

int launch_quad_gauss(int32_t n, const double* xy, const double* props, double r, double s_, double* J, double* Bk,
                      double* Bg, double* Bm, double* Cb, double* Cs, double* Cm, hipStream_t s) {
    if (n <= 0) return JSSO_OK;
    hipLaunchKernelGGL(quad_gauss_kernel, dim3((n + 255) / 256), dim3(256), 0, s, n, xy, props, r, s_, J, Bk, Bg,
                       Bm, Cb, Cs, Cm);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

// ---------------------------------------------------------------------------
// Adjoint of the element energy phi = -lam_e^T K_e u_e.  Beams: in closed form.
// Quads: in reverse mode, a Gauss point per lane.
// Beam directions: 6 coordinates, then E,G,Iy,Iz,J,A.
// Quad directions: 12 coordinates, then t,E,nu,kx_mod,ky_mod.
// gbuf[(elem_dir) * nrhs + rhs] receives dphi/dp (coordinate directions);
// property directions go straight to dprop (layout [e*nprop + k][rhs]).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double load_lam(const double* u, const double* lam, double scale, int64_t i) {
    return lam ? lam[i] : scale * u[i];
}

// Beams: thread per (element, load case), in closed form.  With u' = D u and
// l' = D^-T lam per triple (D^-T = D unless the member is parallel to global Y),
// phi = l'^T k(L, E, ..) u' is a handful of products of differences and sums of the
// local displacements; its derivatives by the properties and L are those products,
// those by D the outer products of the local forces k u', k l' with lam, u, and the
// chain through the direction cosines C = d / L ends in the node coordinates.  Dual
// numbers through all 144 entries of k per direction (12 threads an element) took
// 4.8 ms for 256 gridshells (228k beams) x 4 load cases; this takes 48 us.
__device__ __forceinline__ void beam_force(const double v[12], double a, double t, double z1, double z2, double z3,
                                           double y1, double y2, double y3, double w[12]) {
    const double dz = v[1] - v[7], sz = v[5] + v[11], dy = v[2] - v[8], sy = v[4] + v[10];
    w[0] = a * (v[0] - v[6]);
    w[3] = t * (v[3] - v[9]);
    w[1] = z3 * dz + z2 * sz;
    w[5] = z2 * dz + z1 * (4.0 * v[5] + 2.0 * v[11]);
    w[11] = z2 * dz + z1 * (2.0 * v[5] + 4.0 * v[11]);
    w[2] = y3 * dy - y2 * sy;
    w[4] = y1 * (4.0 * v[4] + 2.0 * v[10]) - y2 * dy;
    w[10] = y1 * (2.0 * v[4] + 4.0 * v[10]) - y2 * dy;
    w[6] = -w[0];
    w[7] = -w[1];
    w[8] = -w[2];
    w[9] = -w[3];
}

__global__ __launch_bounds__(256) void adj_beam_kernel(int32_t n, const int32_t* __restrict__ cnct,
                                                       const double* __restrict__ crds,
                                                       const double* __restrict__ props,
                                                       const double* __restrict__ u,
                                                       const double* __restrict__ lam, double lam_scale,
                                                       int nrhs, double* __restrict__ gbuf,
                                                       double* __restrict__ dprop) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= (int64_t)n * nrhs) return;
    const int64_t e = tid / nrhs;
    const int rhs = (int)(tid % nrhs);
    const int nd[2] = {cnct[2 * e], cnct[2 * e + 1]};
    double c[6], pr[6], ug[12], lg[12];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        c[k] = crds[3 * (int64_t)nd[0] + k];
        c[3 + k] = crds[3 * (int64_t)nd[1] + k];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) pr[k] = props[6 * e + k];
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        const int64_t gi = ((int64_t)6 * nd[k / 6] + k % 6) * nrhs + rhs;
        ug[k] = u[gi];
        lg[k] = load_lam(u, lam, lam_scale, gi);
    }
    double D[3][3], Dt[3][3], L;
    const bool special = beam_dircos<double>(c, D, L);
    if (special) {
        double Di[3][3];
        inv3(D, Di);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) Dt[i][j] = Di[j][i];
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) Dt[i][j] = D[i][j];
    }
    double ul[12], ll[12];
#pragma unroll
    for (int t = 0; t < 12; t += 3)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            ul[t + i] = D[i][0] * ug[t] + D[i][1] * ug[t + 1] + D[i][2] * ug[t + 2];
            ll[t + i] = Dt[i][0] * lg[t] + Dt[i][1] * lg[t + 1] + Dt[i][2] * lg[t + 2];
        }
    const double E = pr[0], G = pr[1], Iy = pr[2], Iz = pr[3], Jt = pr[4], A = pr[5];
    const double i1 = 1.0 / L, i2 = i1 * i1, i3 = i2 * i1;
    // the bilinear forms of phi: axial, torsion, bending about both axes
    const double X = (ll[0] - ll[6]) * (ul[0] - ul[6]), T = (ll[3] - ll[9]) * (ul[3] - ul[9]);
    const double dzl = ll[1] - ll[7], dzu = ul[1] - ul[7], dyl = ll[2] - ll[8], dyu = ul[2] - ul[8];
    const double z3 = dzl * dzu, z2 = dzl * (ul[5] + ul[11]) + (ll[5] + ll[11]) * dzu;
    const double z1 = 4.0 * (ll[5] * ul[5] + ll[11] * ul[11]) + 2.0 * (ll[5] * ul[11] + ll[11] * ul[5]);
    const double y3 = dyl * dyu, y2 = -(dyl * (ul[4] + ul[10]) + (ll[4] + ll[10]) * dyu);
    const double y1 = 4.0 * (ll[4] * ul[4] + ll[10] * ul[10]) + 2.0 * (ll[4] * ul[10] + ll[10] * ul[4]);
    const double Bz = 12.0 * z3 * i3 + 6.0 * z2 * i2 + z1 * i1, By = 12.0 * y3 * i3 + 6.0 * y2 * i2 + y1 * i1;
    if (dprop) {
        const double g[6] = {A * i1 * X + Iz * Bz + Iy * By, Jt * i1 * T, E * By, E * Bz, G * i1 * T, E * i1 * X};
#pragma unroll
        for (int k = 0; k < 6; ++k) dprop[(6 * e + k) * nrhs + rhs] = -g[k];
    }
    double gd[3];
    if (special) {
        gd[0] = gd[1] = gd[2] = __builtin_nan("");
    } else {
        double fu[12], fl[12];   // local forces: derivatives of phi by l' and by u'
        const double ka = E * A * i1, kt = G * Jt * i1, kz = E * Iz * i1, ky = E * Iy * i1;
        beam_force(ul, ka, kt, kz, 6.0 * kz * i1, 12.0 * kz * i2, ky, 6.0 * ky * i1, 12.0 * ky * i2, fu);
        beam_force(ll, ka, kt, kz, 6.0 * kz * i1, 12.0 * kz * i2, ky, 6.0 * ky * i1, 12.0 * ky * i2, fl);
        double M[3][3] = {};     // dphi / dD
#pragma unroll
        for (int t = 0; t < 12; t += 3)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) M[i][j] += fu[t + i] * lg[t + j] + fl[t + i] * ug[t + j];
        const double Cx = D[0][0], Cy = D[0][1], Cz = D[0][2], h = D[2][1], ih = 1.0 / h;
        const double gh = M[2][1] + (M[1][2] * Cx - M[1][0] * Cz + (M[2][0] * Cx + M[2][2] * Cz) * Cy) * ih * ih;
        double gC[3];
        gC[0] = M[0][0] + (gh * Cx - M[1][2] - M[2][0] * Cy) * ih;
        gC[1] = M[0][1] - (M[2][0] * Cx + M[2][2] * Cz) * ih;
        gC[2] = M[0][2] + (gh * Cz + M[1][0] - M[2][2] * Cy) * ih;
        const double along = gC[0] * Cx + gC[1] * Cy + gC[2] * Cz;
        const double gL = -(E * A * X + G * Jt * T) * i2 -
                          E * (Iz * (36.0 * z3 * i2 + 12.0 * z2 * i1 + z1) + Iy * (36.0 * y3 * i2 + 12.0 * y2 * i1 + y1)) * i2;
#pragma unroll
        for (int k = 0; k < 3; ++k) gd[k] = (gC[k] - along * D[0][k]) * i1 + gL * D[0][k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        gbuf[(e * BDIR + k) * nrhs + rhs] = gd[k];
        gbuf[(e * BDIR + 3 + k) * nrhs + rhs] = -gd[k];
    }
}

// Quads: four lanes per (element, load case).  Lane g loads and rotates node g and
// works Gauss point g in reverse mode (quad_adjoint.hpp); quad permutations add the
// four points' sums, and lane g ends with the derivative by node g and by property g
// (the fifth goes with lane 0).  Bound by FP64 arithmetic, with two waves a SIMD to
// cover its latency: for that the nodes' local values, the frame and the constants
// stay in LDS until a phase reads them (held in registers they allow one wave, and
// 66 us instead of 52).  The four lanes share an element because one lane for all four
// points would leave the chip idle on small plans.  Forward mode in 11 directions,
// each re-reading and re-rotating the nodes at every Gauss point, took 0.73 ms for 16
// shells of 100 x 100 (160k elements); this takes 52 us.
// SELF: lambda = lam_scale u, so phi is lam_scale times the energy of u alone.
__device__ __forceinline__ double quad_lane(double v, int a) {   // a constant after unrolling
    const long long x = __double_as_longlong(v);
    int lo = (int)x, hi = (int)(x >> 32);
    switch (a) {
        case 0: lo = __builtin_amdgcn_mov_dpp(lo, 0x00, 15, 15, true); hi = __builtin_amdgcn_mov_dpp(hi, 0x00, 15, 15, true); break;
        case 1: lo = __builtin_amdgcn_mov_dpp(lo, 0x55, 15, 15, true); hi = __builtin_amdgcn_mov_dpp(hi, 0x55, 15, 15, true); break;
        case 2: lo = __builtin_amdgcn_mov_dpp(lo, 0xAA, 15, 15, true); hi = __builtin_amdgcn_mov_dpp(hi, 0xAA, 15, 15, true); break;
        default: lo = __builtin_amdgcn_mov_dpp(lo, 0xFF, 15, 15, true); hi = __builtin_amdgcn_mov_dpp(hi, 0xFF, 15, 15, true); break;
    }
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double quad_total(double v) {   // sum over the four lanes, the same in each
    long long x = __double_as_longlong(v);
    int lo = __builtin_amdgcn_mov_dpp((int)x, 0xB1, 15, 15, true);          // lanes 1 0 3 2
    int hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), 0xB1, 15, 15, true);
    v += __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
    x = __double_as_longlong(v);
    lo = __builtin_amdgcn_mov_dpp((int)x, 0x4E, 15, 15, true);              // lanes 2 3 0 1
    hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), 0x4E, 15, 15, true);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <bool SELF>
__global__ __launch_bounds__(256, 2) void adj_quad_kernel(int32_t n, int32_t n_beam, const int32_t* __restrict__ cnct,
                                                       const double* __restrict__ crds,
                                                       const double* __restrict__ props,
                                                       const double* __restrict__ u,
                                                       const double* __restrict__ lam, double lam_scale, int nrhs,
                                                       double* __restrict__ gbuf, double* __restrict__ dprop) {
    struct Shared {
        QuadTurn turn;
        QuadConsts q;
        QuadAxes x;
        double v[SELF ? 1 : 2][6][4];   // local values of u, lambda: component, node
        double pad;   // an odd number of doubles apart: a wave's elements start in different banks
    };
    __shared__ Shared shared[64];   // kept here until it is used: it frees 80 registers
    Shared& sh = shared[threadIdx.x >> 2];
    const int64_t item = (xcd_wg() * 256 + threadIdx.x) >> 2;
    if (item >= (int64_t)n * nrhs) return;   // all four lanes of an item, or none
    const int g = threadIdx.x & 3;
    const int64_t e = nrhs == 1 ? item : item / nrhs;
    const int rhs = (int)(item - e * nrhs);
    const int64_t nd = cnct[4 * e + g];
    double own[3], c[12], xy[8], ul[6], ll[6];
    V3<double> R[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) own[k] = crds[3 * nd + k];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int64_t gi = (6 * nd + k) * nrhs + rhs;
        ul[k] = u[gi];
        ll[k] = SELF ? 0.0 : lam[gi];
    }
    const double* pr = props + 5 * e;
    QuadConsts q;
    quad_consts(pr[0], pr[1], pr[2], pr[3], pr[4], q);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int k = 0; k < 3; ++k) c[3 * a + k] = quad_lane(own[k], a);
    quad_frame<double>(c, R, xy);
    {
        QuadTurn f;
        quad_turn(c, R, xy, f);
        sh.turn = f;   // the four lanes write the same
    }
    auto rotate = [&](double v[6]) {
#pragma unroll
        for (int h = 0; h < 6; h += 3) {
            const double x = v[h], y = v[h + 1], z = v[h + 2];
#pragma unroll
            for (int i = 0; i < 3; ++i) v[h + i] = R[i].x * x + R[i].y * y + R[i].z * z;
        }
    };
    rotate(ul);
    if (!SELF) rotate(ll);
    const double(&lv)[6] = SELF ? ul : ll;
    QuadPoint P;
    QuadAxes x;
    quad_axes(xy, x);
    sh.x = x;
    sh.q = q;
    quad_point(xy, x, (g == 0 || g == 3) ? GP : -GP, g < 2 ? GP : -GP, P);   // gauss_r, gauss_s
    quad_phase();
    QuadBars b = {};
    double krz, en[3];
    {
        double diag[8], w[8];
        quad_point_diag(P, q, diag);
#pragma unroll
        for (int i = 0; i < 8; ++i) diag[i] = quad_total(diag[i]);
        quad_drill_weights(diag, quad_total(ul[5] * lv[5]), krz, w);
        quad_phase();
        quad_drill_bars(P, q, w, b, en);
    }
    quad_phase();
    double o[13];
    const double d0 = krz * (lv[5] * ul[3] + ul[5] * lv[3]), d1 = krz * (lv[5] * ul[4] + ul[5] * lv[4]);
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        sh.v[0][j][g] = ul[j];
        if (!SELF) sh.v[1][j][g] = ll[j];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // written by lanes of the same wave
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    auto sums = [&](int f, QuadSums& s) {
        keep_loads_here();
        const double(*v)[4] = sh.v[SELF ? 0 : f];
#pragma unroll
        for (int j = 0; j < 6; ++j) quad_sums(P, j, v[j][0], v[j][1], v[j][2], v[j][3], s);
    };
    keep_loads_here();
    quad_phase();
    const double W = quad_point_adjoint(P, sh.q, sums, b, en, o);
    keep_loads_here();
    quad_phase();
    quad_point_xy(P, sh.x, b, W, o);
    quad_phase();
    o[6] -= d0;   // drilling, the lane's own node
    o[7] -= d1;
#pragma unroll
    for (int i = 0; i < 13; ++i) o[i] = quad_total(o[i]);
    const double sg = SELF ? -lam_scale : -1.0;
    double d[3];
    keep_loads_here();
    const QuadTurn f = sh.turn;
    quad_node_adjoint(f, o, g, d);
    double* out = gbuf + ((int64_t)n_beam * BDIR + e * QDIR + 3 * g) * nrhs + rhs;
#pragma unroll
    for (int k = 0; k < 3; ++k) out[(int64_t)k * nrhs] = sg * d[k];
    if (dprop) {
        double* dp = dprop + 5 * e * nrhs + rhs;
        dp[(int64_t)g * nrhs] = sg * (g == 0 ? o[8] : g == 1 ? o[9] : g == 2 ? o[10] : o[11]);
        if (g == 0) dp[(int64_t)4 * nrhs] = sg * o[12];
    }
}

// node gradient: sum of the coordinate derivatives of the elements incident to
// each node, in a fixed order (no atomics).
__global__ void gather_grad_kernel(int32_t n_nodes, int nrhs, const int32_t* __restrict__ nptr,
                                   const int32_t* __restrict__ nsrc, const double* __restrict__ gbuf,
                                   double* __restrict__ dcrds) {
    const int64_t tid = xcd_wg() * blockDim.x + threadIdx.x;
    if (tid >= (int64_t)n_nodes * 3 * nrhs) return;
    const int rhs = (int)(tid % nrhs);
    const int64_t nc = tid / nrhs;
    const int node = (int)(nc / 3), comp = (int)(nc % 3);
    double s = 0.0;
    for (int k = nptr[node]; k < nptr[node + 1]; ++k) s += gbuf[((int64_t)nsrc[k] + comp) * nrhs + rhs];
    dcrds[tid] = s;
}

int launch_adjoint(Plan* p, const double* crds, const double* prop_beam, const double* prop_quad,
                        const double* u, const double* lam, double lam_scale, int nrhs, double* gbuf,
                        double* dprop_beam, double* dprop_quad, hipStream_t s) {
    JSSO_REQUIRE(p->on_device, JSSO_EINVAL, "plan not uploaded to the device");
    if (p->n_beam > 0) {
        const int64_t total = (int64_t)p->n_beam * nrhs;
        hipLaunchKernelGGL(adj_beam_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                           p->n_beam, p->d_cnct_beam, crds, prop_beam, u, lam, lam_scale, nrhs, gbuf,
                           dprop_beam);
        JSSO_HIP(hipGetLastError());
    }
    if (p->n_quad > 0) {
        const dim3 grid = xcd_grid((4 * (int64_t)p->n_quad * nrhs + 255) / 256);
        if (lam)
            hipLaunchKernelGGL(adj_quad_kernel<false>, grid, dim3(256), 0, s, p->n_quad, p->n_beam, p->d_cnct_quad,
                               crds, prop_quad, u, lam, lam_scale, nrhs, gbuf, dprop_quad);
        else
            hipLaunchKernelGGL(adj_quad_kernel<true>, grid, dim3(256), 0, s, p->n_quad, p->n_beam, p->d_cnct_quad,
                               crds, prop_quad, u, lam, lam_scale, nrhs, gbuf, dprop_quad);
        JSSO_HIP(hipGetLastError());
    }
    return JSSO_OK;
}

// ---------------------------------------------------------------------------
// Fixed gradient scratch for jsso_adjoint_grad_noalloc: a file-scope device
// array (one copy per GPU, held until the process ends), so that callers that
// cannot allocate (graph capture, serving loops) get the adjoint without a
// hipMalloc.  Its device address is looked up once per device with
// hipGetSymbolAddress; host code never passes the array's name itself (that is
// a host-side stand-in, not a device address).  Every call on a GPU shares
// that GPU's array: calls that overlap on one GPU race.
// ---------------------------------------------------------------------------
static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_DOUBLES];

int noalloc_scratch(double** ptr, size_t* bytes) {
    static std::mutex mu;
    static void* dev_ptr[64] = {};
    int dev = -1;
    JSSO_HIP(hipGetDevice(&dev));
    JSSO_REQUIRE(dev >= 0 && dev < 64, JSSO_EINVAL, "device %d out of range", dev);
    std::lock_guard<std::mutex> lock(mu);
    if (!dev_ptr[dev]) {
        void* p = nullptr;
        JSSO_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        JSSO_REQUIRE(p, JSSO_EHIP, "hipGetSymbolAddress gave no address for the adjoint scratch");
        dev_ptr[dev] = p;
    }
    *ptr = (double*)dev_ptr[dev];
    *bytes = sizeof(double) * (size_t)NOALLOC_SCRATCH_DOUBLES;
    return JSSO_OK;
}

int launch_gather_grad(Plan* p, const double* gbuf, int nrhs, double* dcrds, hipStream_t s) {
    JSSO_REQUIRE(p->on_device, JSSO_EINVAL, "plan not uploaded to the device");
    if (!dcrds || p->n_nodes == 0) return JSSO_OK;
    const int64_t total = (int64_t)p->n_nodes * 3 * nrhs;
    hipLaunchKernelGGL(gather_grad_kernel, xcd_grid((total + 255) / 256), dim3(256), 0, s,
                       p->n_nodes, nrhs, p->d_nptr, p->d_nsrc, gbuf, dcrds);
    JSSO_HIP(hipGetLastError());
    return JSSO_OK;
}

}  // namespace jsso
