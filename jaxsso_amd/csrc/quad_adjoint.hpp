// Reverse mode of the MITC-4 element energy phi = lambda_e^T K_e u_e (the element
// term of the reference's VJP through K, JaxSSO/solver.py:221-250, with K_e of
// element.py:880-1084): all 12 coordinate and 5 property derivatives of one load
// case in one pass, one Gauss point at a time.  The GPU runs the four Gauss points
// of an element on four adjacent lanes and adds their partial sums across them
// (adj_quad_kernel); the functions here are what one lane does between those sums.
//
// What makes the reverse pass short:
//   - u and lambda enter a Gauss point only through sums over the nodes: the natural
//     derivatives n0 = sum dN0_a v_a, n1 = sum dN1_a v_a, and the rotations summed
//     over the two nodes of each edge (the tied shear interpolation's terms);
//   - phi = phi(R, xy), and the frame R stays orthonormal as the nodes move, so that
//     only the antisymmetric part of (dphi/dR) R^T acts: three numbers, multiplied by
//     the rotation rates of the frame, which are in closed form.
#pragma once
#include "element_math.hpp"

namespace jsso {

// Keeps the compiler from mixing the instructions of two phases: hoisted together they
// need more registers than a wave has.
JDEV void quad_phase() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// The element's constants: plate cb, cs with their derivatives, and Cm.
struct QuadConsts {
    double cb, cb_t, cb_E, cb_nu, cs, cs_t, cs_E, cs_nu, f, G, t, E, nu, kx, ky;
};

JDEV void quad_consts(double t, double E, double nu, double kx, double ky, QuadConsts& c) {
    c.t = t;
    c.E = E;
    c.nu = nu;
    c.kx = kx;
    c.ky = ky;
    c.f = 1.0 / (1.0 - nu * nu);
    const double i1 = 1.0 / (1.0 + nu), b = t * t * c.f * (1.0 / 12.0), s = (5.0 / 12.0) * i1;
    c.cb_E = t * b;
    c.cb_t = 3.0 * E * b;
    c.cb = E * c.cb_E;
    c.cb_nu = 2.0 * nu * c.f * c.cb;
    c.cs_E = t * s;
    c.cs_t = E * s;
    c.cs = E * c.cs_E;
    c.cs_nu = -c.cs * i1;
    c.G = 0.5 * i1;   // shear modulus over E
}

// Geometry at one Gauss point.  The shear row i of rotation theta_x / theta_y of node a
// has the tied coefficients -yr, -ys / xr, xs: [0] for the nodes of edge 1-2 (r) or 1-4
// (s), [1] for those of edge 4-3 or 2-3 (coefficients of Quad.B_gamma_MITC4,
// element.py:735-801); pr_i, ps_i turn the covariant rows into gamma_i.
struct QuadPoint {
    double r1, r0, s1, s0;             // (1 + r)/4, (1 - r)/4, (1 + s)/4, (1 - s)/4
    double J00, J01, J10, J11, D, iD;  // Jacobian, determinant, its reciprocal
    double in0, in1;                   // 1 / |(J00, J01)|^2, 1 / |(J10, J11)|^2
    double gr, gs;                     // shear factors (quad_gp_rs)
    double pr[2], ps[2];
    double xr[2], yr[2], xs[2], ys[2];
};

// Unit vectors along r and s (quad_gp_rs: (cos, -|sin|) alpha, (cos, |sin|) beta) and the
// reciprocal lengths they were divided by.
struct QuadAxes {
    double ca, ry, rn, cb, sy, sn;
};

JDEV void quad_axes(const double xy[8], QuadAxes& x) {
    const double rx = 0.5 * (xy[0] + xy[6] - xy[2]), ry = 0.5 * (xy[1] + xy[7] - xy[3]);
    const double sx = 0.5 * (xy[0] + xy[2] - xy[6]), sy = 0.5 * (xy[1] + xy[3] - xy[7]);
    x.rn = 1.0 / ::sqrt(rx * rx + ry * ry);
    x.sn = 1.0 / ::sqrt(sx * sx + sy * sy);
    x.ca = rx * x.rn;
    x.ry = ry * x.rn;
    x.cb = sx * x.sn;
    x.sy = sy * x.sn;
}

JDEV void quad_point(const double xy[8], const QuadAxes& x, double r, double s, QuadPoint& P) {
    const double x1 = xy[0], y1 = xy[1], x2 = xy[2], y2 = xy[3], x4 = xy[6], y4 = xy[7];   // node 3: the origin
    P.r1 = 0.25 * (1.0 + r);
    P.r0 = 0.25 * (1.0 - r);
    P.s1 = 0.25 * (1.0 + s);
    P.s0 = 0.25 * (1.0 - s);
    P.xr[0] = P.s1 * (x1 - x2);
    P.yr[0] = P.s1 * (y1 - y2);
    P.xr[1] = P.s0 * x4;
    P.yr[1] = P.s0 * y4;
    P.xs[0] = P.r1 * (x1 - x4);
    P.ys[0] = P.r1 * (y1 - y4);
    P.xs[1] = P.r0 * x2;
    P.ys[1] = P.r0 * y2;
    P.J00 = P.xr[0] + P.xr[1];
    P.J01 = P.yr[0] + P.yr[1];
    P.J10 = P.xs[0] + P.xs[1];
    P.J11 = P.ys[0] + P.ys[1];
    P.D = P.J00 * P.J11 - P.J01 * P.J10;
    P.iD = 1.0 / P.D;
    const double q0 = P.J00 * P.J00 + P.J01 * P.J01, q1 = P.J10 * P.J10 + P.J11 * P.J11;
    P.in0 = 1.0 / q0;
    P.in1 = 1.0 / q1;
    P.gr = 0.5 * ::sqrt(q1) * P.iD;
    P.gs = 0.5 * ::sqrt(q0) * P.iD;
    P.pr[0] = P.gr * fabs(x.sy);
    P.pr[1] = -P.gr * x.cb;
    P.ps[0] = P.gs * fabs(x.ry);
    P.ps[1] = P.gs * x.ca;
}

// Natural derivatives of node a's shape function at the point.
JDEV double quad_dn0(const QuadPoint& P, int a) { return a == 0 ? P.s1 : a == 1 ? -P.s1 : a == 2 ? -P.s0 : P.s0; }
JDEV double quad_dn1(const QuadPoint& P, int a) { return a == 0 ? P.r1 : a == 1 ? P.r0 : a == 2 ? -P.r0 : -P.r1; }

// This point's share of the drilling candidates (quad_rot_diag's entries).
JDEV void quad_point_diag(const QuadPoint& P, const QuadConsts& c, double diag[8]) {
    const double cbD = c.cb * P.D, csD = c.cs * P.D, hn = 0.5 * (1.0 - c.nu);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const double n0 = quad_dn0(P, a), n1 = quad_dn1(P, a);
        const double h0 = (P.J11 * n0 - P.J01 * n1) * P.iD, h1 = (P.J00 * n1 - P.J10 * n0) * P.iD;
        const int ir = a < 2 ? 0 : 1, is = (a == 0 || a == 3) ? 0 : 1;
        const double x0 = P.pr[0] * P.yr[ir] + P.ps[0] * P.ys[is], x1 = P.pr[1] * P.yr[ir] + P.ps[1] * P.ys[is];
        const double y0 = P.pr[0] * P.xr[ir] + P.ps[0] * P.xs[is], y1 = P.pr[1] * P.xr[ir] + P.ps[1] * P.xs[is];
        const double a0 = h0 * h0, a1 = h1 * h1;
        diag[2 * a] = cbD * (a1 + hn * a0) + csD * (x0 * x0 + x1 * x1);
        diag[2 * a + 1] = cbD * (a0 + hn * a1) + csD * (y0 * y0 + y1 * y1);
    }
}

// Drilling stiffness from the summed candidates, and the weight that each candidate's
// change has in phi: the tie-averaged derivative (quad_drill) times the drilling energy ed.
JDEV void quad_drill_weights(const double diag[8], double ed, double& krz, double w[8]) {
    double m = fabs(diag[0]);
#pragma unroll
    for (int i = 1; i < 8; ++i) m = fmin(m, fabs(diag[i]));
    krz = m / 1000.0;
    double cnt = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) cnt += fabs(diag[i]) - m <= TIE_RTOL * m ? 1.0 : 0.0;
    const double each = ed / (1000.0 * cnt);
#pragma unroll
    for (int i = 0; i < 8; ++i)
        w[i] = fabs(diag[i]) - m <= TIE_RTOL * m ? (diag[i] >= 0.0 ? each : -each) : 0.0;
}

// The sums over the nodes through which a field's local values enter a point.
struct QuadSums {
    double n0[6], n1[6];
    double r[2][3], s[2][3];   // rotations summed over edges 1-2, 4-3 (r) and 1-4, 2-3 (s)
};

// Component j of the sums, from its values at the four nodes.
JDEV void quad_sums(const QuadPoint& P, int j, double v0, double v1, double v2, double v3, QuadSums& S) {
    S.n0[j] = P.s1 * (v0 - v1) + P.s0 * (v3 - v2);
    S.n1[j] = P.r1 * (v0 - v3) + P.r0 * (v1 - v2);
    if (j >= 3) {
        S.r[0][j - 3] = v0 + v1;
        S.r[1][j - 3] = v2 + v3;
        S.s[0][j - 3] = v0 + v3;
        S.s[1][j - 3] = v1 + v2;
    }
}

// Strains of one field at a point; S: the tied shear sums that g combines.
struct QuadStrain {
    double mu[3], ku[3], g[2], S[2];
};

JDEV double quad_h0(const QuadPoint& P, const QuadSums& s, int j) { return (P.J11 * s.n0[j] - P.J01 * s.n1[j]) * P.iD; }
JDEV double quad_h1(const QuadPoint& P, const QuadSums& s, int j) { return (P.J00 * s.n1[j] - P.J10 * s.n0[j]) * P.iD; }

JDEV void quad_strain(const QuadPoint& P, const QuadSums& s, QuadStrain& e) {
    e.mu[0] = quad_h0(P, s, 0);
    e.mu[1] = quad_h1(P, s, 1);
    e.mu[2] = quad_h1(P, s, 0) + quad_h0(P, s, 1);
    e.ku[0] = -quad_h0(P, s, 4);
    e.ku[1] = quad_h1(P, s, 3);
    e.ku[2] = quad_h0(P, s, 3) - quad_h1(P, s, 4);
    e.S[0] = 2.0 * s.n0[2] - P.yr[0] * s.r[0][0] - P.yr[1] * s.r[1][0] + P.xr[0] * s.r[0][1] + P.xr[1] * s.r[1][1];
    e.S[1] = 2.0 * s.n1[2] - P.ys[0] * s.s[0][0] - P.ys[1] * s.s[1][0] + P.xs[0] * s.s[0][1] + P.xs[1] * s.s[1][1];
    e.g[0] = P.pr[0] * e.S[0] + P.ps[0] * e.S[1];
    e.g[1] = P.pr[1] * e.S[0] + P.ps[1] * e.S[1];
}

// Bars of the Jacobian and the shear coefficients, gathered over the two fields and the
// drilling candidates.
struct QuadBars {
    double a00, a01, a10, a11;   // sums of dphi/dh0, dphi/dh1 with n0, n1
    double pr[2], ps[2], xr[2], yr[2], xs[2], ys[2];
};

// The drilling candidates' part, with the energies (bending, its nu derivative, shear)
// over D that their weights w stand for.
JDEV void quad_drill_bars(const QuadPoint& P, const QuadConsts& c, const double w[8], QuadBars& b, double en[3]) {
    const double cbD = c.cb * P.D, csD = c.cs * P.D, hn = 0.5 * (1.0 - c.nu);
    double eb = 0.0, ebn = 0.0, es = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const double wx = w[2 * a], wy = w[2 * a + 1];
        const double n0 = quad_dn0(P, a), n1 = quad_dn1(P, a);
        const double h0 = (P.J11 * n0 - P.J01 * n1) * P.iD, h1 = (P.J00 * n1 - P.J10 * n0) * P.iD;
        const double b0 = 2.0 * cbD * h0 * (hn * wx + wy), b1 = 2.0 * cbD * h1 * (wx + hn * wy);
        b.a00 += b0 * n0;
        b.a01 += b0 * n1;
        b.a10 += b1 * n0;
        b.a11 += b1 * n1;
        const double q0 = h0 * h0, q1 = h1 * h1;
        eb += wx * (q1 + hn * q0) + wy * (q0 + hn * q1);
        ebn -= 0.5 * (wx * q0 + wy * q1);
        const int ir = a < 2 ? 0 : 1, is = (a == 0 || a == 3) ? 0 : 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const double x = P.pr[i] * P.yr[ir] + P.ps[i] * P.ys[is], y = P.pr[i] * P.xr[ir] + P.ps[i] * P.xs[is];
            const double ex = 2.0 * csD * wx * x, ey = 2.0 * csD * wy * y;
            es += wx * x * x + wy * y * y;
            b.pr[i] += ex * P.yr[ir] + ey * P.xr[ir];
            b.ps[i] += ex * P.ys[is] + ey * P.xs[is];
            b.yr[ir] += P.pr[i] * ex;
            b.ys[is] += P.ps[i] * ex;
            b.xr[ir] += P.pr[i] * ey;
            b.xs[is] += P.ps[i] * ey;
        }
    }
    en[0] = eb;
    en[1] = ebn;
    en[2] = es;
}

// One field's part: (sm, sk, sg) = dphi / d(its strains).  Adds to the bars and to the
// antisymmetric part (01, 02, 12) of (dphi/dR) R^T.
JDEV void quad_field_bars(const QuadPoint& P, const QuadSums& s, const QuadStrain& e, const double sm[3],
                          const double sk[3], const double sg[2], QuadBars& b, double rot[3]) {
    b.a00 += sm[0] * s.n0[0] + sm[2] * s.n0[1] + sk[2] * s.n0[3] - sk[0] * s.n0[4];
    b.a01 += sm[0] * s.n1[0] + sm[2] * s.n1[1] + sk[2] * s.n1[3] - sk[0] * s.n1[4];
    b.a10 += sm[2] * s.n0[0] + sm[1] * s.n0[1] + sk[1] * s.n0[3] - sk[2] * s.n0[4];
    b.a11 += sm[2] * s.n1[0] + sm[1] * s.n1[1] + sk[1] * s.n1[3] - sk[2] * s.n1[4];
    const double p = P.pr[0] * sg[0] + P.pr[1] * sg[1], q = P.ps[0] * sg[0] + P.ps[1] * sg[1];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        b.pr[i] += sg[i] * e.S[0];
        b.ps[i] += sg[i] * e.S[1];
        b.xr[i] += p * s.r[i][1];
        b.yr[i] -= p * s.r[i][0];
        b.xs[i] += q * s.s[i][1];
        b.ys[i] -= q * s.s[i][0];
    }
    double h0[6], h1[6], X[3], Y[3];   // X, Y: bars of theta_y, theta_x through the shear
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        h0[j] = quad_h0(P, s, j);
        h1[j] = quad_h1(P, s, j);
    }
    const double px0 = p * P.xr[0], px1 = p * P.xr[1], py0 = p * P.yr[0], py1 = p * P.yr[1];
    const double qx0 = q * P.xs[0], qx1 = q * P.xs[1], qy0 = q * P.ys[0], qy1 = q * P.ys[1];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        X[j] = px0 * s.r[0][j] + px1 * s.r[1][j] + qx0 * s.s[0][j] + qx1 * s.s[1][j];
        Y[j] = py0 * s.r[0][j] + py1 * s.r[1][j] + qy0 * s.s[0][j] + qy1 * s.s[1][j];
    }
    rot[0] += sm[0] * h0[1] + sm[2] * h1[1] - sm[1] * h1[0] - sm[2] * h0[0] + sk[1] * h1[4] + sk[2] * h0[4] - Y[1] +
              sk[0] * h0[3] + sk[2] * h1[3] - X[0];
    rot[1] += sm[0] * h0[2] + sm[2] * h1[2] + sk[1] * h1[5] + sk[2] * h0[5] - Y[2] - 2.0 * (p * s.n0[0] + q * s.n1[0]);
    rot[2] += sm[1] * h1[2] + sm[2] * h0[2] - sk[0] * h0[5] - sk[2] * h1[5] + X[2] - 2.0 * (p * s.n0[1] + q * s.n1[1]);
}

// The point's share of dphi by: xy (x1, x2, y2, x4, y4: out[0..4] of quad_point_xy; y1
// stays 0, node 1 lies on the frame's x axis), the frame's antisymmetric part (out[5..7])
// and the properties t, E, nu, kx_mod, ky_mod (out[8..12]).  b, en: from quad_drill_bars;
// sums(0 / 1, s): those of u / lambda, formed twice each so as not to hold them meanwhile.
// Completes the bars and returns the point's energy over D.
template <typename SUMS>
JDEV double quad_point_adjoint(const QuadPoint& P, const QuadConsts& c, const SUMS& sums, QuadBars& b,
                               const double en[3], double out[13]) {
    QuadStrain u, l;
    {
        QuadSums s;
        sums(0, s);
        quad_strain(P, s, u);
        quad_phase();
        sums(1, s);
        quad_strain(P, s, l);
    }
    const double cbD = c.cb * P.D, csD = c.cs * P.D, hn = 0.5 * (1.0 - c.nu);
    // energies over D: membrane products, bending (and its nu derivative), shear
    quad_phase();
    const double A0 = l.mu[0] * u.mu[0], A1 = l.mu[0] * u.mu[1], A2 = l.mu[1] * u.mu[0], A3 = l.mu[1] * u.mu[1];
    const double A4 = l.mu[2] * u.mu[2];
    const double kx2 = l.ku[0] * u.ku[1] + l.ku[1] * u.ku[0], kt = l.ku[2] * u.ku[2];
    const double eb = l.ku[0] * u.ku[0] + l.ku[1] * u.ku[1] + c.nu * kx2 + hn * kt + en[0];
    const double ebn = kx2 - 0.5 * kt + en[1];
    const double es = en[2] + l.g[0] * u.g[0] + l.g[1] * u.g[1];
    const double Ex = c.E * c.kx * c.f, Ey = c.E * c.ky * c.f, GE = c.G * c.E;
    const double fx = A0 + c.nu * A1, fy = c.nu * A2 + A3;
    const double form = Ex * fx + Ey * fy + GE * A4;
    out[8] = P.D * (form + c.cb_t * eb + c.cs_t * es);
    out[9] = P.D * (c.t * (c.f * (c.kx * fx + c.ky * fy) + c.G * A4) + c.cb_E * eb + c.cs_E * es);
    out[10] = P.D * (c.t * (2.0 * c.nu * c.f * (Ex * fx + Ey * fy) + Ex * A1 + Ey * A2 - 2.0 * c.G * GE * A4) +
                     c.cb_nu * eb + c.cb * ebn + c.cs_nu * es);
    out[11] = P.D * c.t * c.E * c.f * fx;
    out[12] = P.D * c.t * c.E * c.f * fy;
    const double W = c.t * form + c.cb * eb + c.cs * es;
    // dphi / d(strains of u), d(strains of lambda)
    const double tD = c.t * P.D, m00 = tD * Ex, m01 = m00 * c.nu, m11 = tD * Ey, m10 = m11 * c.nu, m22 = tD * GE;
    const double smu[3] = {m00 * l.mu[0] + m10 * l.mu[1], m01 * l.mu[0] + m11 * l.mu[1], m22 * l.mu[2]};
    const double sml[3] = {m00 * u.mu[0] + m01 * u.mu[1], m10 * u.mu[0] + m11 * u.mu[1], m22 * u.mu[2]};
    const double sku[3] = {cbD * (l.ku[0] + c.nu * l.ku[1]), cbD * (c.nu * l.ku[0] + l.ku[1]), cbD * hn * l.ku[2]};
    const double skl[3] = {cbD * (u.ku[0] + c.nu * u.ku[1]), cbD * (c.nu * u.ku[0] + u.ku[1]), cbD * hn * u.ku[2]};
    const double sgu[2] = {csD * l.g[0], csD * l.g[1]}, sgl[2] = {csD * u.g[0], csD * u.g[1]};
    double rot[3] = {0.0, 0.0, 0.0};
    quad_phase();
    {
        QuadSums s;
        sums(0, s);
        quad_field_bars(P, s, u, smu, sku, sgu, b, rot);
        quad_phase();
        sums(1, s);
        quad_field_bars(P, s, l, sml, skl, sgl, b, rot);
    }
    out[5] = rot[0];
    out[6] = rot[1];
    out[7] = rot[2];
    return W;
}

// Back through gr, gs, the axes' directions and the Jacobian: out[0..4].
JDEV void quad_point_xy(const QuadPoint& P, const QuadAxes& x, const QuadBars& b, double W, double out[5]) {
    // (the sines: -|x.ry| and |x.sy|)
    const double bgr = fabs(x.sy) * b.pr[0] - x.cb * b.pr[1], bgs = x.ca * b.ps[1] + fabs(x.ry) * b.ps[0];
    const double bsy_ = P.gr * b.pr[0], bcb = -P.gr * b.pr[1], bry_ = P.gs * b.ps[0], bca = P.gs * b.ps[1];
    const double egr = bgr * P.gr, egs = bgs * P.gs;
    const double bD = W - P.iD * (egr + egs + P.iD * (P.J11 * b.a00 - P.J01 * b.a01 + P.J00 * b.a11 - P.J10 * b.a10));
    const double bJ00 = b.a11 * P.iD + egs * P.in0 * P.J00 + bD * P.J11;
    const double bJ01 = -b.a01 * P.iD + egs * P.in0 * P.J01 - bD * P.J10;
    const double bJ10 = -b.a10 * P.iD + egr * P.in1 * P.J10 - bD * P.J01;
    const double bJ11 = b.a00 * P.iD + egr * P.in1 * P.J11 + bD * P.J00;
    // |y| of a unit axis: its derivative is undefined (0/0) where the axis is the frame's x
    const double bry = bry_ * (x.ry / fabs(x.ry)), bsy = bsy_ * (x.sy / fabs(x.sy));
    const double br = bca * x.ca + bry * x.ry, bs = bcb * x.cb + bsy * x.sy;
    const double rx = 0.5 * x.rn * (bca - x.ca * br), ry = 0.5 * x.rn * (bry - x.ry * br);
    const double sx = 0.5 * x.sn * (bcb - x.cb * bs), sy = 0.5 * x.sn * (bsy - x.sy * bs);
    out[0] = P.s1 * (bJ00 + b.xr[0]) + P.r1 * (bJ10 + b.xs[0]) + rx + sx;
    out[1] = -P.s1 * (bJ00 + b.xr[0]) + P.r0 * (bJ10 + b.xs[1]) - rx + sx;
    out[2] = -P.s1 * (bJ01 + b.yr[0]) + P.r0 * (bJ11 + b.ys[1]) - ry + sy;
    out[3] = P.s0 * (bJ00 + b.xr[1]) - P.r1 * (bJ10 + b.xs[0]) + rx - sx;
    out[4] = P.s0 * (bJ01 + b.yr[1]) - P.r1 * (bJ11 + b.ys[0]) + ry - sy;
}

// What the last step needs of the frame: R, xy of nodes 1, 2, 4, the heights z2, z4 of
// nodes 2 and 4 over node 3, and p/q, 1/q, 1/L for v42 = p x + q y, L = |v31|.
struct QuadTurn {
    V3<double> R[3];
    double x1, x2, y2, x4, y4, z2, z4, pq, iq, iL;
};

JDEV void quad_turn(const double c[12], const V3<double> R[3], const double xy[8], QuadTurn& f) {
    const V3<double> v42{c[3] - c[9], c[4] - c[10], c[5] - c[11]};
    const V3<double> v32{c[3] - c[6], c[4] - c[7], c[5] - c[8]}, v34{c[9] - c[6], c[10] - c[7], c[11] - c[8]};
#pragma unroll
    for (int i = 0; i < 3; ++i) f.R[i] = R[i];
    f.x1 = xy[0];
    f.x2 = xy[2];
    f.y2 = xy[3];
    f.x4 = xy[6];
    f.y4 = xy[7];
    f.z2 = dot(v32, R[2]);
    f.z4 = dot(v34, R[2]);
    f.iq = 1.0 / dot(v42, R[1]);
    f.pq = dot(v42, R[0]) * f.iq;
    f.iL = 1.0 / xy[0];
}

// dphi by the position of node a, from the summed out[0..7] of quad_point_adjoint (with
// the drilling term in out[6], out[7]).  The frame turns by alpha = y.dv31 / L about z,
// beta = z.dv31 / L and gamma = -z.(p dv31 - L dv42) / (L q).
JDEV void quad_node_adjoint(const QuadTurn& f, const double o[8], int a, double g[3]) {
    const double A = o[5] + o[1] * f.y2 - o[2] * f.x2 + o[3] * f.y4 - o[4] * f.x4;
    const double B = o[6] + o[1] * f.z2 + o[3] * f.z4, C = o[7] + o[2] * f.z2 + o[4] * f.z4;
    // local components of dphi/dv31, dv32, dv34, dv42
    const double y1 = A * f.iL, z1 = (B - C * f.pq) * f.iL, z42 = C * f.iq;
    double lx, ly, lz;
    if (a == 0) {
        lx = o[0];
        ly = y1;
        lz = z1;
    } else if (a == 1) {
        lx = o[1];
        ly = o[2];
        lz = z42;
    } else if (a == 2) {
        lx = -(o[0] + o[1] + o[3]);
        ly = -(y1 + o[2] + o[4]);
        lz = -z1;
    } else {
        lx = o[3];
        ly = o[4];
        lz = -z42;
    }
    g[0] = lx * f.R[0].x + ly * f.R[1].x + lz * f.R[2].x;
    g[1] = lx * f.R[0].y + ly * f.R[1].y + lz * f.R[2].y;
    g[2] = lx * f.R[0].z + ly * f.R[1].z + lz * f.R[2].z;
}

}  // namespace jsso
