// Host check of the quad adjoint's reverse mode (quad_adjoint.hpp, with the sums that
// the GPU forms across four lanes formed in loops here) against forward mode through the
// frame and the element routines, one dual direction at a time.  Prints, over random
// warped, square, orthotropic, thin and large elements, the largest difference of the
// coordinate derivatives (relative to the element's largest) and of each property
// derivative (relative to the energies of u and lambda).  Run by tests/test_adjoint_reverse.py.
#include "quad_adjoint.hpp"
#include <cstdio>
#include <cstdlib>
#include <random>
using namespace jsso;

static int plant = 0;   // mistakes for the check to find

// phi with one dual direction p
static Dual phi(const double crds[12], const double pr[5], const double* u, const double* l, int p) {
    const int nd[4] = {0, 1, 2, 3};
    Dual c[12], m[5];
    for (int k = 0; k < 12; ++k) c[k] = Dual(crds[k], k == p ? 1.0 : 0.0);
    for (int k = 0; k < 5; ++k) m[k] = Dual(pr[k], 12 + k == p ? 1.0 : 0.0);
    V3<Dual> R[3];
    Dual xy[8];
    quad_frame<Dual>(c, R, xy);
    Dual cb, cs, Cm[3][3], diag[8];
    quad_plate_consts<Dual>(m[0], m[1], m[2], cb, cs);
    quad_cm<Dual>(m[1], m[2], m[3], m[4], Cm);
    quad_rot_diag<Dual, Dual>(xy, cb, cs, m[2], diag);
    const Dual krz = quad_drill<Dual>(diag);
    Dual v[2][24];
    for (int f = 0; f < 2; ++f)
        for (int t = 0; t < 24; t += 3) {
            const double* s = (f ? l : u) + 6 * nd[t / 6] + t % 6;
            for (int i = 0; i < 3; ++i) v[f][t + i] = R[i].x * s[0] + R[i].y * s[1] + R[i].z * s[2];
        }
    Dual sum(0.0);
    for (int g = 0; g < 4; ++g) {
        QuadGP<Dual> G;
        quad_gp<Dual>(xy, g, G);
        Dual mu[2][3], ku[2][3], ga[2][2];
        for (int f = 0; f < 2; ++f)
            for (int a = 0; a < 4; ++a) {
                const Dual *w = v[f] + 6 * a, h0 = G.dH[0][a], h1 = G.dH[1][a];
                mu[f][0] = mu[f][0] + h0 * w[0];
                mu[f][1] = mu[f][1] + h1 * w[1];
                mu[f][2] = mu[f][2] + h1 * w[0] + h0 * w[1];
                for (int k = 0; k < 3; ++k) {
                    Dual k0, k1, k2, b0, b1;
                    quad_bkappa_col(G, a, k, k0, k1, k2);
                    quad_bgamma_col(xy, G, 3 * a + k, b0, b1);
                    ku[f][0] = ku[f][0] + k0 * w[2 + k];
                    ku[f][1] = ku[f][1] + k1 * w[2 + k];
                    ku[f][2] = ku[f][2] + k2 * w[2 + k];
                    ga[f][0] = ga[f][0] + b0 * w[2 + k];
                    ga[f][1] = ga[f][1] + b1 * w[2 + k];
                }
            }
        Dual mf(0.0);
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) mf = mf + mu[1][i] * Cm[i][j] * mu[0][j];
        sum = sum + (m[0] * mf + cb_form(cb, m[2], ku[1][0], ku[1][1], ku[1][2], ku[0][0], ku[0][1], ku[0][2]) +
                     cs * (ga[0][0] * ga[1][0] + ga[0][1] * ga[1][1])) * G.detJ;
    }
    for (int a = 0; a < 4; ++a) sum = sum + krz * v[0][6 * a + 5] * v[1][6 * a + 5];
    return sum;
}

static void reverse(const double c[12], const double pr[5], const double* u, const double* l, double out[17]) {
    V3<double> R[3];
    double xy[8], ul[4][6], ll[4][6], diag[8] = {}, ed = 0.0, o[13] = {};
    quad_frame<double>(c, R, xy);
    QuadConsts q;
    quad_consts(pr[0], pr[1], pr[2], pr[3], pr[4], q);
    for (int a = 0; a < 4; ++a) {
        quad_local_vals(R, u, l, 0.0, a, 1, 0, ul[a], ll[a]);
        ed += ul[a][5] * ll[a][5];
    }
    QuadPoint P[4];
    QuadAxes x;
    quad_axes(xy, x);
    for (int g = 0; g < 4; ++g) {
        double d[8];
        quad_point(xy, x, gauss_r(g), gauss_s(g), P[g]);
        quad_point_diag(P[g], q, d);
        for (int i = 0; i < 8; ++i) diag[i] += d[i];
    }
    double krz, w[8];
    quad_drill_weights(diag, ed, krz, w);
    for (int g = 0; g < 4; ++g) {
        double d[13];
        auto sums = [&](int f, QuadSums& t) {
            for (int j = 0; j < 6; ++j) {
                if (f) quad_sums(P[g], j, ll[0][j], ll[1][j], ll[2][j], ll[3][j], t);
                else quad_sums(P[g], j, ul[0][j], ul[1][j], ul[2][j], ul[3][j], t);
            }
        };
        QuadBars b = {};
        double en[3];
        quad_drill_bars(P[g], q, w, b, en);
        const double W = quad_point_adjoint(P[g], q, sums, b, en, d);
        quad_point_xy(P[g], x, b, W, d);
        for (int i = 0; i < 13; ++i) o[i] += d[i];
    }
    if (plant == 1) o[6] = -o[6];
    if (plant != 2)
        for (int a = 0; a < 4; ++a) {
            o[6] -= krz * (ll[a][5] * ul[a][3] + ul[a][5] * ll[a][3]);
            o[7] -= krz * (ll[a][5] * ul[a][4] + ul[a][5] * ll[a][4]);
        }
    QuadTurn f;
    quad_turn(c, R, xy, f);
    for (int a = 0; a < 4; ++a) quad_node_adjoint(f, o, a, out + 3 * a);
    for (int k = 0; k < 5; ++k) out[12 + k] = o[8 + k];
    if (plant == 3) out[14] *= 1.0 + 1e-6;
}

int main(int argc, char** argv) {
    if (argc > 1) plant = atoi(argv[1]);
    std::mt19937_64 rng(11);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    double worst = 0.0;
    for (int trial = 0; trial < 600; ++trial) {
        const double base[4][2] = {{1, 1}, {0, 1}, {0, 0}, {1, 0}};
        const double sc = trial % 5 == 0 ? 40.0 : 0.05 + 0.2 * (trial % 5), ax = trial % 3 == 2 ? 6.0 : 1.0;
        double c[12], u[24], l[24];
        for (int a = 0; a < 4; ++a) {
            c[3 * a] = sc * ax * (base[a][0] + 0.15 * U(rng));
            c[3 * a + 1] = sc * (base[a][1] + 0.15 * U(rng));
            c[3 * a + 2] = sc * (0.2 * U(rng) + (trial % 2 ? 0.0 : 0.8 * base[a][0])) + 3.0;
        }
        if (trial % 7 == 0)   // a perfect square: ties in the drilling minimum
            for (int a = 0; a < 4; ++a) { c[3 * a] = base[a][0]; c[3 * a + 1] = 0.0; c[3 * a + 2] = base[a][1]; }
        const double t = trial % 4 == 1 ? 1e-3 : 0.05 + 0.1 * (U(rng) + 1);
        const double pr[5] = {sc * t, 3e10 * (1 + 0.2 * U(rng)), trial % 11 == 0 ? 0.0 : 0.2 + 0.2 * U(rng), 1.0,
                              trial % 3 == 0 ? 0.4 : 1.0};
        for (auto& v : u) v = 1e-3 * U(rng);
        for (int k = 0; k < 24; ++k) l[k] = trial % 2 ? 1e-3 * U(rng) : 0.5 * u[k];
        double ref[17], got[17], scale = 0.0;
        for (int p = 0; p < 17; ++p) ref[p] = phi(c, pr, u, l, p).d;
        reverse(c, pr, u, l, got);
        for (int p = 0; p < 12; ++p) scale = fmax(scale, fabs(ref[p]));
        // a property's derivative is of the size of the energies over it
        const double en = fabs(phi(c, pr, u, u, -1).v) + fabs(phi(c, pr, l, l, -1).v);
        const double size[5] = {en / pr[0], en / pr[1], en, en, en};
        for (int p = 0; p < 17; ++p) {
            const double e = fabs(ref[p] - got[p]) / (p < 12 ? scale : size[p - 12]);
            if (!(e <= worst)) worst = e;
            if (!(e < 1e-11) && plant == 0)
                printf("trial %d direction %d forward %.16e reverse %.16e rel %.2e\n", trial, p, ref[p], got[p], e);
        }
    }
    printf("worst relative difference %.3e\n", worst);
    return worst < 1e-11 ? 0 : 1;
}
