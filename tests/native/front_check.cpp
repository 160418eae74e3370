// Checks the symbolic analysis of the direct solve (direct_symbolic.hpp) on the
// CPU: for a set of graphs, a multifrontal Cholesky over its fronts (one unknown
// per node) must solve a random SPD matrix of the graph's pattern to the accuracy
// of a dense Cholesky.  Prints one line per graph: name, nodes, fronts, levels,
// largest front, relative difference.  `mistake` 1 drops a border node of one
// front, 2 shifts one relative index (planted errors the check must show).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <string>

#include "../../jaxsso_amd/csrc/direct_symbolic.hpp"

using jsso::FrontTree;
typedef std::vector<std::set<int>> Graph;

static Graph grid(int nx, int ny, bool nine) {
    Graph g(nx * ny);
    for (int y = 0; y < ny; ++y)
        for (int x = 0; x < nx; ++x)
            for (int dy = -1; dy <= 1; ++dy)
                for (int dx = -1; dx <= 1; ++dx) {
                    if (!nine && dx && dy) continue;
                    const int a = x + dx, b = y + dy;
                    if (a >= 0 && b >= 0 && a < nx && b < ny) g[y * nx + x].insert(b * nx + a);
                }
    return g;
}
static Graph edges(int n, const std::vector<std::pair<int, int>>& e) {
    Graph g(n);
    for (int i = 0; i < n; ++i) g[i].insert(i);
    for (auto& p : e) {
        g[p.first].insert(p.second);
        g[p.second].insert(p.first);
    }
    return g;
}
static Graph relabel(const Graph& g, unsigned seed) {
    std::vector<int> p(g.size());
    for (size_t i = 0; i < p.size(); ++i) p[i] = (int)i;
    std::mt19937 rng(seed);
    std::shuffle(p.begin(), p.end(), rng);
    Graph h(g.size());
    for (size_t i = 0; i < g.size(); ++i)
        for (int j : g[i]) h[p[i]].insert(p[j]);
    return h;
}

static int check(const std::string& name, const Graph& g, int leaf, int mistake) {
    const int n = (int)g.size();
    std::vector<int32_t> rp(n + 1, 0), ci;
    for (int i = 0; i < n; ++i) {
        for (int j : g[i]) ci.push_back(j);
        rp[i + 1] = (int32_t)ci.size();
    }
    FrontTree T;
    jsso::build_fronts(n, rp.data(), ci.data(), leaf, T);
    std::mt19937 rng(7);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    std::vector<double> A((size_t)n * n, 0.0), val(ci.size(), 0.0), f(n);
    for (int i = 0; i < n; ++i) {
        f[i] = u(rng);
        for (int k = rp[i]; k < rp[i + 1]; ++k)
            if (ci[k] > i) A[(size_t)i * n + ci[k]] = A[(size_t)ci[k] * n + i] = u(rng);
    }
    for (int i = 0; i < n; ++i) {
        double s = 0.05;
        for (int j = 0; j < n; ++j) s += std::fabs(A[(size_t)i * n + j]);
        A[(size_t)i * n + i] = s;
    }
    // multifrontal elimination: L of every front kept for the two solves
    const int nt = (int)T.fronts.size();
    int max_m = 0, pivots = 0;
    std::vector<std::vector<double>> F(nt);
    std::vector<double> x(f);
    std::vector<std::vector<double>> upd(nt);
    for (int t = 0; t < nt; ++t) {
        const auto& fr = T.fronts[t];
        const int np = fr.np, m = fr.np + fr.nb;
        const int32_t* nd = T.nodes.data() + fr.node0;
        max_m = std::max(max_m, m);
        pivots += np;
        F[t].assign((size_t)m * m, 0.0);
        upd[t].assign(m, 0.0);
        for (int l = 0; l < np; ++l) {
            F[t][(size_t)l * m + l] = A[(size_t)nd[l] * n + nd[l]];
            upd[t][l] = f[nd[l]];
        }
        for (int b = fr.blk0; b < fr.blk0 + fr.nblk; ++b) {
            const int32_t* t3 = &T.blk[3 * (size_t)b];
            const int row = nd[t3[1]], col = nd[t3[2]];
            if (t3[1] <= t3[2] || t3[2] >= np || ci[t3[0]] != row) return 1;
            F[t][(size_t)t3[1] * m + t3[2]] += A[(size_t)row * n + col];
        }
        for (int c = T.child_ptr[t]; c < T.child_ptr[t + 1]; ++c) {
            const auto& ch = T.fronts[T.child[c]];
            const int cm = ch.np + ch.nb;
            if (ch.parent != t || ch.level >= fr.level) return 2;
            for (int i = 0; i < ch.nb; ++i) {
                int ri = T.rel[ch.node0 + ch.np + i];
                if (mistake == 2 && t == nt - 1 && i == 0 && ri + 1 < m) ++ri;
                if (mistake == 1 && t == nt - 1 && i == 0) continue;
                if (ri < 0 || ri >= m || (i && T.rel[ch.node0 + ch.np + i - 1] >= T.rel[ch.node0 + ch.np + i])) return 3;
                upd[t][ri] += upd[T.child[c]][ch.np + i];
                for (int j = 0; j <= i; ++j) {
                    int rj = T.rel[ch.node0 + ch.np + j];
                    if (mistake == 1 && t == nt - 1 && j == 0) continue;
                    F[t][(size_t)ri * m + rj] += F[T.child[c]][(size_t)(ch.np + i) * cm + ch.np + j];
                }
            }
        }
        for (int k = 0; k < np; ++k) {
            const double d = std::sqrt(F[t][(size_t)k * m + k]);
            for (int i = k; i < m; ++i) F[t][(size_t)i * m + k] /= d;
            upd[t][k] /= d;
            for (int i = k + 1; i < m; ++i) {
                upd[t][i] -= F[t][(size_t)i * m + k] * upd[t][k];
                for (int j = k + 1; j <= i; ++j) F[t][(size_t)i * m + j] -= F[t][(size_t)i * m + k] * F[t][(size_t)j * m + k];
            }
        }
    }
    if (pivots != n) return 4;
    for (int t = nt - 1; t >= 0; --t) {
        const auto& fr = T.fronts[t];
        const int np = fr.np, m = fr.np + fr.nb;
        const int32_t* nd = T.nodes.data() + fr.node0;
        for (int k = np - 1; k >= 0; --k) {
            double s = upd[t][k];
            for (int i = k + 1; i < m; ++i) s -= F[t][(size_t)i * m + k] * x[nd[i]];
            x[nd[k]] = s / F[t][(size_t)k * m + k];
        }
    }
    // dense
    std::vector<double> L(A), y(f);
    for (int k = 0; k < n; ++k) {
        const double d = std::sqrt(L[(size_t)k * n + k]);
        for (int i = k; i < n; ++i) L[(size_t)i * n + k] /= d;
        for (int i = k + 1; i < n; ++i)
            for (int j = k + 1; j <= i; ++j) L[(size_t)i * n + j] -= L[(size_t)i * n + k] * L[(size_t)j * n + k];
    }
    for (int k = 0; k < n; ++k) {
        y[k] /= L[(size_t)k * n + k];
        for (int i = k + 1; i < n; ++i) y[i] -= L[(size_t)i * n + k] * y[k];
    }
    for (int k = n - 1; k >= 0; --k) {
        for (int i = k + 1; i < n; ++i) y[k] -= L[(size_t)i * n + k] * y[i];
        y[k] /= L[(size_t)k * n + k];
    }
    double num = 0, den = 0;
    for (int i = 0; i < n; ++i) {
        num += (x[i] - y[i]) * (x[i] - y[i]);
        den += y[i] * y[i];
    }
    std::printf("%s %d %d %d %d %.3e\n", name.c_str(), n, nt, T.n_levels, max_m, std::sqrt(num / den));
    return 0;
}

int main(int argc, char** argv) {
    const int mistake = argc > 1 ? std::atoi(argv[1]) : 0;
    std::vector<std::pair<std::string, Graph>> g;
    g.push_back({"one", edges(1, {})});
    g.push_back({"pair", edges(2, {{0, 1}})});
    g.push_back({"loose", edges(40, {})});                        // no edges at all
    std::vector<std::pair<int, int>> chain, star, clique;
    for (int i = 0; i + 1 < 300; ++i) chain.push_back({i, i + 1});
    for (int i = 1; i < 120; ++i) star.push_back({0, i});
    for (int i = 0; i < 40; ++i)
        for (int j = 0; j < i; ++j) clique.push_back({i, j});
    g.push_back({"chain", edges(300, chain)});
    g.push_back({"star", edges(120, star)});
    g.push_back({"clique", edges(40, clique)});
    g.push_back({"quad_13x13", grid(13, 13, true)});
    g.push_back({"quad_31x8", grid(31, 8, true)});
    g.push_back({"quad_2x200", grid(2, 200, true)});
    g.push_back({"beam_20x17", grid(20, 17, false)});
    g.push_back({"quad_shuffled", relabel(grid(19, 22, true), 3)});
    Graph two = grid(9, 9, true), more = grid(14, 5, false);      // two components in one structure
    for (auto& s : more) {
        std::set<int> t;
        for (int j : s) t.insert(j + 81);
        two.push_back(t);
    }
    g.push_back({"components", two});
    std::mt19937 rng(11);
    std::vector<std::pair<int, int>> rnd;
    for (int i = 0; i < 500; ++i) rnd.push_back({(int)(rng() % 250), (int)(rng() % 250)});
    g.push_back({"random", edges(250, rnd)});
    for (auto& p : g)
        for (int leaf : {1, 12}) {
            const int rc = check(p.first + "_leaf" + std::to_string(leaf), p.second, leaf, mistake);
            if (rc) {
                std::printf("%s failed %d\n", p.first.c_str(), rc);
                return rc;
            }
        }
    return 0;
}
