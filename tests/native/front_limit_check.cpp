// The limit of the symbolic analysis (build_fronts with max_nodes) on the CPU: for quad
// meshes, beam grids, a chain, a star and two components, a limit at the largest front
// gives the same fronts as none, a limit one below gives none.  Then the time that a mesh
// far past its limit takes, over the time of its whole analysis.  Prints one line per
// graph: name, largest front, 1 where all of that holds; last: "ratio", its value.
#include <chrono>
#include <cstdio>
#include <string>

#include "../../jaxsso_amd/csrc/direct_symbolic.hpp"

using jsso::FrontTree;

struct Pattern {
    std::vector<int32_t> rp{0}, ci;
    int n() const { return (int)rp.size() - 1; }
};

static void grid(Pattern& g, int nx, int ny, bool nine) {
    const int base = g.n();
    for (int y = 0; y < ny; ++y)
        for (int x = 0; x < nx; ++x) {
            for (int dy = -1; dy <= 1; ++dy)
                for (int dx = -1; dx <= 1; ++dx) {
                    const int a = x + dx, b = y + dy;
                    if ((nine || !dx || !dy) && a >= 0 && b >= 0 && a < nx && b < ny) g.ci.push_back(base + b * nx + a);
                }
            g.rp.push_back((int32_t)g.ci.size());
        }
}

static void star(Pattern& g, int n) {
    for (int i = 0; i < n; ++i) {
        g.ci.push_back(i);
        if (i) g.ci.push_back(0);
        if (!i)
            for (int j = 1; j < n; ++j) g.ci.push_back(j);
        g.rp.push_back((int32_t)g.ci.size());
    }
}

static bool same(const FrontTree& a, const FrontTree& b) {
    return a.nodes == b.nodes && a.rel == b.rel && a.child == b.child && a.child_ptr == b.child_ptr && a.blk == b.blk &&
           a.blkrow == b.blkrow && a.n_levels == b.n_levels && a.fronts.size() == b.fronts.size();
}

static int check(const char* name, const Pattern& g) {
    FrontTree all, at, below;
    int32_t seen = 0, most = 0;
    bool ok = jsso::build_fronts(g.n(), g.rp.data(), g.ci.data(), 10, all, INT32_MAX, &seen);
    for (auto& f : all.fronts) most = std::max(most, f.np + f.nb);
    ok = ok && seen == most;
    ok = ok && jsso::build_fronts(g.n(), g.rp.data(), g.ci.data(), 10, at, most) && same(all, at);
    ok = ok && !jsso::build_fronts(g.n(), g.rp.data(), g.ci.data(), 10, below, most - 1, &seen) && below.fronts.empty() &&
         seen >= most;
    std::printf("%s %d %d\n", name, most, ok ? 1 : 0);
    return ok ? 0 : 1;
}

int main() {
    int bad = 0;
    for (int nine = 0; nine < 2; ++nine)
        for (auto& s : {std::pair<int, int>{1, 1}, {1, 300}, {3, 4}, {13, 13}, {47, 31}, {90, 70}}) {
            Pattern g;
            grid(g, s.first, s.second, nine);
            bad += check((std::string(nine ? "quads_" : "beams_") + std::to_string(s.first) + "x" + std::to_string(s.second)).c_str(), g);
        }
    Pattern s, two;
    star(s, 120);
    bad += check("star", s);
    grid(two, 9, 9, true);
    grid(two, 14, 5, false);
    bad += check("components", two);
    Pattern big;
    grid(big, 401, 401, true);
    double t[2];
    for (int lim = 0; lim < 2; ++lim) {
        FrontTree T;
        const auto t0 = std::chrono::steady_clock::now();
        if (jsso::build_fronts(big.n(), big.rp.data(), big.ci.data(), 10, T, lim ? 383 : INT32_MAX) == (lim == 1)) ++bad;
        t[lim] = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    }
    std::printf("ratio %.4f\n", t[1] / t[0]);
    return bad;
}
