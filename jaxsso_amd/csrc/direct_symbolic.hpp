// Host-side symbolic analysis of the sparse direct solve (jsso_direct.hip): a
// nested-dissection elimination tree of one connectivity pattern (nodes of 6
// DOFs, 6x6 blocks) and its fronts.  Structures of a plan with the same pattern
// share one analysis.
//
// Dissection.  A set of nodes is cut by a vertex separator that is read off a
// level function f on its nodes: with four mutually distant nodes a, b, c, d
// (farthest-point sampling, nodes of fewest neighbours first, so the corners of
// a mesh region), f = dist(., {a, b}) - dist(., {c, d}) for the three pairings
// and f = dist(., a) - dist(., b); distances are breadth-first in the set.  On
// the quad and beam grids these models are made of two of the pairings have
// straight mesh lines as level sets.  For each f every threshold is tried (the
// separator {f <= t with a neighbour > t}, or its mirror image) and the smallest
// separator, weighed with the balance of the two sides, is taken.
//
// Fronts.  A tree node eliminates its own nodes (pivots); its border is the set
// of later-eliminated nodes that its pivots or its children's borders touch.
// Borders are kept in elimination order, so the map from a child's border into
// the parent's nodes is increasing and a lower triangle maps into a lower
// triangle.
//
// Large sets are cut level by level, before all others, so that a pattern whose fronts
// are past a caller's limit shows at its first few cuts (the others go depth first, while
// their nodes are in the cache): the front that a set ends
// in is its separator and the set's own border, both known once it is cut.  (With a
// limit of 383 nodes, meshes of 300 x 300, 600 x 600 and 1000 x 1000 quads take 23, 65
// and 215 ms on one core; cut to the end, 0.22, 1.0 and 3.1 s.)
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace jsso {

struct FrontTree {
    struct Front {
        int32_t np = 0, nb = 0;       // pivot and border nodes
        int32_t node0 = 0;            // first entry in `nodes`: pivots, then border
        int32_t parent = -1, level = 0;
        int32_t blk0 = 0, nblk = 0;   // stored blocks of K that enter here
    };
    std::vector<Front> fronts;              // children before parents
    std::vector<int32_t> nodes;             // node ids of every front
    std::vector<int32_t> rel;               // per border entry (same offsets as `nodes`): local index in the parent, -1 at pivots
    std::vector<int32_t> child_ptr, child;  // children of every front
    std::vector<int32_t> blk;               // triples: block of the CSR, local row, local column (row > column), by row
    std::vector<int32_t> blkrow;            // per entry of `nodes`: first triple of that local row
    int32_t n_levels = 0;
};

class Dissector {
public:
    Dissector(int32_t n, const int32_t* rowptr, const int32_t* colind, int leaf)
        : n_(n), rp_(rowptr), ci_(colind), leaf_(leaf), part_(n, 0), dist_(4, std::vector<int32_t>(n, -1)), f_(n) {}

    // tree nodes in postorder: own nodes and the subtrees directly below
    struct Node {
        std::vector<int32_t> own;
        std::vector<int32_t> kids;
    };
    std::vector<Node> tree;
    int32_t largest = 0;   // nodes of the largest front seen

    // false (and no tree) as soon as a front has more than max_nodes nodes
    bool run(int32_t max_nodes) {
        std::vector<Set> sets(1);
        sets[0].nodes.resize(n_);
        for (int i = 0; i < n_; ++i) sets[0].nodes[i] = i;
        std::vector<int32_t> large{0}, others;   // sets to come (part_ of a set's nodes: its number)
        for (size_t next = 0; next < large.size() || !others.empty();) {
            int32_t t;
            if (next < large.size()) {
                t = large[next++];
            } else {
                t = others.back();
                others.pop_back();
            }
            std::vector<int32_t> side[2], sep;
            if ((int)sets[t].nodes.size() <= leaf_ || !cut(t, sets[t].nodes, side, sep))
                sep = std::move(sets[t].nodes);
            else
                std::sort(sep.begin(), sep.end());
            largest = std::max(largest, (int32_t)(sep.size() + sets[t].border.size()));
            if (largest > max_nodes) return false;
            for (auto& s : side) {
                if (s.empty()) continue;
                std::sort(s.begin(), s.end());
                const int32_t kid = (int32_t)sets.size();
                for (int v : s) part_[v] = kid;
                ((int64_t)s.size() > 4 * (int64_t)max_nodes ? large : others).push_back(kid);
                Set below;
                below.nodes = std::move(s);
                for (const auto* from : {&sets[t].border, &sep})
                    for (int w : *from)
                        for (int k = rp_[w]; k < rp_[w + 1]; ++k)
                            if (part_[ci_[k]] == kid) {
                                below.border.push_back(w);
                                break;
                            }
                sets[t].node.kids.push_back(kid);
                sets.push_back(std::move(below));
            }
            sets[t].node.own = std::move(sep);
            std::vector<int32_t>().swap(sets[t].nodes);
            std::vector<int32_t>().swap(sets[t].border);
        }
        // postorder
        tree.reserve(sets.size());
        std::vector<std::pair<int32_t, size_t>> path{{0, 0}};
        std::vector<int32_t> at(sets.size());
        while (!path.empty()) {
            const int32_t t = path.back().first;
            auto& node = sets[t].node;
            if (path.back().second < node.kids.size()) {
                path.push_back({node.kids[path.back().second++], 0});
                continue;
            }
            for (auto& k : node.kids) k = at[k];
            at[t] = (int32_t)tree.size();
            tree.push_back(std::move(node));
            path.pop_back();
        }
        return true;
    }

private:
    int32_t n_;
    const int32_t *rp_, *ci_;
    int leaf_;
    std::vector<int32_t> part_;                 // set label of every node
    std::vector<std::vector<int32_t>> dist_;
    std::vector<int32_t> f_, queue_;
    struct Set {
        std::vector<int32_t> nodes, border;   // border: the nodes outside that touch them
        Node node;
    };

    // breadth-first distances inside the set `lab` from `src`; returns the number of nodes reached
    int bfs(int32_t lab, int32_t src, std::vector<int32_t>& d) {
        queue_.clear();
        queue_.push_back(src);
        d[src] = 0;
        for (size_t q = 0; q < queue_.size(); ++q) {
            const int v = queue_[q];
            for (int k = rp_[v]; k < rp_[v + 1]; ++k) {
                const int w = ci_[k];
                if (w != v && part_[w] == lab && d[w] < 0) {
                    d[w] = d[v] + 1;
                    queue_.push_back(w);
                }
            }
        }
        return (int)queue_.size();
    }
    int degree(int32_t lab, int v) const {
        int d = 0;
        for (int k = rp_[v]; k < rp_[v + 1]; ++k) d += ci_[k] != v && part_[ci_[k]] == lab;
        return d;
    }
    // node of `set` with the largest key, fewest neighbours on ties, lowest id then
    template <typename K>
    int32_t farthest(int32_t lab, const std::vector<int32_t>& set, K&& key) const {
        int32_t best = set[0], bk = -1, bd = 0;
        for (int v : set) {
            const int32_t k = key(v);
            if (k < bk) continue;
            const int d = degree(lab, v);
            if (k > bk || d < bd) {
                best = v;
                bk = k;
                bd = d;
            }
        }
        return best;
    }

    // smallest separator over the thresholds of f_ on `set`; cost < 0: none found yet
    struct Cut {
        double cost = -1.0;
        int which = 0, t = 0, mirror = 0;
    };
    void thresholds(int32_t lab, const std::vector<int32_t>& set, int which, Cut& best) {
        int fmin = f_[set[0]], fmax = fmin;
        for (int v : set) {
            fmin = std::min(fmin, f_[v]);
            fmax = std::max(fmax, f_[v]);
        }
        const int m = fmax - fmin + 1;
        if (m < 2) return;
        std::vector<int32_t> le(m + 1, 0), sl(m + 1, 0), sr(m + 1, 0);
        for (int v : set) {
            int mx = f_[v], mn = f_[v];
            for (int k = rp_[v]; k < rp_[v + 1]; ++k) {
                const int w = ci_[k];
                if (part_[w] != lab) continue;
                mx = std::max(mx, f_[w]);
                mn = std::min(mn, f_[w]);
            }
            const int a = f_[v] - fmin;
            ++le[a];
            ++sl[a];              // in the left boundary for t in [f(v), max neighbour)
            --sl[mx - fmin];
            ++sr[mn - fmin];      // in the right boundary for t in [min neighbour, f(v))
            --sr[a];
        }
        const int n = (int)set.size();
        int below = 0, bl = 0, br = 0;
        for (int t = 0; t + 1 < m; ++t) {
            below += le[t];
            bl += sl[t];
            br += sr[t];
            for (int mirror = 0; mirror < 2; ++mirror) {
                const int s = mirror ? br : bl;
                const int left = mirror ? below : below - bl, right = mirror ? n - below - br : n - below;
                if (left <= 0 || right <= 0) continue;
                const double share = (double)std::max(left, right) / (left + right);
                if (share > 0.8) continue;
                const double over = share - 0.5;
                const double cost = s * (1.0 + 2.0 * over + 12.0 * over * over);
                if (best.cost < 0.0 || cost < best.cost) best = Cut{cost, which, t + fmin, mirror};
            }
        }
    }
    void level_function(int which, const std::vector<int32_t>& set) {
        const auto &a = dist_[0], &b = dist_[1], &c = dist_[2], &d = dist_[3];
        for (int v : set) {
            switch (which) {
                case 0: f_[v] = std::min(a[v], b[v]) - std::min(c[v], d[v]); break;
                case 1: f_[v] = std::min(a[v], c[v]) - std::min(b[v], d[v]); break;
                case 2: f_[v] = std::min(a[v], d[v]) - std::min(b[v], c[v]); break;
                case 3: f_[v] = a[v] - b[v]; break;
                default: f_[v] = a[v]; break;
            }
        }
    }

    // cuts a set into two sides and a separator, or into its components without one;
    // false for a clique-like set
    bool cut(int32_t lab, const std::vector<int32_t>& set, std::vector<int32_t> (&side)[2],
             std::vector<int32_t>& sep) {
        for (auto& d : dist_)
            for (int v : set) d[v] = -1;
        auto& tmp = dist_[3];
        const int reached = bfs(lab, set[0], tmp);
        if (reached < (int)set.size()) {   // several components: no separator needed
            std::vector<std::vector<int32_t>> comp;
            for (int v : set) {
                if (dist_[2][v] >= 0) continue;
                bfs(lab, v, dist_[2]);
                comp.push_back(queue_);
                for (int w : queue_) dist_[2][w] = 0;
            }
            std::sort(comp.begin(), comp.end(), [](const auto& x, const auto& y) { return x.size() > y.size(); });
            for (auto& c : comp) {
                auto& s = side[side[0].size() <= side[1].size() ? 0 : 1];
                s.insert(s.end(), c.begin(), c.end());
            }
        } else {
            const int32_t a0 = farthest(lab, set, [&](int v) { return tmp[v]; });
            bfs(lab, a0, dist_[0]);
            const int32_t b0 = farthest(lab, set, [&](int v) { return dist_[0][v]; });
            bfs(lab, b0, dist_[1]);
            const int32_t c0 = farthest(lab, set, [&](int v) { return std::min(dist_[0][v], dist_[1][v]); });
            bfs(lab, c0, dist_[2]);
            for (int v : set) tmp[v] = -1;   // (its first use is over)
            const int32_t e0 = farthest(lab, set, [&](int v) {
                return std::min(dist_[0][v], std::min(dist_[1][v], dist_[2][v]));
            });
            bfs(lab, e0, dist_[3]);
            Cut best;
            for (int w = 0; w < 5; ++w) {
                level_function(w, set);
                thresholds(lab, set, w, best);
            }
            if (best.cost < 0.0) return false;
            level_function(best.which, set);
            for (int v : set) {
                bool in = false;
                for (int k = rp_[v]; k < rp_[v + 1] && !in; ++k) {
                    const int w = ci_[k];
                    if (part_[w] != lab) continue;
                    in = best.mirror ? f_[v] > best.t && f_[w] <= best.t : f_[v] <= best.t && f_[w] > best.t;
                }
                if (in)
                    sep.push_back(v);
                else
                    side[f_[v] <= best.t ? 0 : 1].push_back(v);
            }
        }
        return true;
    }
};

// Fronts of the elimination tree of a pattern (block CSR of n nodes, columns
// local to the structure).  `leaf`: largest set that is eliminated whole.  False (and no
// fronts) where a front has more than max_nodes nodes; *largest: of the fronts seen.
inline bool build_fronts(int32_t n, const int32_t* rowptr, const int32_t* colind, int leaf, FrontTree& out,
                         int32_t max_nodes = INT32_MAX, int32_t* largest = nullptr) {
    Dissector D(n, rowptr, colind, leaf);
    out = FrontTree();
    const bool fits = D.run(max_nodes);
    if (largest) *largest = D.largest;
    if (!fits) return false;
    auto& tree = D.tree;
    const int nt = (int)tree.size();
    std::vector<int32_t> pos(n), owner(n);
    {
        int p = 0;
        for (int t = 0; t < nt; ++t)
            for (int v : tree[t].own) {
                pos[v] = p++;
                owner[v] = t;
            }
    }
    out.fronts.resize(nt);
    std::vector<std::vector<int32_t>> border(nt);
    std::vector<int32_t> mark(n, -1), parent(nt, -1);
    for (int t = 0; t < nt; ++t) {
        auto& b = border[t];
        for (int v : tree[t].own) mark[v] = t;
        for (int v : tree[t].own)
            for (int k = rowptr[v]; k < rowptr[v + 1]; ++k) {
                const int w = colind[k];
                if (mark[w] != t && owner[w] > t) {
                    mark[w] = t;
                    b.push_back(w);
                }
            }
        for (int c : tree[t].kids) {
            parent[c] = t;
            for (int w : border[c])
                if (mark[w] != t) {
                    mark[w] = t;
                    b.push_back(w);
                }
        }
        std::sort(b.begin(), b.end(), [&](int x, int y) { return pos[x] < pos[y]; });
    }
    std::vector<int32_t> local(n, -1), nchild(nt + 1, 0);
    for (int t = 0; t < nt; ++t) {
        auto& F = out.fronts[t];
        F.parent = parent[t];
        F.np = (int32_t)tree[t].own.size();
        F.nb = (int32_t)border[t].size();
        F.node0 = (int32_t)out.nodes.size();
        int lev = 0;
        for (int c : tree[t].kids) lev = std::max(lev, out.fronts[c].level + 1);
        F.level = lev;
        out.n_levels = std::max(out.n_levels, lev + 1);
        out.nodes.insert(out.nodes.end(), tree[t].own.begin(), tree[t].own.end());
        out.nodes.insert(out.nodes.end(), border[t].begin(), border[t].end());
        if (parent[t] >= 0) ++nchild[parent[t] + 1];
    }
    for (int t = 0; t < nt; ++t) nchild[t + 1] += nchild[t];
    out.child_ptr.assign(nchild.begin(), nchild.end());
    out.child.resize(nchild[nt]);
    {
        std::vector<int32_t> fill(nchild.begin(), nchild.end() - 1);
        for (int t = 0; t < nt; ++t)
            if (parent[t] >= 0) out.child[fill[parent[t]]++] = t;
    }
    out.rel.assign(out.nodes.size(), -1);
    for (int t = 0; t < nt; ++t) {
        auto& F = out.fronts[t];
        const int32_t* v = out.nodes.data() + F.node0;
        for (int l = 0; l < F.np + F.nb; ++l) local[v[l]] = l;
        F.blk0 = (int32_t)(out.blk.size() / 3);
        for (int l = 0; l < F.np; ++l)
            for (int k = rowptr[v[l]]; k < rowptr[v[l] + 1]; ++k) {
                const int w = colind[k];
                if (w == v[l] || pos[w] < pos[v[l]]) continue;
                // block (w, v[l]) is the transpose of (v[l], w): the caller reads it through its own map
                out.blk.push_back(k);
                out.blk.push_back(local[w]);
                out.blk.push_back(l);
            }
        F.nblk = (int32_t)(out.blk.size() / 3) - F.blk0;
        struct B3 { int32_t k, r, c; };
        B3* b3 = reinterpret_cast<B3*>(out.blk.data()) + F.blk0;
        std::sort(b3, b3 + F.nblk, [](const B3& x, const B3& y) { return x.r != y.r ? x.r < y.r : x.c < y.c; });
        for (int l = 0, q = 0; l < F.np + F.nb; ++l) {
            while (q < F.nblk && b3[q].r < l) ++q;
            out.blkrow.push_back(F.blk0 + q);
        }
        for (int c = out.child_ptr[t]; c < out.child_ptr[t + 1]; ++c) {
            const auto& G = out.fronts[out.child[c]];
            for (int l = 0; l < G.nb; ++l)
                out.rel[G.node0 + G.np + l] = local[out.nodes[G.node0 + G.np + l]];
        }
    }
    return true;
}

}  // namespace jsso
