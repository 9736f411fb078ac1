// Host-side analysis of the nested-dissection direct solver: elimination
// tree, fronts, index maps and launch lists of a set of independent systems
// (the diagonal blocks of one BSR matrix).
#pragma once
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <functional>
#include <new>
#include <stdexcept>
#include <thread>
#include <utility>
#include <vector>

namespace nd {

constexpr int NF = 32;    // panel width (DOFs)
constexpr int RB = 128;   // rows below the diagonal block per workgroup
constexpr int TS = 64;    // update tile
constexpr double MAX_SIDE = 0.7;  // largest share of a part on one side of a cut
// cost of a cut above which the numbering is halved as well: about the nodes in
// the widest half-bandwidth that the direct solvers take (576 DOF)
constexpr double NARROW = 96.;

// column length of a panel (n rows and the right-hand side's) and of an
// update matrix: whole 128-byte lines
constexpr int32_t LINE = 16;
constexpr int32_t column(int32_t rows) { return (rows + LINE - 1) / LINE * LINE; }

// One front: k own DOFs (eliminated here) and m boundary DOFs.  Its panel
// is k columns of k + m + 1 rows (column-major) at loff, the last row the
// right-hand side; its update matrix, m columns of m + 1 rows, at uoff of
// the buffer of its depth's parity; its diagonal blocks at doff, NF x NF per
// panel.  noff: its own-then-boundary node list in `nodes` and
// `cmap`.  woff: its boundary part of a right-hand side.  c0, c1: its
// children (-1: none).
struct Front {
    int64_t loff, uoff, doff, noff, woff;
    int32_t own0, k, m, c0, c1, depth;
};

struct Task {
    int32_t front, part;
};

struct Level {
    int64_t front0, front1;
    std::vector<std::pair<int64_t, int64_t>> panels;  // task range of each panel
    int64_t upd0, upd1;                                 // update tiles
};

struct Plan {
    int64_t n_nodes = 0, nnzb = 0;
    std::vector<Front> fronts;
    std::vector<int32_t> nodes;   // permuted node of each front's list
    std::vector<int32_t> cmap;    // 2 per list entry: boundary position in child 0, 1 or -1
    std::vector<int32_t> pnode;   // original node of each permuted one
    std::vector<int64_t> dest;    // panel offset of each BSR block, -1: the upper one of its pair
    std::vector<int32_t> ld;      // its panel's column length, negative: the block goes in transposed
    std::vector<int64_t> rdest;   // right-hand side entry of each permuted node's first column
    std::vector<int32_t> rld;
    std::vector<Task> tasks;
    std::vector<Level> levels;    // deepest first
    int64_t l_size = 0, d_size = 0, u_size[2] = {0, 0}, w_size = 0;
    int32_t widest = 0;           // rows of the largest front
    double flops = 0.;
};

// ------------------------------------------------------------------- tree
struct TreeNode {
    std::vector<int32_t> own;
    int kid[2] = {-1, -1};
    int depth = 0;
};

class Dissection {
  public:
    Dissection(const int32_t *rp, const int32_t *ci, const int32_t *coord, int64_t n0, int64_t n1,
               int leaf)
        : rp_(rp), ci_(ci), xy_(coord), n0_(n0), leaf_(leaf), in_(n1 - n0, 0), lev_(n1 - n0, 0)
    {
        std::vector<int32_t> all(n1 - n0);
        for (size_t i = 0; i < all.size(); i++) all[i] = (int32_t)(n0 + i);
        if (all.empty()) return;
        if (xy_) {
            grow(std::move(all));
            return;
        }
        for (auto &part : parts(all)) {
            std::sort(part.begin(), part.end());  // (the tree it has alone)
            grow(std::move(part));
        }
    }
    std::vector<TreeNode> tree;
    std::vector<int> roots;  // one for each connected part

  private:
    const int32_t *rp_, *ci_, *xy_;
    int64_t n0_;
    int leaf_, stamp_ = 0;
    std::vector<int32_t> in_, lev_;

    int32_t &in(int32_t v) { return in_[v - n0_]; }
    int32_t &lev(int32_t v) { return lev_[v - n0_]; }

    int add(std::vector<int32_t> own, int depth)
    {
        TreeNode t;
        t.own = std::move(own);
        t.depth = depth;
        tree.push_back(std::move(t));
        return (int)tree.size() - 1;
    }

    // breadth-first levels (into lev) of the stamped vertices reachable from
    // `from`; returns them in visiting order
    std::vector<int32_t> bfs(const std::vector<int32_t> &from, size_t size)
    {
        std::vector<int32_t> q;
        q.reserve(size);
        const int seen = ++stamp_;
        for (int32_t v : from) {
            in(v) = seen;
            lev(v) = 0;
            q.push_back(v);
        }
        for (size_t h = 0; h < q.size(); h++) {
            const int32_t v = q[h];
            for (int p = rp_[v]; p < rp_[v + 1]; p++) {
                const int32_t w = ci_[p];
                if (in(w) == seen - 1) {
                    in(w) = seen;
                    lev(w) = lev(v) + 1;
                    q.push_back(w);
                }
            }
        }
        return q;
    }

    static std::vector<int32_t> last_level(const std::vector<int32_t> &q,
                                           const std::vector<int32_t> &lev, int64_t n0)
    {
        size_t h = q.size();
        while (h > 0 && lev[q[h - 1] - n0] == lev[q.back() - n0]) h--;
        return std::vector<int32_t>(q.begin() + h, q.end());
    }

    int32_t least_degree(const std::vector<int32_t> &s) const
    {
        int32_t b = s[0];
        for (int32_t v : s)
            if (rp_[v + 1] - rp_[v] < rp_[b + 1] - rp_[b]) b = v;
        return b;
    }

    // cost of a separator of s vertices that leaves at most `side` of n on one
    // side: its size, raised where that is much the larger, above that of every
    // other cut where it is more than MAX_SIDE: a tree of slivers is as deep
    // as the part is long (1,000 levels for a comb of 1,000 teeth)
    static double cut_cost(size_t n, size_t s, size_t side)
    {
        const double big = (double)side / (double)n;
        return (double)s * (1. + 8. * std::max(0., big - 0.55)) + (big > MAX_SIDE ? (double)n : 0.);
    }

    // the same of the level q[c.first .. c.second), none if it is empty
    static double cut_cost(size_t n, std::pair<size_t, size_t> c)
    {
        return c.second <= c.first ? 1e300
                                   : cut_cost(n, c.second - c.first, std::max(c.first, n - c.second));
    }

    // the cheapest inner level of q (in level order): its [begin, end), or
    // an empty range
    std::pair<size_t, size_t> cut(const std::vector<int32_t> &q) const
    {
        const size_t n = q.size();
        std::pair<size_t, size_t> best{0, 0};
        for (size_t a = 0; a < n;) {
            size_t b = a;
            while (b < n && lev_[q[b] - n0_] == lev_[q[a] - n0_]) b++;
            if (a > 0 && b < n && cut_cost(n, {a, b}) < cut_cost(n, best)) best = {a, b};
            a = b;
        }
        return best;
    }

    // the connected parts of V (V itself if there is one)
    std::vector<std::vector<int32_t>> parts(const std::vector<int32_t> &V)
    {
        const int todo = ++stamp_, done = ++stamp_;
        for (int32_t v : V) in(v) = todo;
        std::vector<std::vector<int32_t>> out;
        for (int32_t v : V) {
            if (in(v) != todo) continue;
            std::vector<int32_t> q{v};
            in(v) = done;
            for (size_t h = 0; h < q.size(); h++)
                for (int p = rp_[q[h]]; p < rp_[q[h] + 1]; p++)
                    if (in(ci_[p]) == todo) {
                        in(ci_[p]) = done;
                        q.push_back(ci_[p]);
                    }
            out.push_back(q.size() == V.size() ? V : std::move(q));
        }
        return out;
    }

    // the tree of V, its root at depth 0 (a list of parts to divide: the tree
    // may be deeper than a thread's stack)
    void grow(std::vector<int32_t> V)
    {
        struct Part {
            std::vector<int32_t> v;
            int parent, side, depth;
        };
        std::vector<Part> todo;
        todo.push_back({std::move(V), -1, 0, 0});
        while (!todo.empty()) {
            Part p = std::move(todo.back());
            todo.pop_back();
            std::vector<int32_t> S, A, B;
            const bool cut = (int)p.v.size() > leaf_ &&
                             (xy_ ? by_coordinates(p.v, S, A, B) : by_levels(p.v, S, A, B));
            const int t = add(std::move(cut ? S : p.v), p.depth);
            if (p.parent < 0) roots.push_back(t);
            else tree[p.parent].kid[p.side] = t;
            if (!cut) continue;
            if (!B.empty()) todo.push_back({std::move(B), t, 1, p.depth + 1});
            if (!A.empty()) todo.push_back({std::move(A), t, 0, p.depth + 1});
        }
    }

    // the middle line of the longer direction of a structured grid; vertices
    // that would couple the two sides join the separator
    bool by_coordinates(const std::vector<int32_t> &V, std::vector<int32_t> &S,
                        std::vector<int32_t> &A, std::vector<int32_t> &B)
    {
        int32_t lo[2] = {INT32_MAX, INT32_MAX}, hi[2] = {INT32_MIN, INT32_MIN};
        for (int32_t v : V)
            for (int d = 0; d < 2; d++) {
                lo[d] = std::min(lo[d], xy_[2 * v + d]);
                hi[d] = std::max(hi[d], xy_[2 * v + d]);
            }
        const int d = hi[0] - lo[0] >= hi[1] - lo[1] ? 0 : 1;
        if (hi[d] - lo[d] < 2) return false;
        const int32_t mid = lo[d] + (hi[d] - lo[d]) / 2;
        const int right = ++stamp_;
        for (int32_t v : V)
            if (xy_[2 * v + d] > mid) in(v) = right;
        for (int32_t v : V) {
            const int32_t c = xy_[2 * v + d];
            bool sep = c == mid;
            if (c < mid)
                for (int p = rp_[v]; p < rp_[v + 1] && !sep; p++) sep = in(ci_[p]) == right;
            (sep ? S : c < mid ? A : B).push_back(v);
        }
        return !A.empty() && !B.empty();
    }

    // A level of a breadth-first search is a separator.  Several searches are
    // tried: from the far side of a search, and from what two far sides have
    // in common (on a square grid the far side of a corner is two edges; the
    // common one gives straight levels).  The cheapest level may still be a
    // short diagonal one, within MAX_SIDE.
    bool by_levels(const std::vector<int32_t> &V, std::vector<int32_t> &S,
                   std::vector<int32_t> &A, std::vector<int32_t> &B)
    {
        auto stamp = [&]() {
            ++stamp_;
            for (int32_t v : V) in(v) = stamp_;
        };
        const size_t n = V.size();
        stamp();
        std::vector<int32_t> q = bfs({V[0]}, n);
        if (q.size() < n) {
            // not connected: the parts go to the two sides, a part of more
            // than half of V is cut as well
            auto some = parts(V);
            std::stable_sort(some.begin(), some.end(),
                             [](auto &x, auto &y) { return x.size() > y.size(); });
            const bool cut = 2 * some[0].size() > n && (int)some[0].size() > leaf_ &&
                             by_levels(some[0], S, A, B);
            for (size_t i = cut; i < some.size(); i++) {
                auto &to = A.size() <= B.size() ? A : B;
                to.insert(to.end(), some[i].begin(), some[i].end());
            }
            return true;
        }
        const int32_t a = least_degree(last_level(q, lev_, n0_));
        stamp();
        q = bfs({a}, n);
        const std::vector<int32_t> La = last_level(q, lev_, n0_);
        std::vector<std::vector<int32_t>> roots{La};
        // corners of the far side: its least-degree vertices, two of them far apart
        std::vector<int32_t> ends{least_degree(La)};
        stamp();
        q = bfs({ends[0]}, n);
        std::vector<int32_t> Lb = last_level(q, lev_, n0_);
        {
            const int dmin = rp_[ends[0] + 1] - rp_[ends[0]];
            int32_t far = -1;
            for (int32_t v : La)
                if (rp_[v + 1] - rp_[v] == dmin && (far < 0 || lev(v) > lev(far))) far = v;
            if (far >= 0 && far != ends[0]) ends.push_back(far);
        }
        for (size_t e = 0; e < ends.size(); e++) {
            if (e) {
                stamp();
                q = bfs({ends[e]}, n);
                Lb = last_level(q, lev_, n0_);
            }
            roots.push_back(Lb);
            const int mark = ++stamp_;
            for (int32_t v : La) in(v) = mark;
            std::vector<int32_t> both;
            for (int32_t v : Lb)
                if (in(v) == mark) both.push_back(v);
            if (both.size() > 1) roots.push_back(both);
        }
        double best = 1e300;
        std::vector<int32_t> bq;
        std::pair<size_t, size_t> bc{0, 0};
        for (const auto &r : roots) {
            stamp();
            q = bfs(r, n);
            const auto c = cut(q);
            const double cost = cut_cost(n, c);
            if (cost < best) {
                best = cost;
                bq = q;
                bc = c;
            }
        }
        if (best > NARROW && by_index(V, best, S, A, B)) return true;
        if (best >= 1e300) return false;
        A.assign(bq.begin(), bq.begin() + bc.first);
        S.assign(bq.begin() + bc.first, bq.begin() + bc.second);
        B.assign(bq.begin() + bc.second, bq.end());
        return true;
    }

    // the given numbering halved, where that costs less: its separator is no
    // larger than the half-bandwidth, which a level can exceed many times
    // (branches that end at the same distance)
    bool by_index(const std::vector<int32_t> &V, double best, std::vector<int32_t> &S,
                  std::vector<int32_t> &A, std::vector<int32_t> &B)
    {
        const size_t n = V.size();
        std::vector<int32_t> order(V);
        std::nth_element(order.begin(), order.begin() + n / 2, order.end());
        const int32_t mid = order[n / 2];
        const int right = ++stamp_;
        for (int32_t v : V)
            if (v >= mid) in(v) = right;
        std::vector<int32_t> sep, left;
        for (int32_t v : V) {
            if (v >= mid) continue;
            bool touches = false;
            for (int p = rp_[v]; p < rp_[v + 1] && !touches; p++) touches = in(ci_[p]) == right;
            (touches ? sep : left).push_back(v);
        }
        if (left.empty() || cut_cost(n, sep.size(), std::max(left.size(), n - n / 2)) >= best)
            return false;
        for (int32_t v : V)
            if (v >= mid) B.push_back(v);
        S = std::move(sep);
        A = std::move(left);
        return true;
    }
};

// --------------------------------------------------------------- analysis
struct SystemFronts {
    struct F {
        int32_t own0, nown, depth;
        int c0, c1;
        std::vector<int32_t> bnd;  // permuted nodes, ascending
    };
    std::vector<F> f;            // children before parents
    std::vector<int32_t> order;  // original node of each permuted one (from the system's first)
};

inline SystemFronts analyse_system(const int32_t *rp, const int32_t *ci, const int32_t *coord,
                                   int64_t n0, int64_t n1, int leaf)
{
    Dissection D(rp, ci, coord, n0, n1, leaf);
    SystemFronts out;
    // post-order: children, then their separator (the reverse of a walk that
    // takes a separator, then its second child's part, then its first's)
    std::vector<int> post, at(D.tree.size(), -1), todo(D.roots);
    while (!todo.empty()) {
        const int t = todo.back();
        todo.pop_back();
        post.push_back(t);
        for (int c : D.tree[t].kid)
            if (c >= 0) todo.push_back(c);
    }
    std::reverse(post.begin(), post.end());
    for (size_t i = 0; i < post.size(); i++) at[post[i]] = (int)i;
    std::vector<int32_t> perm(n1 - n0);  // permuted position of each node
    for (int t : post)
        for (int32_t v : D.tree[t].own) {
            perm[v - n0] = (int32_t)(n0 + out.order.size());
            out.order.push_back(v);
        }
    int32_t next = (int32_t)n0;
    for (int t : post) {
        SystemFronts::F f;
        const TreeNode &T = D.tree[t];
        f.own0 = next;
        f.nown = (int32_t)T.own.size();
        f.depth = T.depth;
        f.c0 = T.kid[0] < 0 ? -1 : at[T.kid[0]];
        f.c1 = T.kid[1] < 0 ? -1 : at[T.kid[1]];
        next += f.nown;
        for (int32_t v : T.own)
            for (int p = rp[v]; p < rp[v + 1]; p++) {
                const int32_t w = perm[ci[p] - n0];
                if (w >= next) f.bnd.push_back(w);
            }
        for (int c : {f.c0, f.c1})
            if (c >= 0)
                for (int32_t w : out.f[c].bnd)
                    if (w >= next) f.bnd.push_back(w);
        std::sort(f.bnd.begin(), f.bnd.end());
        f.bnd.erase(std::unique(f.bnd.begin(), f.bnd.end()), f.bnd.end());
        out.f.push_back(std::move(f));
    }
    return out;
}

// is the block (r, c) in the pattern?
inline bool stored(const int32_t *rp, const int32_t *ci, int32_t r, int32_t c)
{
    return std::find(ci + rp[r], ci + rp[r + 1], c) != ci + rp[r + 1];
}

// the pattern with the transposes of its one-sided blocks
inline void symmetric_pattern(int64_t n, const int32_t *rp, const int32_t *ci,
                              std::vector<int32_t> &srp, std::vector<int32_t> &sci)
{
    std::vector<int64_t> at(n + 1, 0);
    for (int64_t r = 0; r < n; r++) {
        at[r + 1] += rp[r + 1] - rp[r];
        for (int b = rp[r]; b < rp[r + 1]; b++) at[ci[b] + 1] += !stored(rp, ci, ci[b], (int32_t)r);
    }
    for (int64_t r = 0; r < n; r++) at[r + 1] += at[r];
    if (at[n] > INT32_MAX) throw std::length_error("pattern");
    srp.assign(at.begin(), at.end());
    sci.resize(at[n]);
    for (int64_t r = 0; r < n; r++)
        for (int b = rp[r]; b < rp[r + 1]; b++) {
            sci[at[r]++] = ci[b];
            if (!stored(rp, ci, ci[b], (int32_t)r)) sci[at[ci[b]]++] = (int32_t)r;
        }
}

inline void build(Plan &P, int64_t n_nodes, const int32_t *rp, const int32_t *ci,
                  const int32_t *coord, int64_t n_sys, const int64_t *node0, int leaf)
{
    P.n_nodes = n_nodes;
    P.nnzb = rp[n_nodes];
    std::vector<SystemFronts> S(n_sys);
    // fn(0 .. count - 1) on up to 8 threads, at least `grain` calls each; an
    // exception in any of them is thrown again here
    auto each = [&](int64_t count, int64_t grain, const std::function<void(int64_t)> &fn) {
        std::atomic<int64_t> at{0};
        std::atomic<bool> failed{false};
        auto work = [&]() {
            try {
                for (int64_t s; (s = at++) < count;) fn(s);
            } catch (...) {
                failed = true;
            }
        };
        const int64_t cpus = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
        const int nt = (int)std::min(cpus, (count + grain - 1) / grain);
        std::vector<std::thread> th;
        for (int t = 1; t < nt; t++) {
            try {
                th.emplace_back(work);
            } catch (...) {
                break;  // fewer threads
            }
        }
        work();
        for (auto &t : th) t.join();
        if (failed) throw std::bad_alloc();
    };
    // the analysis takes a block that is stored on one side of the diagonal
    // only for both
    std::atomic<bool> one_sided{false};
    each(n_sys, 1, [&](int64_t s) {
        for (int64_t r = node0[s]; r < node0[s + 1] && !one_sided; r++)
            for (int b = rp[r]; b < rp[r + 1]; b++)
                if (!stored(rp, ci, ci[b], (int32_t)r)) one_sided = true;
    });
    std::vector<int32_t> srp, sci;
    if (one_sided) symmetric_pattern(n_nodes, rp, ci, srp, sci);
    each(n_sys, 1, [&](int64_t s) {
        S[s] = analyse_system(one_sided ? srp.data() : rp, one_sided ? sci.data() : ci, coord,
                              node0[s], node0[s + 1], leaf);
    });
    // fronts of all systems by depth, deepest first
    int maxd = 0;
    for (auto &s : S)
        for (auto &f : s.f) maxd = std::max(maxd, (int)f.depth);
    std::vector<std::vector<std::pair<int64_t, int>>> by(maxd + 1);
    for (int64_t s = 0; s < n_sys; s++)
        for (size_t i = 0; i < S[s].f.size(); i++) by[S[s].f[i].depth].push_back({s, (int)i});
    std::vector<std::vector<int32_t>> id(n_sys);
    for (int64_t s = 0; s < n_sys; s++) id[s].assign(S[s].f.size(), -1);
    P.pnode.resize(n_nodes);
    for (int64_t s = 0; s < n_sys; s++)
        std::copy(S[s].order.begin(), S[s].order.end(), P.pnode.begin() + node0[s]);
    std::vector<std::pair<int64_t, int>> src;
    for (int d = maxd; d >= 0; d--) {
        Level lv;
        lv.front0 = (int64_t)P.fronts.size();
        int64_t uoff = 0;
        // largest first, so that a launch's long tasks start early
        std::stable_sort(by[d].begin(), by[d].end(), [&](auto &x, auto &y) {
            return S[x.first].f[x.second].bnd.size() > S[y.first].f[y.second].bnd.size();
        });
        for (auto &si : by[d]) {
            const auto &f = S[si.first].f[si.second];
            Front F{};
            F.own0 = f.own0;
            F.k = 6 * f.nown;
            F.m = 6 * (int32_t)f.bnd.size();
            F.depth = d;
            F.c0 = f.c0 < 0 ? -1 : id[si.first][f.c0];
            F.c1 = f.c1 < 0 ? -1 : id[si.first][f.c1];
            const int32_t n = F.k + F.m, np = (F.k + NF - 1) / NF;
            F.loff = P.l_size;
            P.l_size += (int64_t)column(n + 1) * F.k;
            F.doff = P.d_size;
            P.d_size += (int64_t)np * NF * NF;
            F.uoff = uoff;
            uoff += (int64_t)F.m * column(F.m + 1);
            F.woff = P.w_size;
            P.w_size += F.m;
            F.noff = (int64_t)P.nodes.size();
            for (int i = 0; i < f.nown; i++) P.nodes.push_back(f.own0 + i);
            P.nodes.insert(P.nodes.end(), f.bnd.begin(), f.bnd.end());
            P.widest = std::max(P.widest, (int32_t)n);
            const double k = F.k, m = F.m;
            P.flops += k * k * k / 3 + k * k * m + k * m * m;
            id[si.first][si.second] = (int32_t)P.fronts.size();
            P.fronts.push_back(F);
            src.push_back(si);
        }
        P.u_size[d & 1] = std::max(P.u_size[d & 1], uoff);
        lv.front1 = (int64_t)P.fronts.size();
        // launch lists
        int pmax = 0;
        for (int64_t f = lv.front0; f < lv.front1; f++)
            pmax = std::max(pmax, (P.fronts[f].k + NF - 1) / NF);
        for (int p = 0; p < pmax; p++) {
            const int64_t t0 = (int64_t)P.tasks.size();
            for (int64_t f = lv.front0; f < lv.front1; f++) {
                const Front &F = P.fronts[f];
                if (F.k <= p * NF) continue;
                const int below = F.k + F.m + 1 - std::min(F.k, (p + 1) * NF);
                const int parts = (below + RB - 1) / RB;
                for (int q = 0; q < parts; q++) P.tasks.push_back({(int32_t)f, q});
            }
            lv.panels.push_back({t0, (int64_t)P.tasks.size()});
        }
        lv.upd0 = (int64_t)P.tasks.size();
        for (int64_t f = lv.front0; f < lv.front1; f++) {
            const int m = P.fronts[f].m;
            for (int j = 0; j < (m + TS - 1) / TS; j++)
                for (int i = j; i < (m + TS) / TS; i++) P.tasks.push_back({(int32_t)f, (i << 16) | j});
        }
        lv.upd1 = (int64_t)P.tasks.size();
        P.levels.push_back(std::move(lv));
    }
    // positions of each list entry in the children's boundaries
    P.cmap.assign(2 * P.nodes.size(), -1);
    each((int64_t)P.fronts.size(), 2048, [&](int64_t f) {
        const Front &F = P.fronts[f];
        const int32_t *mine = P.nodes.data() + F.noff;
        const int cnt = (F.k + F.m) / 6;
        for (int c = 0; c < 2; c++) {
            const int32_t ch = c ? F.c1 : F.c0;
            if (ch < 0) continue;
            const Front &C = P.fronts[ch];
            const int32_t *b = P.nodes.data() + C.noff + C.k / 6;
            for (int i = 0, j = 0; j < C.m / 6; j++) {
                while (i < cnt && mine[i] < b[j]) i++;
                P.cmap[2 * (F.noff + i) + c] = j;
            }
        }
    });
    // where each BSR block goes: the panel of the earlier of its two nodes
    std::vector<int32_t> perm(n_nodes), owner(n_nodes);
    for (int64_t i = 0; i < n_nodes; i++) perm[P.pnode[i]] = (int32_t)i;
    P.rdest.resize(n_nodes);
    P.rld.resize(n_nodes);
    for (size_t f = 0; f < P.fronts.size(); f++) {
        const Front &F = P.fronts[f];
        const int32_t n = F.k + F.m;
        for (int i = 0; i < F.k / 6; i++) {
            owner[F.own0 + i] = (int32_t)f;
            P.rld[F.own0 + i] = column(n + 1);
            P.rdest[F.own0 + i] = F.loff + (int64_t)6 * i * column(n + 1) + n;
        }
    }
    P.dest.assign(P.nnzb, -1);
    P.ld.assign(P.nnzb, 0);
    each(n_sys, 1, [&](int64_t s) {
        for (int64_t R = node0[s]; R < node0[s + 1]; R++)
            for (int b = rp[R]; b < rp[R + 1]; b++) {
                int32_t p = perm[R], q = perm[ci[b]];
                const bool upper = p < q;
                if (upper) {
                    if (!one_sided || stored(rp, ci, ci[b], (int32_t)R)) continue;
                    std::swap(p, q);
                }
                const Front &F = P.fronts[owner[q]];
                const int32_t *mine = P.nodes.data() + F.noff;
                const int cnt = (F.k + F.m) / 6;
                const int64_t row = std::lower_bound(mine, mine + cnt, p) - mine;
                const int32_t ld = column(F.k + F.m + 1);
                P.ld[b] = upper ? -ld : ld;
                P.dest[b] = F.loff + (int64_t)6 * (q - F.own0) * ld + 6 * row;
            }
    });
}

}  // namespace nd
