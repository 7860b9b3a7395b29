// nd_order.h -- nested-dissection order of a mesh graph and the symbolic
// structure of its multifrontal Cholesky factor (host code, no device calls).
//
// A node set is cut by a vertex separator found along one of four sweeps of
// the set: the three coordinates (shell meshes are surfaces, so a plane cuts
// them in short lines) and the breadth-first distance from a far node (which
// needs no coordinates).  For a sweep the separator of every cut position
// comes from two prefix sums over the edges, so all positions between 30 and
// 70 per cent of the set are compared, not only the median.  The two sides
// are cut again down to leaves of at most `leaf` nodes; a leaf and every
// separator is one front.
#pragma once

#include <algorithm>
#include <atomic>
#include <cmath>
#include <future>
#include <memory>
#include <utility>
#include <vector>

namespace shellgpu {

struct NdFront {
  int j0 = 0;      // first pivot node (elimination position)
  int ns = 0;      // pivot nodes
  int parent = -1;
  int child[2] = {-1, -1};
  int depth = 0;            // distance from the root
  std::vector<int> bnd;     // boundary nodes: elimination positions, ascending
};

struct NdTree {
  std::vector<int> perm;       // elimination position -> node
  std::vector<int> pos;        // node -> elimination position
  std::vector<NdFront> fronts; // children before parents
  int ndepth = 0;
};

class NdBuilder {
 public:
  NdBuilder(int nn, const int *rowp, const int *cols, const double *X, int leaf)
      : nn_(nn), rowp_(rowp), cols_(cols), leaf_(leaf), where_(nn), rank_(nn), dist_(nn), side_(nn) {
    for (auto &w : where_) w.store(-1, std::memory_order_relaxed);
    // the whole mesh along each coordinate; the sets below keep these orders
    // (a stable partition), so nothing is sorted again
    all_.reset(new Part());
    std::vector<std::future<void>> wait;
    for (int d = 0; d < 3; d++)
      wait.push_back(std::async(nn > kFork ? kThread : std::launch::deferred, [this, X, d] {
        std::vector<std::pair<double, int>> key(nn_);
        for (int i = 0; i < nn_; i++) key[i] = {X[3 * i + d], i};
        std::sort(key.begin(), key.end());
        all_->along[d].resize(nn_);
        for (int i = 0; i < nn_; i++) all_->along[d][i] = key[i].second;
      }));
    for (auto &w : wait) w.get();
  }

  NdTree build() {
    t_.perm.clear();
    t_.pos.assign(nn_, -1);
    cut(*all_, 0);
    collect(*all_, 0);
    for (int p = 0; p < nn_; p++) t_.pos[t_.perm[p]] = p;
    symbolic();
    return std::move(t_);
  }

 private:
  // sets of more nodes are cut on a thread of their own, 4 levels deep
  static constexpr int kFork = 2000, kForkDepth = 4;
  // a thread where the system has one to give, else in the caller's get()
  static constexpr std::launch kThread = std::launch::async | std::launch::deferred;

  struct Part {
    std::vector<int> along[3];  // the same nodes along the three coordinates
    std::vector<int> sep;       // the separator, or a leaf's nodes
    std::unique_ptr<Part> side[2];
  };
  struct Cut {
    double cost = -1.0;
    bool right = false;  // the separator is taken from the nodes after the cut
    int at = 0, sweep = -1;
  };

  int nn_;
  const int *rowp_, *cols_;
  int leaf_;
  // by node: stamp of its set (neighbours of other sets, cut by other
  // threads, are looked at too), rank in the sweep, BFS distance, side
  std::vector<std::atomic<int>> where_;
  std::vector<int> rank_, dist_;
  std::vector<signed char> side_;
  std::atomic<int> stamps_{0};
  std::unique_ptr<Part> all_;
  NdTree t_;

  bool in(int v, int stamp) const { return where_[v].load(std::memory_order_relaxed) == stamp; }

  // best cut of a set along an order
  void sweep(const std::vector<int> &order, int stamp, int which, Cut &best) {
    const int n = (int)order.size();
    for (int k = 0; k < n; k++) rank_[order[k]] = k;
    std::vector<int> left(n + 2, 0), right(n + 2, 0);
    for (int k = 0; k < n; k++) {
      const int v = order[k];
      int lo = k, hi = k;
      for (int p = rowp_[v]; p < rowp_[v + 1]; p++) {
        const int w = cols_[p];
        if (!in(w, stamp)) continue;
        lo = std::min(lo, rank_[w]);
        hi = std::max(hi, rank_[w]);
      }
      // v is in the separator of cut c when it lies before (after) the cut
      // and has a neighbour after (before) it: k < c <= hi, lo < c <= k
      left[k + 1]++;
      left[hi + 1]--;
      right[lo + 1]++;
      right[k + 1]--;
    }
    const int c0 = std::max(1, (3 * n) / 10), c1 = std::min(n - 1, n - (3 * n) / 10);
    int l = 0, r = 0;
    for (int c = 1; c <= c1; c++) {
      l += left[c];
      r += right[c];
      if (c < c0) continue;
      const double b = 2.0 * c / n - 1.0, pen = 1.0 + 2.0 * b * b;
      for (int side = 0; side < 2; side++) {
        const double cost = (side ? r : l) * pen;
        if (best.cost < 0.0 || cost < best.cost) best = {cost, side == 1, c, which};
      }
    }
  }

  // cut a set down to its leaves
  void cut(Part &set, int depth) {
    const int n = (int)set.along[0].size();
    if (n <= leaf_) {
      set.sep.swap(set.along[0]);
      return;
    }
    const int stamp = ++stamps_;
    for (int v : set.along[0]) where_[v].store(stamp, std::memory_order_relaxed);
    Cut best;
    for (int d = 0; d < 3; d++) sweep(set.along[d], stamp, d, best);
    // breadth-first sweep where planes do not find the short lines of a
    // surface (coordinates that coincide or fold)
    std::vector<int> order;
    if (best.cost > 3.0 * std::sqrt((double)n)) {
      bfs(set.along[0], stamp, order);
      sweep(order, stamp, 3, best);
    }
    const std::vector<int> &along = best.sweep == 3 ? order : set.along[best.sweep];
    for (int k = 0; k < n; k++) side_[along[k]] = k >= best.at;
    // the separator: nodes of one side with a neighbour on the other
    std::vector<int> &s = set.sep;
    for (int k = 0; k < n; k++) {
      const int v = along[k];
      if ((k >= best.at) != best.right) continue;
      for (int p = rowp_[v]; p < rowp_[v + 1]; p++) {
        const int w = cols_[p];
        if (in(w, stamp) && (side_[w] & 1) != (int)best.right) {
          s.push_back(v);
          break;
        }
      }
    }
    // disconnected sides: any node keeps the tree binary
    if (s.empty()) s.push_back(along[best.right ? n - 1 : 0]);
    for (int v : s) side_[v] = 2 + (side_[v] & 1);
    for (auto &p : set.side) p.reset(new Part());
    for (int d = 0; d < 3; d++) {
      for (auto &p : set.side) p->along[d].reserve(n / 2 + 1);
      for (int v : set.along[d])
        if (side_[v] < 2) set.side[(int)side_[v]]->along[d].push_back(v);
      std::vector<int>().swap(set.along[d]);
    }
    std::vector<int>().swap(order);
    for (auto &p : set.side)
      if (p->along[0].empty()) p.reset();
    std::future<void> other;
    if (n > kFork && depth < kForkDepth && set.side[0] && set.side[1])
      other = std::async(kThread, [this, &set, depth] { cut(*set.side[0], depth + 1); });
    else if (set.side[0])
      cut(*set.side[0], depth + 1);
    if (set.side[1]) cut(*set.side[1], depth + 1);
    if (other.valid()) other.get();
  }

  // the set in breadth-first order from a far node (components one after another)
  void bfs(const std::vector<int> &set, int stamp, std::vector<int> &order) {
    int start = set[0];
    for (int it = 0; it < 3; it++) {
      for (int v : set) dist_[v] = -1;
      order.clear();
      size_t next = 0;
      int root = start;
      while (order.size() < set.size()) {
        size_t h = order.size();
        dist_[root] = 0;
        order.push_back(root);
        for (; h < order.size(); h++) {
          const int v = order[h];
          for (int p = rowp_[v]; p < rowp_[v + 1]; p++) {
            const int w = cols_[p];
            if (in(w, stamp) && dist_[w] < 0) {
              dist_[w] = dist_[v] + 1;
              order.push_back(w);
            }
          }
        }
        while (next < set.size() && dist_[set[next]] >= 0) next++;
        if (next < set.size()) root = set[next];
      }
      start = order.back();
    }
  }

  // fronts and elimination order from the cut sets, children first
  int collect(Part &set, int depth) {
    int child[2] = {-1, -1};
    for (int k = 0; k < 2; k++)
      if (set.side[k]) {
        child[k] = collect(*set.side[k], depth + 1);
        set.side[k].reset();
      }
    if (child[0] < 0) std::swap(child[0], child[1]);
    NdFront f;
    f.j0 = (int)t_.perm.size();
    f.ns = (int)set.sep.size();
    f.depth = depth;
    f.child[0] = child[0];
    f.child[1] = child[1];
    t_.perm.insert(t_.perm.end(), set.sep.begin(), set.sep.end());
    const int id = (int)t_.fronts.size();
    for (int c : child)
      if (c >= 0) t_.fronts[c].parent = id;
    t_.fronts.push_back(std::move(f));
    t_.ndepth = std::max(t_.ndepth, depth + 1);
    return id;
  }

  // boundary of a front: later neighbours of its pivots and of its children's
  // boundaries
  void symbolic() {
    std::vector<int> mark(nn_, -1);
    for (size_t s = 0; s < t_.fronts.size(); s++) {
      NdFront &f = t_.fronts[s];
      const int end = f.j0 + f.ns;
      for (int j = f.j0; j < end; j++) {
        const int v = t_.perm[j];
        for (int p = rowp_[v]; p < rowp_[v + 1]; p++) {
          const int q = t_.pos[cols_[p]];
          if (q >= end && mark[q] != (int)s) {
            mark[q] = (int)s;
            f.bnd.push_back(q);
          }
        }
      }
      for (int c : f.child)
        if (c >= 0)
          for (int q : t_.fronts[c].bnd)
            if (q >= end && mark[q] != (int)s) {
              mark[q] = (int)s;
              f.bnd.push_back(q);
            }
      std::sort(f.bnd.begin(), f.bnd.end());
    }
  }
};

}  // namespace shellgpu
