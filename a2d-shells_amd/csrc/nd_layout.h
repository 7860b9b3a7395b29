// nd_layout.h -- where the fronts of a nested-dissection factor lie in the
// device buffers (host code, no device calls).
#pragma once

#include <algorithm>
#include <vector>

#include "nd_order.h"

namespace shellgpu {

// one front on the device; sizes in dofs, offsets in doubles per design
struct NdDev {
  int ns, m;        // pivot dofs, front dofs (pivots, then boundary)
  int child[2];     // fronts whose Schur complements it takes, or -1
  int lists;        // first entry of its node lists: m / 6 node ids, then per
                    // child m / 6 places in the child's boundary (or -1)
  int pad;
  long M, Q, S, V;  // panel (m x ns), scaled panels of the level (m x ns),
                    // Schur complement (m - ns)^2, front vector (m)
};

struct NdLevel {
  int f0, nf;          // fronts f0 .. f0 + nf
  int max_ns, max_nb;  // largest pivot and boundary blocks
  int max_m;
  bool inner;          // some front has children
};

struct NdLayout {
  std::vector<NdDev> fronts;  // deepest level first
  std::vector<int> lists;
  std::vector<NdLevel> levels;  // deepest first
  long per_design = 0, q_len = 0, s_len[2] = {0, 0}, v_len = 0;
  // per BSR block where it goes in M (base -1: the transpose of a stored block)
  std::vector<long> blk_base;
  std::vector<int> blk_ld;
};

inline NdLayout nd_layout(int nn, const std::vector<int> &rowp, const std::vector<int> &cols, const double *X, int leaf) {
  NdLayout L;
  const NdTree tree = NdBuilder(nn, rowp.data(), cols.data(), X, leaf).build();
  const int nf = (int)tree.fronts.size();
  // device order: deepest level first
  std::vector<int> at(nf), by(nf);
  {
    std::vector<int> cnt(tree.ndepth + 1, 0);
    for (const NdFront &f : tree.fronts) cnt[tree.ndepth - 1 - f.depth + 1]++;
    for (int l = 0; l < tree.ndepth; l++) cnt[l + 1] += cnt[l];
    for (int s = 0; s < nf; s++) {
      at[s] = cnt[tree.ndepth - 1 - tree.fronts[s].depth]++;
      by[at[s]] = s;
    }
  }
  std::vector<NdDev> &dev = L.fronts;
  std::vector<int> &lists = L.lists;
  std::vector<long> &blk_base = L.blk_base;
  std::vector<int> &blk_ld = L.blk_ld;
  dev.resize(nf);
  long off_m = 0, off_v = 0;
  L.levels.assign(tree.ndepth, NdLevel{0, 0, 0, 0, 0, false});
  std::vector<long> q_at(tree.ndepth, 0), s_at(tree.ndepth, 0);
  std::vector<int> place(nn, -1);
  for (int k = 0; k < nf; k++) {
    const NdFront &f = tree.fronts[by[k]];
    const int l = tree.ndepth - 1 - f.depth, nb = 6 * (int)f.bnd.size();
    NdDev &d = dev[k];
    d = NdDev();
    d.ns = 6 * f.ns;
    d.m = d.ns + nb;
    d.M = off_m;
    d.V = off_v;
    d.Q = q_at[l];
    d.S = s_at[l];
    off_m += (long)d.m * d.ns;
    off_v += d.m;
    q_at[l] += (long)d.m * d.ns;
    s_at[l] += (long)nb * nb;
    d.lists = (int)lists.size();
    for (int j = 0; j < f.ns; j++) {
      lists.push_back(tree.perm[f.j0 + j]);
    }
    for (int q : f.bnd) lists.push_back(tree.perm[q]);
    for (int c = 0; c < 2; c++) {
      d.child[c] = f.child[c] >= 0 ? at[f.child[c]] : -1;
      if (f.child[c] >= 0) {
        const std::vector<int> &cb = tree.fronts[f.child[c]].bnd;
        for (size_t i = 0; i < cb.size(); i++) place[cb[i]] = (int)i;
      }
      for (int j = 0; j < f.ns; j++) lists.push_back(place[f.j0 + j]);
      for (int q : f.bnd) lists.push_back(place[q]);
      if (f.child[c] >= 0)
        for (int q : tree.fronts[f.child[c]].bnd) place[q] = -1;
    }
    NdLevel &lv = L.levels[l];
    if (lv.nf == 0) lv.f0 = k;
    lv.nf++;
    lv.max_ns = std::max(lv.max_ns, d.ns);
    lv.max_nb = std::max(lv.max_nb, nb);
    lv.max_m = std::max(lv.max_m, d.m);
    lv.inner = lv.inner || d.child[0] >= 0;
  }
  L.per_design = off_m;
  L.v_len = off_v;
  for (int l = 0; l < tree.ndepth; l++) {
    L.q_len = std::max(L.q_len, q_at[l]);
    L.s_len[l & 1] = std::max(L.s_len[l & 1], std::max(2L, s_at[l]));
  }
  L.s_len[1] = std::max(L.s_len[1], 2L);
  // where the matrix blocks go: block (i, j) with i at or after j in the
  // order belongs to the front that eliminates j
  blk_base.assign(cols.size(), -1);
  blk_ld.assign(cols.size(), 0);
  std::vector<int> row_of(nn, -1);
  for (int k = 0; k < nf; k++) {
    const NdFront &f = tree.fronts[by[k]];
    for (int j = 0; j < f.ns; j++) row_of[f.j0 + j] = j;
    for (size_t i = 0; i < f.bnd.size(); i++) row_of[f.bnd[i]] = f.ns + (int)i;
    for (int j = 0; j < f.ns; j++) {
      const int v = tree.perm[f.j0 + j];
      for (int p = rowp[v]; p < rowp[v + 1]; p++) {
        const int w = cols[p];
        if (tree.pos[w] < f.j0 + j) continue;
        // the block (w, v): the pattern's rows are sorted
        const int *row = cols.data() + rowp[w];
        const int q = rowp[w] + (int)(std::lower_bound(row, cols.data() + rowp[w + 1], v) - row);
        blk_base[q] = dev[k].M + 6L * row_of[tree.pos[w]] + 6L * j * dev[k].m;
        blk_ld[q] = dev[k].m;
      }
    }
  }
  return L;
}

}  // namespace shellgpu
