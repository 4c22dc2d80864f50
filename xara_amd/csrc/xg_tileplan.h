// Plan of the tiled sparse factorisation (host code, no HIP): a nested-
// dissection order of the equations from the nodes' coordinates, cut into
// tile columns of at most 64 equations, the tile pattern of the factor, and
// the task lists of its launches.
//
// Order.  A set of nodes is cut across the axis with the lightest
// separator: the nodes sorted along the axis, cut at the widest gap near the
// middle (a layered mesh is cut between layers, also where its nodes are
// slightly off them), the separator the nodes of one side that a matrix entry
// joins to the other.  Both sides are ordered first, the separator last,
// its nodes by bisection so that a tile holds nodes near each other.  The
// chain of dependent tile columns is then one branch of separators (37 levels
// on a 10 x 10 x 20 frame) instead of the whole band (227).
//
// Tiles.  Tile column k holds equations at positions 64 k .. 64 k + wid - 1;
// the rest of its 64 positions are padding.  Its tiles are the diagonal one
// (slot colptr[k] + k) followed by one per row tile row[colptr[k] ..
// colptr[k+1] - 1]: the diagonal adds one slot per column, so the slot of the
// j-th row tile of column k is colptr[k] + k + 1 + j.
//
// Levels.  level(k) = 1 + the highest level of a column whose factor updates
// column k; the columns of one level are independent.
//
// Groups.  Runs of up to kTileGroup columns of one piece in which each
// updates the next: inside a run a column's update is applied at its level,
// to the tiles beyond the run all its columns' at the level of the last one,
// in one pass over each target.  (Every tile that a column of the run updates
// beyond it lies in a column of a higher level than the run's last, which
// has inherited the run's rows.)
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace xg {

constexpr int kTile = 64;
constexpr int kTileGroup = 4;

struct TilePlan {
  int nt = 0;                 // tile columns
  int nlev = 0;               // levels
  std::vector<int> pos;       // position of each equation, 64 * column + offset
  std::vector<int> wid;       // equations of each column
  std::vector<int> colptr;    // nt + 1
  std::vector<int> row;       // row tiles of each column, ascending
  std::vector<int> lev;       // level of each column
  long long tiles() const { return (long long)row.size() + nt; }
  long long diag(int k) const { return (long long)colptr[k] + k; }
  // columns by level: levptr (nlev + 1) into levcol
  std::vector<int> levptr, levcol;
  // updates by level: targets upptr[l] .. upptr[l+1]-1, target t the tile
  // slot uptgt[t] minus the sum over s = upsrc[t] .. upsrc[t+1]-1 of
  // G(slot srcg[s]) A(slot srca[s])^T over srck[s] columns
  std::vector<int> upptr, uptgt, upsrc, srcg, srca, srck;
  // forward sweep by level: row tiles fwptr[l] .. fwptr[l+1]-1, row fwrow[t]
  // minus the sum over s = fwsrc[t] .. fwsrc[t+1]-1 of G(slot fwg[s])
  // y(column fwk[s])
  std::vector<int> fwptr, fwrow, fwsrc, fwg, fwk;
  // backward sweep by level (of the row tiles): columns bwptr[l] ..
  // bwptr[l+1]-1, column bwcol[t] minus the sum over s = bwsrc[t] ..
  // bwsrc[t+1]-1 of G(slot bwg[s])^T x(row tile bwr[s])
  std::vector<int> bwptr, bwcol, bwsrc, bwg, bwr;
  double flops = 0;           // multiply-adds of the updates and panels, x 2
};

namespace tileplan {

struct Graph {
  int dim = 3;
  const std::vector<int>* ptr = nullptr;  // node adjacency
  const std::vector<int>* adj = nullptr;
  const double* xyz = nullptr;            // dim per node
  const int* w = nullptr;                 // equations per node
};

inline int weight(const Graph& g, const std::vector<int>& v) {
  int s = 0;
  for (int n : v) s += g.w[n];
  return s;
}

// nodes by repeated bisection across the longest extent, until a part fits
// a tile (ties by the other axes, then by index: a total order)
inline void bisect_order(const Graph& g, int* b, int* e) {
  int tot = 0;
  for (int* p = b; p != e; p++) tot += g.w[*p];
  if (tot <= kTile || e - b < 3) {
    std::sort(b, e);
    return;
  }
  int ax = 0;
  double best = -1;
  for (int d = 0; d < g.dim; d++) {
    double lo = 1e300, hi = -1e300;
    for (int* p = b; p != e; p++) {
      lo = std::min(lo, g.xyz[(size_t)*p * g.dim + d]);
      hi = std::max(hi, g.xyz[(size_t)*p * g.dim + d]);
    }
    if (hi - lo > best) {
      best = hi - lo;
      ax = d;
    }
  }
  std::sort(b, e, [&](int a, int c) {
    const double x = g.xyz[(size_t)a * g.dim + ax], y = g.xyz[(size_t)c * g.dim + ax];
    return x != y ? x < y : a < c;
  });
  // the first half a whole number of tiles
  const int half = std::max(kTile, (tot / 2 + kTile - 1) / kTile * kTile);
  int run = 0;
  int* m = b;
  while (m != e && run + g.w[*m] <= half) run += g.w[*m++];
  if (m == b || m == e) {
    std::sort(b, e);
    return;
  }
  bisect_order(g, b, m);
  bisect_order(g, m, e);
}

// One cut of `v` along axis ax: the index after which the sorted nodes go
// right, at the widest coordinate gap between 40% and 60% of the weight (the
// nearest to the middle of gaps within 0.1% of the widest).
inline size_t widest_gap(const Graph& g, const std::vector<int>& v, int ax, int tot) {
  size_t at = 0;
  double gap = -1.0;
  int off = 0;
  long long run = 0;
  for (size_t i = 0; i + 1 < v.size(); i++) {
    run += g.w[v[i]];
    if (run * 10 < 4LL * tot || run * 10 > 6LL * tot) {
      if (run * 10 > 6LL * tot) break;
      continue;
    }
    const double d = g.xyz[(size_t)v[i + 1] * g.dim + ax] - g.xyz[(size_t)v[i] * g.dim + ax];
    const int o = (int)std::abs(2 * run - tot);
    if (d > 1.001 * gap || (d > 0.999 * gap && o < off)) {
      gap = std::max(gap, d);
      at = i + 1;
      off = o;
    }
  }
  if (at == 0) {  // no node boundary in the window: the one nearest the middle
    run = 0;
    off = tot + 1;
    for (size_t i = 0; i + 1 < v.size(); i++) {
      run += g.w[v[i]];
      const int o = (int)std::abs(2 * run - tot);
      if (o < off) {
        off = o;
        at = i + 1;
      }
    }
  }
  return at;
}

// Appends the nodes of `v` in elimination order to `out`, and the end of
// each piece (leaf or separator) to `ends`.  mark: 0 on entry and exit.
inline void dissect(const Graph& g, std::vector<int> v, std::vector<char>& mark, std::vector<int>& out,
                    std::vector<int>& ends, int depth) {
  if (v.empty()) return;
  auto emit = [&](std::vector<int>& s) {
    if (s.empty()) return;
    bisect_order(g, s.data(), s.data() + s.size());
    out.insert(out.end(), s.begin(), s.end());
    ends.push_back((int)out.size());
  };
  const int tot = weight(g, v);
  if (tot <= kTile || v.size() < 3 || depth > 60) {
    emit(v);
    return;
  }
  std::vector<int> L, R, S, bl, br, bs;
  long long best = -1;
  for (int ax = 0; ax < g.dim; ax++) {
    std::sort(v.begin(), v.end(), [&](int a, int c) {
      const double x = g.xyz[(size_t)a * g.dim + ax], y = g.xyz[(size_t)c * g.dim + ax];
      return x != y ? x < y : a < c;
    });
    const size_t cut = widest_gap(g, v, ax, tot);
    if (cut == 0 || cut >= v.size()) continue;
    for (size_t i = 0; i < v.size(); i++) mark[v[i]] = i < cut ? 1 : 2;
    int sw[2] = {0, 0};
    for (int side = 0; side < 2; side++)
      for (size_t i = side ? cut : 0; i < (side ? v.size() : cut); i++)
        for (int q = (*g.ptr)[v[i]]; q < (*g.ptr)[v[i] + 1]; q++)
          if (mark[(*g.adj)[q]] == 2 - side) {
            sw[side] += g.w[v[i]];
            break;
          }
    const int side = sw[1] <= sw[0] ? 1 : 0;  // the lighter boundary separates
    L.clear();
    R.clear();
    S.clear();
    for (size_t i = 0; i < v.size(); i++) {
      const bool right = i >= cut;
      bool sep = false;
      if (right == (side == 1))
        for (int q = (*g.ptr)[v[i]]; q < (*g.ptr)[v[i] + 1] && !sep; q++)
          sep = mark[(*g.adj)[q]] == (right ? 1 : 2);
      (sep ? S : right ? R : L).push_back(v[i]);
    }
    for (int n : v) mark[n] = 0;
    // lightest separator; of equal ones the better balanced cut
    const int lw = weight(g, L), rw = weight(g, R);
    const long long score = (long long)weight(g, S) * 1024 + 256LL * std::abs(lw - rw) / std::max(1, tot);
    if (!L.empty() && !R.empty() && (best < 0 || score < best)) {
      best = score;
      bl.swap(L);
      br.swap(R);
      bs.swap(S);
    }
  }
  if (best < 0) {  // every cut leaves one side empty: one dense piece
    emit(v);
    return;
  }
  v.clear();
  v.shrink_to_fit();
  dissect(g, std::move(bl), mark, out, ends, depth + 1);
  dissect(g, std::move(br), mark, out, ends, depth + 1);
  emit(bs);
}

}  // namespace tileplan

// Builds the plan of an n-equation matrix (CSR pattern, symmetric) whose
// equations belong to nodes with coordinates (eq: nnode*ndf equation numbers,
// -1 for a fixed DOF).  Returns false, leaving the plan unusable, when the
// factor would exceed max_tiles tiles or its updates max_flops.
inline bool tile_plan(int n, const std::vector<int>& rowptr, const std::vector<int>& colind, int nnode, int ndf,
                      int ndm, const std::vector<int>& eq, const std::vector<double>& crd, long long max_tiles,
                      double max_flops, TilePlan& P) {
  P = TilePlan{};
  if (n <= 0) return false;
  // node graph of the free equations
  std::vector<int> node_of(n, -1), wt(nnode, 0), aptr(nnode + 1, 0), adj, first(nnode, -1);
  for (int i = 0; i < nnode; i++)
    for (int j = 0; j < ndf; j++) {
      const int e = eq[(size_t)i * ndf + j];
      if (e < 0) continue;
      node_of[e] = i;
      wt[i]++;
    }
  for (int e = 0; e < n; e++)
    if (node_of[e] < 0) return false;
  {
    std::vector<int> seen(nnode, -1);
    for (int i = 0; i < nnode; i++) {
      for (int j = 0; j < ndf; j++) {
        const int e = eq[(size_t)i * ndf + j];
        if (e < 0) continue;
        for (int q = rowptr[e]; q < rowptr[e + 1]; q++) {
          const int m = node_of[colind[q]];
          if (m != i && seen[m] != i) {
            seen[m] = i;
            adj.push_back(m);
          }
        }
      }
      aptr[i + 1] = (int)adj.size();
    }
  }
  tileplan::Graph g;
  g.dim = ndm;
  g.ptr = &aptr;
  g.adj = &adj;
  g.xyz = crd.data();
  g.w = wt.data();
  std::vector<int> all, order, ends;
  for (int i = 0; i < nnode; i++)
    if (wt[i]) all.push_back(i);
  std::vector<char> mark(nnode, 0);
  tileplan::dissect(g, std::move(all), mark, order, ends, 0);
  // tile columns: a piece's equations in runs of 64
  P.pos.assign(n, -1);
  std::vector<int> col_of(n);
  size_t b = 0;
  std::vector<int> piece;  // of each tile column
  for (int en : ends) {
    int fill = kTile;
    for (; b < (size_t)en; b++)
      for (int j = 0; j < ndf; j++) {
        const int e = eq[(size_t)order[b] * ndf + j];
        if (e < 0) continue;
        if (fill == kTile) {
          P.wid.push_back(0);
          piece.push_back(en);
          fill = 0;
        }
        col_of[e] = (int)P.wid.size() - 1;
        P.pos[e] = kTile * col_of[e] + fill++;
        P.wid.back() = fill;
      }
  }
  const int nt = P.nt = (int)P.wid.size();
  // tile pattern of the factor: the matrix's, with each column's rows
  // handed on to its parent (its first row tile)
  std::vector<std::vector<int>> str(nt);
  {
    std::vector<std::vector<int>> in(nt);  // equations of each column
    for (int e = 0; e < n; e++) in[col_of[e]].push_back(e);
    std::vector<int> seen(nt, -1);
    std::vector<std::vector<int>> kids(nt);
    long long tiles = 0;
    double flops = 0;
    for (int k = 0; k < nt; k++) {
      seen[k] = k;
      std::vector<int>& s = str[k];
      for (int e : in[k])
        for (int q = rowptr[e]; q < rowptr[e + 1]; q++) {
          const int c = col_of[colind[q]];
          if (c > k && seen[c] != k) {
            seen[c] = k;
            s.push_back(c);
          }
        }
      for (int c : kids[k]) {
        for (int r : str[c])
          if (r > k && seen[r] != k) {
            seen[r] = k;
            s.push_back(r);
          }
      }
      std::sort(s.begin(), s.end());
      if (!s.empty()) kids[s[0]].push_back(k);
      tiles += 1 + (long long)s.size();
      const double m = (double)s.size();
      flops += 2.0 * kTile * kTile * ((P.wid[k] + 15) / 16 * 16) * (0.5 * m * (m + 1) + m + 1);
      if (tiles > max_tiles || flops > max_flops) return false;
    }
    P.flops = flops;
  }
  P.colptr.assign(nt + 1, 0);
  for (int k = 0; k < nt; k++) P.colptr[k + 1] = P.colptr[k] + (int)str[k].size();
  P.row.reserve(P.colptr[nt]);
  for (auto& s : str) P.row.insert(P.row.end(), s.begin(), s.end());
  // levels
  P.lev.assign(nt, 0);
  for (int k = 0; k < nt; k++) {
    for (int r : str[k]) P.lev[r] = std::max(P.lev[r], P.lev[k] + 1);
    P.nlev = std::max(P.nlev, P.lev[k] + 1);
  }
  P.levptr.assign(P.nlev + 1, 0);
  for (int k = 0; k < nt; k++) P.levptr[P.lev[k] + 1]++;
  for (int l = 0; l < P.nlev; l++) P.levptr[l + 1] += P.levptr[l];
  P.levcol.resize(nt);
  {
    std::vector<int> at(P.levptr.begin(), P.levptr.end() - 1);
    for (int k = 0; k < nt; k++) P.levcol[at[P.lev[k]]++] = k;
  }
  // updates and forward rows of each level, grouped by target; a target's
  // sources in ascending column order
  auto slot = [&](int i, int j) {  // tile (i, j), i >= j
    if (i == j) return (int)P.diag(j);
    const std::vector<int>& s = str[j];
    return (int)(P.diag(j) + 1 + (std::lower_bound(s.begin(), s.end(), i) - s.begin()));
  };
  struct Src {
    int tgt, g, a, k;
  };
  // last column of each column's group
  std::vector<int> last(nt);
  for (int k = nt - 1, left = 0; k >= 0; k--) {
    const bool chain = k + 1 < nt && piece[k + 1] == piece[k] && !str[k].empty() && str[k][0] == k + 1;
    left = chain && left > 1 ? left - 1 : kTileGroup;
    last[k] = left < kTileGroup ? last[k + 1] : k;
  }
  std::vector<Src> fw;
  std::vector<std::vector<Src>> ups(P.nlev);
  for (int k = 0; k < nt; k++) {
    const std::vector<int>& s = str[k];
    const int base = (int)P.diag(k) + 1;
    for (size_t b2 = 0; b2 < s.size(); b2++)
      for (size_t a2 = b2; a2 < s.size(); a2++)
        ups[P.lev[s[b2] <= last[k] ? k : last[k]]].push_back(
            {slot(s[a2], s[b2]), base + (int)a2, base + (int)b2, k});
  }
  P.upptr.assign(1, 0);
  P.fwptr.assign(1, 0);
  P.upsrc.assign(1, 0);
  P.fwsrc.assign(1, 0);
  for (int l = 0; l < P.nlev; l++) {
    std::vector<Src>& up = ups[l];
    fw.clear();
    for (int c = P.levptr[l]; c < P.levptr[l + 1]; c++) {
      const int k = P.levcol[c];
      const std::vector<int>& s = str[k];
      const int base = (int)P.diag(k) + 1;
      for (size_t b2 = 0; b2 < s.size(); b2++) fw.push_back({s[b2], base + (int)b2, 0, k});
    }
    auto less = [](const Src& x, const Src& y) { return x.tgt != y.tgt ? x.tgt < y.tgt : x.k < y.k; };
    std::sort(up.begin(), up.end(), less);
    std::sort(fw.begin(), fw.end(), less);
    for (size_t i = 0; i < up.size(); i++) {
      if (i == 0 || up[i].tgt != up[i - 1].tgt) {
        if (i) P.upsrc.push_back((int)P.srcg.size());
        P.uptgt.push_back(up[i].tgt);
      }
      P.srcg.push_back(up[i].g);
      P.srca.push_back(up[i].a);
      P.srck.push_back((P.wid[up[i].k] + 15) / 16 * 16);
    }
    if (!up.empty()) P.upsrc.push_back((int)P.srcg.size());
    P.upptr.push_back((int)P.uptgt.size());
    for (size_t i = 0; i < fw.size(); i++) {
      if (i == 0 || fw[i].tgt != fw[i - 1].tgt) {
        if (i) P.fwsrc.push_back((int)P.fwg.size());
        P.fwrow.push_back(fw[i].tgt);
      }
      P.fwg.push_back(fw[i].g);
      P.fwk.push_back(fw[i].k);
    }
    if (!fw.empty()) P.fwsrc.push_back((int)P.fwg.size());
    P.fwptr.push_back((int)P.fwrow.size());
  }
  // backward columns of each level, a column's row tiles ascending
  std::vector<std::vector<Src>> bw(P.nlev);
  for (int k = 0; k < nt; k++)
    for (size_t j = 0; j < str[k].size(); j++)
      bw[P.lev[str[k][j]]].push_back({k, (int)(P.diag(k) + 1 + j), 0, str[k][j]});
  P.bwptr.assign(1, 0);
  P.bwsrc.assign(1, 0);
  for (int l = 0; l < P.nlev; l++) {
    for (size_t i = 0; i < bw[l].size(); i++) {
      if (i == 0 || bw[l][i].tgt != bw[l][i - 1].tgt) {
        if (i) P.bwsrc.push_back((int)P.bwg.size());
        P.bwcol.push_back(bw[l][i].tgt);
      }
      P.bwg.push_back(bw[l][i].g);
      P.bwr.push_back(bw[l][i].k);
    }
    if (!bw[l].empty()) P.bwsrc.push_back((int)P.bwg.size());
    P.bwptr.push_back((int)P.bwcol.size());
  }
  return true;
}

}  // namespace xg
