// Supernodal multifrontal Cholesky with geometric nested dissection (setup).
#include "cholesky.hpp"

#include <omp.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <stdexcept>
#include <string>

namespace pecs {

namespace {

struct NDNode {
  std::vector<int> dofs;  // DoFs in grid order
  std::vector<int> children;
  int parent = -1;
};

// The couplings between single DoFs of the systems: neighbours of each DoF
// (grid-order numbering, one system after the other), from the nonzero entries
// of the blocks in either triangle, of the system or of one of its twins.
struct DofGraph {
  std::vector<std::vector<int>> dof0;  // per system: per cell, and its end
  std::vector<int> cell;               // per DoF
  std::vector<int> sys;                // per DoF
  std::vector<int64_t> ptr;            // per DoF
  std::vector<int> adj;
  int n = 0;

  DofGraph(const Systems& Ss, const std::vector<int>& twin) {
    for (const BlockSPD* S : Ss) {
      const int NG = S->NXc * S->NYc;
      std::vector<int> d(NG + 1, n);
      for (int X = 0; X < NG; ++X) d[X + 1] = d[X] + S->ndof[X];
      n = d[NG];
      dof0.push_back(std::move(d));
    }
    cell.resize(n);
    sys.resize(n);
    for (size_t k = 0; k < Ss.size(); ++k)
      for (int X = 0; X + 1 < (int)dof0[k].size(); ++X)
        for (int d = dof0[k][X]; d < dof0[k][X + 1]; ++d) {
          cell[d] = X;
          sys[d] = (int)k;
        }
    ptr.assign((size_t)n + 1, 0);
    for (int pass = 0; pass < 2; ++pass) {
      for (size_t k = 0; k < Ss.size(); ++k) {
        const BlockSPD& S = *Ss[k];
        const int NG = S.NXc * S.NYc, no = S.noff();
        std::vector<const BlockSPD*> like;  // the system and its twins
        for (size_t j = 0; j < Ss.size(); ++j)
          if (j == k || (!twin.empty() && twin[j] == twin[k])) like.push_back(Ss[j]);
        for (const BlockSPD* T : like)
          if (T->ndof != S.ndof || T->offi != S.offi || T->offj != S.offj)
            throw std::runtime_error("twin systems on different grids");
        std::vector<int> opp(no, -1);  // the opposite offset
        for (int o = 0; o < no; ++o)
          for (int q = 0; q < no; ++q)
            if (S.offi[q] == -S.offi[o] && S.offj[q] == -S.offj[o]) opp[o] = q;
#pragma omp parallel for schedule(dynamic, 256)
        for (int X = 0; X < NG; ++X) {
          const int nx = S.ndof[X];
          if (nx == 0) continue;
          const int xi = X % S.NXc, xj = X / S.NXc;
          for (int a = 0; a < nx; ++a) {
            int64_t cnt = 0;
            const int64_t at = pass ? ptr[dof0[k][X] + a] : 0;  // (the counting pass writes ptr)
            for (int o = 0; o < no; ++o) {
              const int yi = xi + S.offi[o], yj = xj + S.offj[o];
              if (yi < 0 || yi >= S.NXc || yj < 0 || yj >= S.NYc) continue;
              const int Y = yi + S.NXc * yj, ny = S.ndof[Y];
              for (int b = 0; b < ny; ++b) {
                bool nz = false;
                for (const BlockSPD* T : like) {
                  const std::vector<double>& B = T->blk[(size_t)X * no + o];
                  nz = nz || (!B.empty() && B[(size_t)a * ny + b] != 0.0);
                  if (nz || opp[o] < 0) continue;
                  const std::vector<double>& C = T->blk[(size_t)Y * no + opp[o]];
                  nz = !C.empty() && C[(size_t)b * nx + a] != 0.0;
                }
                if (!nz) continue;
                if (pass) adj[at + cnt] = dof0[k][Y] + b;
                ++cnt;
              }
            }
            if (!pass) ptr[dof0[k][X] + a + 1] = cnt;
          }
        }
      }
      if (!pass) {
        for (int d = 0; d < n; ++d) ptr[d + 1] += ptr[d];
        adj.resize(ptr[n]);
      }
    }
  }
};

struct NDBuilder {
  const BlockSPD& S;
  const DofGraph& G;
  const std::vector<int>& dof0;  // of this system
  int leaf, reach = 0;
  std::vector<NDNode>& nodes;  // postorder
  std::vector<char> taken;    // per DoF: already in a separator
  // scratch of cover(): per DoF its index on its side of the cut
  std::vector<int> side;

  NDBuilder(const BlockSPD& s, const DofGraph& g, int k, int l, std::vector<NDNode>& out)
      : S(s), G(g), dof0(g.dof0[k]), leaf(l), nodes(out), taken(g.n, 0), side(g.n, -1) {
    for (int o = 0; o < S.noff(); ++o) reach = std::max({reach, std::abs(S.offi[o]), std::abs(S.offj[o])});
  }

  // Minimum vertex cover of the couplings between the free DoFs of the
  // rectangle before and after the cut at column (row) mid: a maximum
  // matching of the bipartite graph (augmenting paths, a greedy start) and
  // Koenig's construction.
  std::vector<int> cover(int i0, int i1, int j0, int j1, int mid, bool vertical) {
    std::vector<int> L, R;                  // DoFs with a crossing coupling
    std::vector<int> eptr{0}, e;            // edges of L
    const int lo = std::max(vertical ? i0 : j0, mid - reach);
    const int u0 = vertical ? j0 : i0, u1 = vertical ? j1 : i1;
    for (int u = u0; u < u1; ++u)
      for (int t = lo; t < mid; ++t) {
        const int X = vertical ? t + S.NXc * u : u + S.NXc * t;
        for (int d = dof0[X]; d < dof0[X + 1]; ++d) {
          if (taken[d]) continue;
          const size_t before = e.size();
          for (int64_t q = G.ptr[d]; q < G.ptr[d + 1]; ++q) {
            const int v = G.adj[q], Y = G.cell[v], yi = Y % S.NXc, yj = Y / S.NXc;
            if (taken[v] || (vertical ? yi : yj) < mid || yi < i0 || yi >= i1 || yj < j0 || yj >= j1) continue;
            if (side[v] < 0) {
              side[v] = (int)R.size();
              R.push_back(v);
            }
            e.push_back(side[v]);
          }
          if (e.size() > before) {
            L.push_back(d);
            eptr.push_back((int)e.size());
          }
        }
      }
    for (int v : R) side[v] = -1;
    const int nl = (int)L.size(), nr = (int)R.size();
    std::vector<int> ml(nl, -1), mr(nr, -1);
    for (int l = 0; l < nl; ++l)
      for (int q = eptr[l]; q < eptr[l + 1] && ml[l] < 0; ++q)
        if (mr[e[q]] < 0) {
          ml[l] = e[q];
          mr[e[q]] = l;
        }
    std::vector<char> seen(nr);
    std::vector<int> stack, cur(nl);
    for (bool grew = true; grew;) {  // phases of disjoint augmenting paths
      grew = false;
      std::fill(seen.begin(), seen.end(), 0);
      for (int l = 0; l < nl; ++l) cur[l] = eptr[l];
      for (int l = 0; l < nl; ++l) {
        if (ml[l] >= 0) continue;
        stack.assign(1, l);
        while (!stack.empty()) {
          const int x = stack.back();
          if (cur[x] == eptr[x + 1]) {
            stack.pop_back();
            continue;
          }
          const int r = e[cur[x]++];
          if (seen[r]) continue;
          seen[r] = 1;
          if (mr[r] >= 0) {
            stack.push_back(mr[r]);
            continue;
          }
          // free: flip the path on the stack (each entry's edge is cur - 1)
          for (size_t i = stack.size(); i-- > 0;) {
            const int y = stack[i];
            ml[y] = e[cur[y] - 1];
            mr[ml[y]] = y;
          }
          grew = true;
          break;
        }
      }
    }
    // Koenig: reachable from the unmatched L by alternating paths
    std::vector<char> zl(nl, 0), zr(nr, 0);
    stack.clear();
    for (int l = 0; l < nl; ++l)
      if (ml[l] < 0) {
        zl[l] = 1;
        stack.push_back(l);
      }
    while (!stack.empty()) {
      const int x = stack.back();
      stack.pop_back();
      for (int q = eptr[x]; q < eptr[x + 1]; ++q) {
        if (zr[e[q]]) continue;
        zr[e[q]] = 1;
        const int y = mr[e[q]];
        if (y >= 0 && !zl[y]) {
          zl[y] = 1;
          stack.push_back(y);
        }
      }
    }
    std::vector<int> c;
    for (int l = 0; l < nl; ++l)
      if (!zl[l]) c.push_back(L[l]);
    for (int r = 0; r < nr; ++r)
      if (zr[r]) c.push_back(R[r]);
    // along the cut
    auto key = [&](int d) {
      const int X = G.cell[d], i = X % S.NXc, j = X / S.NXc;
      return vertical ? j : i;
    };
    std::sort(c.begin(), c.end(), [&](int a, int b) { return std::make_pair(key(a), a) < std::make_pair(key(b), b); });
    return c;
  }

  int push(NDNode&& node) {
    const int id = (int)nodes.size();
    for (int k : node.children) nodes[k].parent = id;
    nodes.push_back(std::move(node));
    return id;
  }

  int build(int i0, int i1, int j0, int j1) {
    const int ni = i1 - i0, nj = j1 - j0;
    if (ni <= 0 || nj <= 0) return -1;
    NDNode node;
    if (ni * nj <= leaf || (ni == 1 && nj == 1)) {
      for (int j = j0; j < j1; ++j)
        for (int i = i0; i < i1; ++i)
          for (int d = dof0[i + S.NXc * j]; d < dof0[i + S.NXc * j + 1]; ++d)
            if (!taken[d]) node.dofs.push_back(d);
      return node.dofs.empty() ? -1 : push(std::move(node));
    }
    const bool vertical = ni >= nj;
    const int mid = vertical ? i0 + ni / 2 : j0 + nj / 2;
    node.dofs = cover(i0, i1, j0, j1, mid, vertical);
    for (int d : node.dofs) taken[d] = 1;
    const int a = vertical ? build(i0, mid, j0, j1) : build(i0, i1, j0, mid);
    const int b = vertical ? build(mid, i1, j0, j1) : build(i0, i1, mid, j1);
    if (a >= 0) node.children.push_back(a);
    if (b >= 0) node.children.push_back(b);
    if (node.dofs.empty()) {
      if (node.children.size() < 2) return a >= 0 ? a : b;
      // uncoupled halves: a node needs DoFs of its own, so it takes the last
      // one of its second child's subtree root (any set containing a
      // separator is one)
      NDNode& r = nodes[b];
      node.dofs.push_back(r.dofs.back());
      r.dofs.pop_back();
      if (r.dofs.empty()) {  // the root held one DoF: this node replaces it
        for (int k : r.children) node.children.push_back(k);
        node.children.erase(node.children.begin() + 1);
        nodes.pop_back();  // b was the last node pushed
      }
    }
    return push(std::move(node));
  }
};

// F[i][j] -= sum_t P[i][t] P[j][t] for k1 <= j <= i < nf, P = F[:, k0:k0+pw].
// Register-blocked 4 x 8 micro-kernel over a packed copy of the panel and of
// its transpose.
void trailing_update(double* F, int nf, int k0, int k1, int pw) {
  const int nt = nf - k1;
  const int ntp = (nt + 7) & ~7;
  std::vector<double> P((size_t)(nt + 4) * pw, 0.0), PT((size_t)pw * (ntp + 8), 0.0);
  const int ld = ntp + 8;
#pragma omp parallel for schedule(static) if (nt > 256)
  for (int i = 0; i < nt; ++i)
    for (int t = 0; t < pw; ++t) {
      const double v = F[(size_t)(k1 + i) * nf + k0 + t];
      P[(size_t)i * pw + t] = v;
      PT[(size_t)t * ld + i] = v;
    }
  const int nib = (nt + 3) / 4;
#pragma omp parallel for schedule(dynamic, 4) if (nt > 64)
  for (int ib = nib - 1; ib >= 0; --ib) {
    const int i0 = 4 * ib;
    const double* a0 = &P[(size_t)(i0 + 0) * pw];
    const double* a1 = &P[(size_t)(i0 + 1) * pw];
    const double* a2 = &P[(size_t)(i0 + 2) * pw];
    const double* a3 = &P[(size_t)(i0 + 3) * pw];
    for (int j0 = 0; j0 <= i0 + 3 && j0 < nt; j0 += 8) {
      double acc[4][8];
      for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 8; ++c) acc[r][c] = 0.0;
      const double* bt = &PT[j0];
      for (int t = 0; t < pw; ++t) {
        const double* b = bt + (size_t)t * ld;
        const double x0 = a0[t], x1 = a1[t], x2 = a2[t], x3 = a3[t];
#pragma omp simd
        for (int c = 0; c < 8; ++c) {
          acc[0][c] += x0 * b[c];
          acc[1][c] += x1 * b[c];
          acc[2][c] += x2 * b[c];
          acc[3][c] += x3 * b[c];
        }
      }
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + r;
        if (i >= nt) break;
        double* Fi = &F[(size_t)(k1 + i) * nf + k1];
        const int jmax = std::min(j0 + 8, i + 1);
        for (int j = j0; j < jmax; ++j) Fi[j] -= acc[r][j - j0];
      }
    }
  }
}

// Partial Cholesky of the leading ns columns of the lower triangle of the
// nf x nf row-major front F (upper triangle ignored).  On return F holds L11,
// L21 and the Schur update in its lower triangle.
void partial_cholesky(double* F, int nf, int ns, double& flops) {
  const int BS = 64;
  for (int k0 = 0; k0 < ns; k0 += BS) {
    const int k1 = std::min(ns, k0 + BS);
    // factor diagonal block and the panel below it (rows k0..nf-1, cols k0..k1-1)
    for (int k = k0; k < k1; ++k) {
      double d = F[(size_t)k * nf + k];
      for (int t = k0; t < k; ++t) d -= F[(size_t)k * nf + t] * F[(size_t)k * nf + t];
      if (!(d > 0.0)) throw std::runtime_error("Cholesky: matrix not positive definite (pivot " + std::to_string(d) + ")");
      d = std::sqrt(d);
      F[(size_t)k * nf + k] = d;
      const double inv = 1.0 / d;
#pragma omp parallel for schedule(static) if (nf - k > 2048)
      for (int i = k + 1; i < nf; ++i) {
        double s = F[(size_t)i * nf + k];
        const double* Li = &F[(size_t)i * nf];
        const double* Lk = &F[(size_t)k * nf];
        for (int t = k0; t < k; ++t) s -= Li[t] * Lk[t];
        F[(size_t)i * nf + k] = s * inv;
      }
    }
    // trailing update of rows/cols >= k1 with the panel columns [k0, k1)
    const int nt = nf - k1;
    if (nt <= 0) continue;
    const int pw = k1 - k0;
    flops += (double)nt * nt * pw;
    trailing_update(F, nf, k0, k1, pw);
  }
}

// Inverse of a lower-triangular n x n block stored with leading dimension ld.
// Blocked: each column block J of X = L^{-1} is independent; row block I of it
// is L_II^{-1} (delta_IJ - sum_{J<=K<I} L_IK X_KJ), computed with contiguous
// row segments.
void lower_inverse(const double* L, int n, int ld, double* X) {
  const int B = 32;
  const int nbk = (n + B - 1) / B;
#pragma omp parallel for schedule(static) if (n > 256)
  for (size_t t = 0; t < (size_t)n * n; ++t) X[t] = 0.0;
#pragma omp parallel for schedule(dynamic, 1) if (n > 128)
  for (int jb = 0; jb < nbk; ++jb) {
    const int j0 = jb * B, j1 = std::min(n, j0 + B), w = j1 - j0;
    double T[32];
    for (int i = j0; i < n; ++i) {
      // T = delta_i - sum_{t in [j0, i)} L[i][t] X[t][j0:j1]
      for (int c = 0; c < w; ++c) T[c] = (i == j0 + c) ? 1.0 : 0.0;
      const double* Li = &L[(size_t)i * ld];
      for (int t = j0; t < i; ++t) {
        const double l = Li[t];
        if (l == 0.0) continue;
        const double* Xt = &X[(size_t)t * n + j0];
#pragma omp simd
        for (int c = 0; c < 32; ++c)
          if (c < w) T[c] -= l * Xt[c];
      }
      const double inv = 1.0 / Li[i];
      double* Xi = &X[(size_t)i * n + j0];
      for (int c = 0; c < w; ++c) Xi[c] = (j0 + c <= i) ? T[c] * inv : 0.0;
    }
  }
}

}  // namespace

namespace {

// Levels of a postordered tree: height above the lowest leaf below.
std::vector<int> tree_levels(const std::vector<NDNode>& nodes, int& nlevels) {
  std::vector<int> lv(nodes.size(), 0);
  nlevels = 0;
  for (size_t s = 0; s < nodes.size(); ++s) {
    for (int c : nodes[s].children) lv[s] = std::max(lv[s], lv[c] + 1);
    nlevels = std::max(nlevels, lv[s] + 1);
  }
  return lv;
}

// Positions of the DoFs in the postordered nodes, and every node's struct
// rows: the DoFs after the node that it or its descendants couple to
// (positions, ascending).  Nodes of one level are independent.
void structure(const DofGraph& G, const std::vector<NDNode>& nodes, std::vector<int>& pos,
               std::vector<int>& p1, std::vector<std::vector<int>>& st) {
  const int nn = (int)nodes.size();
  pos.assign(G.n, -1);
  p1.assign(nn, 0);
  int p = 0;
  for (int s = 0; s < nn; ++s) {
    for (int d : nodes[s].dofs) pos[d] = p++;
    p1[s] = p;
  }
  int nl = 0;
  const std::vector<int> lv = tree_levels(nodes, nl);
  std::vector<std::vector<int>> by(nl);
  for (int s = 0; s < nn; ++s) by[lv[s]].push_back(s);
  st.assign(nn, {});
  for (int l = 0; l < nl; ++l) {
#pragma omp parallel for schedule(dynamic, 4)
    for (size_t i = 0; i < by[l].size(); ++i) {
      const int s = by[l][i];
      std::vector<int>& r = st[s];
      // (sorted, not marked in an array over all DoFs, of which every thread
      // would hold one; neighbours have most rows in common, so that a small
      // table of recent ones keeps most repeats out)
      int recent[1024];
      std::fill(recent, recent + 1024, -1);
      auto consider = [&](int q) {
        if (q < p1[s] || recent[q & 1023] == q) return;
        recent[q & 1023] = q;
        r.push_back(q);
      };
      for (int d : nodes[s].dofs)
        for (int64_t q = G.ptr[d]; q < G.ptr[d + 1]; ++q) consider(pos[G.adj[q]]);
      for (int c : nodes[s].children)
        for (int q : st[c]) consider(q);
      std::sort(r.begin(), r.end());
      r.erase(std::unique(r.begin(), r.end()), r.end());
      r.shrink_to_fit();
    }
  }
}

// Merge runs of adjacent tree levels.  A run [a, b] becomes one level: every
// node in it whose parent lies above b absorbs its descendants of levels a..b.
// The runs minimise the sum over levels of cost.level + cost.entry * stored
// entries + cost.row * front rows, by dynamic programming over the levels.
std::vector<NDNode> merge_levels(const std::vector<NDNode>& nodes, const std::vector<std::vector<int>>& st,
                                 const SolveCost& cost) {
  const int nn = (int)nodes.size();
  int nl = 0;
  const std::vector<int> lv = tree_levels(nodes, nl);
  std::vector<double> best(nl + 1, 0.0);
  std::vector<int> from(nl + 1, 0);
  std::vector<std::vector<double>> run(nl, std::vector<double>(nl, 0.0));  // [a][b]
#pragma omp parallel for schedule(dynamic, 1)
  for (int a = 0; a < nl; ++a) {
    std::vector<double> own(nn, 0.0);  // DoFs of levels >= a in the subtree
    for (int s = 0; s < nn; ++s) {
      if (lv[s] < a) continue;
      own[s] += (double)nodes[s].dofs.size();
      if (nodes[s].parent >= 0) own[nodes[s].parent] += own[s];
      const int up = nodes[s].parent >= 0 ? lv[nodes[s].parent] : nl;  // s is a run's root for lv <= b < up
      const double n = own[s], m = (double)st[s].size();
      const double c = cost.entry * (0.5 * n * (n + 1.0) + m * n) + cost.row * (n + m);
      for (int b = lv[s]; b < up; ++b) run[a][b] += c;
    }
  }
  for (int b = 0; b < nl; ++b) {
    best[b + 1] = -1.0;
    for (int a = 0; a <= b; ++a) {
      const double c = best[a] + cost.level + run[a][b];
      if (best[b + 1] < 0 || c < best[b + 1]) {
        best[b + 1] = c;
        from[b + 1] = a;
      }
    }
  }
  std::vector<int> group(nl, 0);
  for (int b = nl; b > 0; b = from[b])
    for (int l = from[b]; l < b; ++l) group[l] = b;
  // roots of the runs, in postorder, with their members' DoFs in postorder
  std::vector<NDNode> out;
  std::vector<int> root(nn), id(nn, -1);
  for (int s = nn; s-- > 0;) {
    const int pa = nodes[s].parent;
    root[s] = (pa >= 0 && group[lv[pa]] == group[lv[s]]) ? root[pa] : s;
  }
  std::vector<std::vector<int>> members(nn);
  for (int s = 0; s < nn; ++s) members[root[s]].push_back(s);
  for (int s = 0; s < nn; ++s) {
    if (root[s] != s) continue;
    NDNode m;
    for (int t : members[s]) {
      m.dofs.insert(m.dofs.end(), nodes[t].dofs.begin(), nodes[t].dofs.end());
      for (int c : nodes[t].children)
        if (root[c] == c) m.children.push_back(id[c]);
    }
    id[s] = (int)out.size();
    for (int c : m.children) out[c].parent = id[s];
    out.push_back(std::move(m));
  }
  return out;
}

// Ordering, supernodes, row structure and levels (no numeric values).
SupernodalFactor symbolic(const Systems& S, const DofGraph& G, int leaf_cells, const SolveCost& cost) {
  std::vector<NDNode> nodes;
  for (size_t k = 0; k < S.size(); ++k)
    NDBuilder(*S[k], G, (int)k, leaf_cells, nodes).build(0, S[k]->NXc, 0, S[k]->NYc);
  SupernodalFactor F;
  std::vector<int> p1;
  std::vector<std::vector<int>> st;
  structure(G, nodes, F.perm, p1, st);
  if (cost.level > 0) {
    nodes = merge_levels(nodes, st, cost);
    structure(G, nodes, F.perm, p1, st);
  }
  const int nn = (int)nodes.size();
  F.n = G.n;
  for (const std::vector<int>& d : G.dof0) {
    F.sys_p0.push_back(d.front());
    F.cell_dof0.emplace_back(d.begin(), d.end() - 1);
  }
  F.sys_p0.push_back(G.n);
  F.sys_node0.assign(S.size() + 1, nn);
  for (int s = nn; s-- > 0;)
    if (!nodes[s].dofs.empty()) F.sys_node0[G.sys[nodes[s].dofs[0]]] = s;
  for (size_t k = S.size(); k-- > 0;) F.sys_node0[k] = std::min(F.sys_node0[k], F.sys_node0[k + 1]);
  const std::vector<int> lv = tree_levels(nodes, F.nlevels);
  F.level_nodes.assign(F.nlevels, {});
  F.nodes.resize(nn);
  F.children.resize(nn);
  int64_t linv = 0, l21 = 0, rows = 0;
  for (int s = 0; s < nn; ++s) {
    SNode& N = F.nodes[s];
    N.ns = (int)nodes[s].dofs.size();
    N.p0 = p1[s] - N.ns;
    N.ms = (int)st[s].size();
    N.parent = nodes[s].parent;
    N.level = lv[s];
    F.level_nodes[lv[s]].push_back(s);
    F.children[s] = nodes[s].children;
    N.linv_off = linv;
    N.l21_off = l21;
    N.rows_off = rows;
    linv += (int64_t)N.ns * N.ns;
    l21 += (int64_t)N.ms * N.ns;
    rows += N.ms;
  }
  F.rows.resize(rows);
  for (int s = 0; s < nn; ++s) std::copy(st[s].begin(), st[s].end(), F.rows.begin() + F.nodes[s].rows_off);
  F.linv_size = linv;
  F.l21_size = l21;
  // forward contribution lists
  std::vector<int64_t> cnt(F.n + 1, 0);
  for (int s = 0; s < nn; ++s)
    for (int r = 0; r < F.nodes[s].ms; ++r) cnt[F.rows[F.nodes[s].rows_off + r] + 1]++;
  for (int i = 0; i < F.n; ++i) cnt[i + 1] += cnt[i];
  F.contrib_ptr = cnt;
  F.contrib_node.assign(cnt[F.n], 0);
  F.contrib_row.assign(cnt[F.n], 0);
  std::vector<int64_t> fill(cnt.begin(), cnt.end() - 1);
  for (int s = 0; s < nn; ++s)
    for (int r = 0; r < F.nodes[s].ms; ++r) {
      const int pp = F.rows[F.nodes[s].rows_off + r];
      F.contrib_node[fill[pp]] = s;
      F.contrib_row[fill[pp]] = r;
      fill[pp]++;
    }
  return F;
}

// Positions of child c's struct rows in its parent's front (own rows, then
// struct rows; both lists ascend).
std::vector<int> child_map(const SupernodalFactor& F, int c) {
  const SNode& C = F.nodes[c];
  const SNode& N = F.nodes[C.parent];
  std::vector<int> m(C.ms);
  int j = 0;
  for (int r = 0; r < C.ms; ++r) {
    const int q = F.rows[C.rows_off + r];
    if (q < N.p0 + N.ns) {
      m[r] = q - N.p0;
    } else {
      while (j < N.ms && F.rows[N.rows_off + j] < q) ++j;
      if (j == N.ms || F.rows[N.rows_off + j] != q) throw std::runtime_error("child_map: a child row is not in the parent");
      m[r] = N.ns + j;
    }
    if (m[r] < 0) throw std::runtime_error("child_map: a child row precedes the parent");
  }
  return m;
}

}  // namespace

SupernodalFactor cholesky_factor(const Systems& Ss, int leaf_cells, const SolveCost& cost,
                                 const std::vector<int>& twin) {
  const DofGraph G(Ss, twin);
  SupernodalFactor F = symbolic(Ss, G, leaf_cells, cost);
  const int nn = (int)F.nodes.size();
  std::vector<int> dof_at(F.n);  // permuted index -> DoF
  for (int d = 0; d < F.n; ++d) dof_at[F.perm[d]] = d;
  F.Linv.assign(F.linv_size, 0.0);
  F.L21.assign(F.l21_size, 0.0);
  // numeric multifrontal factorisation, level by level on the elimination tree:
  // nodes of one level are independent (their children are in lower levels).
  std::vector<std::vector<double>> upd(nn);
  const int nthreads = omp_get_max_threads();
  std::vector<double> flops_t(nthreads, 0.0), ta_t(nthreads, 0.0), tf_t(nthreads, 0.0), ti_t(nthreads, 0.0);
  std::vector<int64_t> lost_t(nthreads, 0);  // entries outside their fronts
  auto process = [&](int s, int tid) {
    const SNode& N = F.nodes[s];
    const int ns = N.ns, ms = N.ms, nf = ns + ms;
    const bool big = nf > 1024;
    auto tA = std::chrono::steady_clock::now();
    std::vector<double> Fr((size_t)nf * nf);
#pragma omp parallel for schedule(static) if (big)
    for (int r = 0; r < nf; ++r) std::fill(&Fr[(size_t)r * nf], &Fr[(size_t)r * nf] + r + 1, 0.0);
    // original entries (p, q), p own and p <= q, into column p
    for (int c = 0; c < ns; ++c) {
      const int d = dof_at[N.p0 + c], X = G.cell[d];
      const BlockSPD& S = *Ss[G.sys[d]];
      const std::vector<int>& dof0 = G.dof0[G.sys[d]];
      const int a = d - dof0[X], no = S.noff();
      const int xi = X % S.NXc, xj = X / S.NXc;
      for (int o = 0; o < no; ++o) {
        const int yi = xi + S.offi[o], yj = xj + S.offj[o];
        if (yi < 0 || yi >= S.NXc || yj < 0 || yj >= S.NYc) continue;
        const int Y = yi + S.NXc * yj, ny = S.ndof[Y];
        const auto& B = S.blk[(size_t)X * no + o];
        if (B.empty()) continue;
        for (int b = 0; b < ny; ++b) {
          const double v = B[(size_t)a * ny + b];
          const int q = F.perm[dof0[Y] + b];
          if (v == 0.0 || q < N.p0 + c) continue;
          const int r = front_row(q, N.p0, ns, ms, F.rows.data() + N.rows_off);
          if (r < 0) {
            ++lost_t[tid];
            continue;
          }
          Fr[(size_t)r * nf + c] += v;
        }
      }
    }
    // extend-add children
    for (int c : F.children[s]) {
      const int mc = F.nodes[c].ms;
      const std::vector<int> map = child_map(F, c);
      const std::vector<double>& U = upd[c];
#pragma omp parallel for schedule(dynamic, 64) if (big)
      for (int r = 0; r < mc; ++r) {
        double* row = &Fr[(size_t)map[r] * nf];
        const double* ur = &U[(size_t)r * mc];
        for (int q = 0; q <= r; ++q) row[map[q]] += ur[q];
      }
      std::vector<double>().swap(upd[c]);
    }
    auto tB = std::chrono::steady_clock::now();
    if (ns > 0) partial_cholesky(Fr.data(), nf, ns, flops_t[tid]);
    flops_t[tid] += (double)ns * ns * ns / 3.0;
    auto tC = std::chrono::steady_clock::now();
    // store Linv, L21 and the update matrix
    if (ns > 0) lower_inverse(Fr.data(), ns, nf, &F.Linv[N.linv_off]);
    auto tD = std::chrono::steady_clock::now();
    ta_t[tid] += std::chrono::duration<double>(tB - tA).count();
    tf_t[tid] += std::chrono::duration<double>(tC - tB).count();
    ti_t[tid] += std::chrono::duration<double>(tD - tC).count();
#pragma omp parallel for schedule(static) if (big)
    for (int r = 0; r < ms; ++r)
      for (int c2 = 0; c2 < ns; ++c2) F.L21[N.l21_off + (int64_t)r * ns + c2] = Fr[(size_t)(ns + r) * nf + c2];
    if (ms > 0) {
      upd[s].resize((size_t)ms * ms);
#pragma omp parallel for schedule(static) if (big)
      for (int r = 0; r < ms; ++r)
        for (int q = 0; q <= r; ++q) upd[s][(size_t)r * ms + q] = Fr[(size_t)(ns + r) * nf + ns + q];
    }
  };
  for (int l = 0; l < F.nlevels; ++l) {
    const std::vector<int>& lv = F.level_nodes[l];
    if ((int)lv.size() >= 2 * nthreads) {
#pragma omp parallel for schedule(dynamic, 1)
      for (int i = 0; i < (int)lv.size(); ++i) process(lv[i], omp_get_thread_num());
    } else {
      for (int s : lv) process(s, 0);
    }
  }
  for (int t = 0; t < nthreads; ++t) {
    if (lost_t[t]) throw std::runtime_error("cholesky_factor: an entry outside its front");
    F.flops += flops_t[t];
    F.t_assemble += ta_t[t];
    F.t_factor += tf_t[t];
    F.t_inverse += ti_t[t];
  }
  return F;
}

SupernodalFactor cholesky_symbolic(const Systems& Ss, int leaf_cells, FrontPlan& plan, const SolveCost& cost,
                                   const std::vector<int>& twin) {
  const DofGraph G(Ss, twin);
  SupernodalFactor F = symbolic(Ss, G, leaf_cells, cost);
  const int nn = (int)F.nodes.size();
  plan = FrontPlan{};
  plan.nlevels = F.nlevels;
  // S blocks
  for (size_t k = 0; k < Ss.size(); ++k) {
    const BlockSPD& S = *Ss[k];
    const int NG = S.NXc * S.NYc, no = S.noff();
    for (int X = 0; X < NG; ++X)
      for (int o = 0; o < no; ++o) {
        const auto& B = S.blk[(size_t)X * no + o];
        if (B.empty()) continue;
        const int Y = X + S.offi[o] + S.NXc * S.offj[o];
        if (S.ndof[X] == 0 || S.ndof[Y] == 0) continue;
        plan.sb_val.push_back(B.data());
        plan.sb_src.push_back(plan.nvals);
        plan.sb_x.push_back(G.dof0[k][X]);
        plan.sb_y.push_back(G.dof0[k][Y]);
        plan.sb_nx.push_back(S.ndof[X]);
        plan.sb_ny.push_back(S.ndof[Y]);
        plan.nvals += (int64_t)B.size();
      }
  }
  plan.node_of.resize(F.n);
  for (int s = 0; s < nn; ++s)
    std::fill_n(plan.node_of.begin() + F.nodes[s].p0, F.nodes[s].ns, s);
  // fronts, level by level (each level's fronts contiguous)
  plan.front_off.assign(nn, 0);
  plan.level_front.assign(F.nlevels + 1, 0);
  int64_t fo = 0;
  for (int l = 0; l < F.nlevels; ++l) {
    plan.level_front[l] = fo;
    for (int s : F.level_nodes[l]) {
      const int64_t nf = F.nodes[s].ns + F.nodes[s].ms;
      plan.front_off[s] = fo;
      fo += nf * nf;
    }
  }
  plan.level_front[F.nlevels] = fo;
  plan.front_total = fo;
  // child row maps into the parent's front
  plan.ea_map_off.assign(nn + 1, 0);
  for (int s = 0; s < nn; ++s)
    plan.ea_map_off[s + 1] = plan.ea_map_off[s] + (F.nodes[s].parent >= 0 ? F.nodes[s].ms : 0);
  plan.ea_map.resize(plan.ea_map_off[nn]);
  for (int s = 0; s < nn; ++s) {
    if (F.nodes[s].parent < 0) continue;
    const std::vector<int> m = child_map(F, s);
    std::copy(m.begin(), m.end(), plan.ea_map.begin() + plan.ea_map_off[s]);
  }
  // extend-add rows, per parent level and pass (child i of every parent)
  size_t kids = 0;
  for (int s = 0; s < nn; ++s) kids = std::max(kids, F.children[s].size());
  plan.npass = (int)kids;
  plan.ea_level.assign((size_t)plan.npass * F.nlevels + 1, 0);
  for (int l = 0; l < F.nlevels; ++l)
    for (int pass = 0; pass < plan.npass; ++pass) {
      plan.ea_level[(size_t)plan.npass * l + pass] = (int)plan.ea_child.size();
      for (int s : F.level_nodes[l]) {
        if ((int)F.children[s].size() <= pass) continue;
        const int c = F.children[s][pass];
        for (int r = 0; r < F.nodes[c].ms; ++r) {
          plan.ea_child.push_back(c);
          plan.ea_row.push_back(r);
          plan.ea_parent.push_back(s);
        }
      }
    }
  plan.ea_level[(size_t)plan.npass * F.nlevels] = (int)plan.ea_child.size();
  return F;
}

void copy_blocks(const FrontPlan& plan, size_t i0, size_t i1, double* dst) {
#pragma omp parallel for schedule(static)
  for (size_t i = i0; i < i1; ++i)
    std::copy_n(plan.sb_val[i], plan.sb_nx[i] * plan.sb_ny[i], dst + (plan.sb_src[i] - plan.sb_src[i0]));
}

void execute_plan_host(const FrontPlan& plan, const SupernodalFactor& F, std::vector<double>& Linv,
                       std::vector<double>& L21) {
  const int nn = (int)F.nodes.size();
  std::vector<double> fr(plan.front_total, 0.0);
  Linv.assign(F.linv_size, 0.0);
  L21.assign(F.l21_size, 0.0);
  double flops = 0.0;
  for (size_t i = 0; i < plan.sb_src.size(); ++i)
    for (int a = 0; a < plan.sb_nx[i]; ++a)
      for (int b = 0; b < plan.sb_ny[i]; ++b) {
        const double v = plan.sb_val[i][a * plan.sb_ny[i] + b];
        const int p = F.perm[plan.sb_x[i] + a], q = F.perm[plan.sb_y[i] + b];
        if (v == 0.0 || q < p) continue;
        const int s = plan.node_of[p];
        const SNode& N = F.nodes[s];
        const int r = front_row(q, N.p0, N.ns, N.ms, F.rows.data() + N.rows_off);
        if (r < 0) throw std::runtime_error("execute_plan_host: an entry outside its front");
        fr.at(plan.front_off[s] + (int64_t)r * (N.ns + N.ms) + (p - N.p0)) += v;
      }
  for (int l = 0; l < F.nlevels; ++l) {
    for (int pass = 0; pass < plan.npass; ++pass)
      for (int i = plan.ea_level[(size_t)plan.npass * l + pass]; i < plan.ea_level[(size_t)plan.npass * l + pass + 1];
           ++i) {
        const int c = plan.ea_child[i], r = plan.ea_row[i], s = plan.ea_parent[i];
        const int nsc = F.nodes[c].ns, nfc = nsc + F.nodes[c].ms, nfp = F.nodes[s].ns + F.nodes[s].ms;
        const int* m = &plan.ea_map[plan.ea_map_off[c]];
        for (int q = 0; q <= r; ++q)
          fr.at(plan.front_off[s] + (int64_t)m[r] * nfp + m[q]) +=
              fr.at(plan.front_off[c] + (int64_t)(nsc + r) * nfc + nsc + q);
      }
    for (int s : F.level_nodes[l]) {
      const SNode& N = F.nodes[s];
      const int nf = N.ns + N.ms;
      double* Fr = &fr[plan.front_off[s]];
      if (N.ns > 0) {
        partial_cholesky(Fr, nf, N.ns, flops);
        lower_inverse(Fr, N.ns, nf, &Linv[N.linv_off]);
      }
      for (int r = 0; r < N.ms; ++r)
        for (int c2 = 0; c2 < N.ns; ++c2) L21[N.l21_off + (int64_t)r * N.ns + c2] = Fr[(size_t)(N.ns + r) * nf + c2];
    }
  }
  (void)nn;
}

PackedFactor pack_layout(const SupernodalFactor& F) {
  PackedFactor P;
  const int nn = (int)F.nodes.size();
  P.n = F.n;
  P.nlevels = F.nlevels;
  P.nsys = F.nsys();
  P.sys_p0 = F.sys_p0;
  P.sys_node0 = F.sys_node0;
  P.cell_dof0 = F.cell_dof0;
  P.perm = F.perm;
  P.tri_bytes.assign(P.nsys, 0.0);
  const int K = P.nsys;
  int sys = 0;
  P.p0.resize(nn);
  P.ns.resize(nn);
  P.ms.resize(nn);
  P.fwd_off.resize(nn);
  P.bwd_off.resize(nn);
  P.rows_off.resize(nn);
  P.z_off.resize(nn);
  int64_t nf = 0, zl = 0;
  for (int s = 0; s < nn; ++s) {
    P.p0[s] = F.nodes[s].p0;
    P.ns[s] = F.nodes[s].ns;
    P.ms[s] = F.nodes[s].ms;
    P.rows_off[s] = F.nodes[s].rows_off;
    const int64_t n_ = P.ns[s], m_ = P.ms[s];
    P.fwd_off[s] = nf;
    P.bwd_off[s] = nf;
    P.z_off[s] = zl;
    nf += n_ * (n_ + 1) / 2 + m_ * n_;
    zl += m_;
    while (s >= F.sys_node0[sys + 1]) ++sys;
    P.tri_bytes[sys] += 2.0 * 8.0 * (0.5 * n_ * (n_ + 1.0) + (double)m_ * n_);
  }
  P.zlen = zl;
  P.nvals = nf;
  // lanes per row: the smallest power of two >= an eighth of the mean row length
  auto lanes = [](double mean) {
    int w = 8;
    while (w < 64 && w * 8 < mean) w *= 2;
    return w;
  };
  P.goff.assign(F.nlevels * K + 1, 0);
  P.xoff.assign(F.nlevels * K + 1, 0);
  P.fw.assign(F.nlevels, 64);
  P.bw.assign(F.nlevels, 64);
  P.fm.assign(F.nlevels, 1);
  P.bm.assign(F.nlevels, 1);
  P.fpf.assign(F.nlevels, 0);
  P.bpf.assign(F.nlevels, 0);
  P.frows.assign(F.nlevels, 4);
  P.brows.assign(F.nlevels, 4);
  P.lnoff.assign(F.nlevels * K + 1, 0);
  for (int l = 0; l < F.nlevels; ++l) {
    double fl = 0, fr = 0, bl = 0, br = 0;
    for (int s : F.level_nodes[l]) {
      const double n_ = P.ns[s], m_ = P.ms[s];
      fl += 0.5 * n_ * (n_ + 1) + m_ * n_;
      fr += n_ + m_;
      bl += 0.5 * n_ * (n_ + 1) + m_ * n_;
      br += n_;
    }
    P.fw[l] = lanes(fr > 0 ? fl / fr : 1);
    P.bw[l] = lanes(br > 0 ? bl / br : 1);
    // tile height: at most sweep_tile_rows(W), smaller on levels with few rows
    // so that each level still spreads over many workgroups
    auto height = [](int w, double nrows) {
      int h = sweep_tile_rows(w);
      const int pass = 256 / w;
      while (h > pass && nrows / h < 8192) h /= 2;
      return h;
    };
    P.frows[l] = height(P.fw[l], fr);
    P.brows[l] = height(P.bw[l], br);
    P.fm[l] = std::max(1, P.frows[l] / (256 / P.fw[l]));
    P.bm[l] = std::max(1, P.brows[l] / (256 / P.bw[l]));
    size_t i = 0;  // (a level's nodes ascend, so its systems follow each other)
    for (int k = 0; k < K; ++k) {
      P.goff[l * K + k] = (int)P.lrows.size();
      P.xoff[l * K + k] = (int)P.xidx.size();
      P.lnoff[l * K + k] = (int)P.lnodes.size();
      for (; i < F.level_nodes[l].size() && F.level_nodes[l][i] < F.sys_node0[k + 1]; ++i) {
        const int s = F.level_nodes[l][i];
        P.lnodes.push_back(s);
        for (int r = 0; r < P.ns[s]; ++r) P.lrows.push_back(P.p0[s] + r);
        for (int j = 0; j < P.ms[s]; ++j) P.xidx.push_back(P.rows_off[s] + j);
      }
    }
  }
  P.goff[F.nlevels * K] = (int)P.lrows.size();
  P.xoff[F.nlevels * K] = (int)P.xidx.size();
  P.lnoff[F.nlevels * K] = (int)P.lnodes.size();
  rebuild_tiles(P);
  P.rows = F.rows;
  P.cptr = F.contrib_ptr;
  // the solves read the leaf level's right-hand side without a gather
  for (int q = P.goff[0]; q < P.goff[K]; ++q)
    if (P.cptr[P.lrows[q] + 1] != P.cptr[P.lrows[q]])
      throw std::runtime_error("pack_layout: a leaf-level row is owed contributions");
  P.czidx.resize(F.contrib_node.size());
  for (size_t t = 0; t < P.czidx.size(); ++t) P.czidx[t] = P.z_off[F.contrib_node[t]] + F.contrib_row[t];
  return P;
}

void pack_values(const SupernodalFactor& F, PackedFactor& P) {
  const int nn = (int)P.p0.size();
  P.fwd.assign(P.nvals, 0.0);
  P.bwd.assign(P.nvals, 0.0);
#pragma omp parallel for schedule(dynamic, 1)
  for (int s = 0; s < nn; ++s) {
    const int n_ = P.ns[s], m_ = P.ms[s];
    const double* Li = &F.Linv[F.nodes[s].linv_off];
    const double* L21 = &F.L21[F.nodes[s].l21_off];
    double* f = &P.fwd[P.fwd_off[s]];
    for (int r = 0; r < n_; ++r)
      for (int j = 0; j <= r; ++j) f[(int64_t)r * (r + 1) / 2 + j] = Li[(int64_t)r * n_ + j];
    // W21 = L21 Linv, 8 panel rows at a time so each Linv row is reused
    double* W = f + (int64_t)n_ * (n_ + 1) / 2;
    for (int i0 = 0; i0 < m_; i0 += 8) {
      const int i1 = std::min(m_, i0 + 8);
      for (int k = 0; k < n_; ++k) {
        const double* Lk = Li + (int64_t)k * n_;
        for (int i = i0; i < i1; ++i) {
          const double a = L21[(int64_t)i * n_ + k];
          if (a == 0.0) continue;
          double* Wi = W + (int64_t)i * n_;
#pragma omp simd
          for (int j = 0; j <= k; ++j) Wi[j] += a * Lk[j];
        }
      }
    }
    double* bw = &P.bwd[P.bwd_off[s]];
    for (int j = 0; j < n_; ++j) {
      double* row = bw + (int64_t)j * (n_ + m_) - (int64_t)j * (j - 1) / 2;
      for (int i = j; i < n_; ++i) row[i - j] = Li[(int64_t)i * n_ + j];
      for (int i = 0; i < m_; ++i) row[n_ - j + i] = -W[(int64_t)i * n_ + j];
    }
  }
}

PackedFactor pack_factor(const SupernodalFactor& F) {
  PackedFactor P = pack_layout(F);
  pack_values(F, P);
  return P;
}

void blocked_layout(PackedFactor& P) {
  const int nn = (int)P.p0.size();
  for (int dir = 0; dir < 2; ++dir) {
    const bool fwd = dir == 0;
    std::vector<int>& b0 = fwd ? P.fblk0 : P.bblk0;
    std::vector<int64_t>& boff = fwd ? P.fblk_off : P.bblk_off;
    b0.assign(nn + 1, 0);
    boff.clear();
    int64_t total = 0;
    for (int s = 0; s < nn; ++s) {
      b0[s] = (int)boff.size();
      const int rows = fwd ? P.ns[s] + P.ms[s] : P.ns[s];
      for (int b = 0; b * 16 < rows; ++b) {
        boff.push_back(total);
        const int nsteps = (blk_chi(fwd, b, P.ns[s], P.ms[s]) - blk_clo(fwd, b) + 15) / 16;
        total += (int64_t)nsteps * 256;
      }
    }
    b0[nn] = (int)boff.size();
    boff.push_back(total);
  }
}

void pack_blocked(PackedFactor& P) {
  const int nn = (int)P.p0.size();
  blocked_layout(P);
  for (int dir = 0; dir < 2; ++dir) {
    const bool fwd = dir == 0;
    const std::vector<int>& b0 = fwd ? P.fblk0 : P.bblk0;
    const std::vector<int64_t>& boff = fwd ? P.fblk_off : P.bblk_off;
    std::vector<double>& dst = fwd ? P.fblk : P.bblk;
    dst.assign(boff.back(), 0.0);
    const std::vector<double>& src = fwd ? P.fwd : P.bwd;
#pragma omp parallel for schedule(dynamic, 1)
    for (int s = 0; s < nn; ++s) {
      const int ns = P.ns[s], ms = P.ms[s];
      const int rows = fwd ? ns + ms : ns;
      const int64_t base = fwd ? P.fwd_off[s] : P.bwd_off[s];
      for (int b = 0; b * 16 < rows; ++b) {
        const int clo = blk_clo(fwd, b), chi = blk_chi(fwd, b, ns, ms);
        const int nsteps = (chi - clo + 15) / 16;
        double* d = &dst[boff[b0[s] + b]];
        for (int i = 0; i < 16; ++i) {
          const int lr = 16 * b + i;
          if (lr >= rows) continue;
          int64_t off;
          int rs, re;
          if (fwd) {
            rs = 0;
            if (lr < ns) {
              off = (int64_t)lr * (lr + 1) / 2;
              re = lr + 1;
            } else {
              off = (int64_t)ns * (ns + 1) / 2 + (int64_t)(lr - ns) * ns;
              re = ns;
            }
          } else {
            off = (int64_t)lr * (ns + ms) - (int64_t)lr * (lr - 1) / 2 - lr;
            rs = lr;
            re = ns + ms;
          }
          for (int st = 0; st < nsteps; ++st)
            for (int k = 0; k < 4; ++k)
              for (int q = 0; q < 4; ++q) {
                const int col = clo + 16 * st + 4 * k + q;
                if (col >= rs && col < re) d[((int64_t)st * 4 + q) * 64 + i + 16 * k] = src[base + off + col];
              }
        }
      }
    }
  }
  std::vector<double>().swap(P.fwd);
  std::vector<double>().swap(P.bwd);
}

bool level_tiles_split(const PackedFactor& P, int l, bool fwd, int rows, int ks, std::vector<int>& tiles,
                       std::vector<int>& rtiles, int sys, int t_base) {
  if (rows < 1) throw std::runtime_error("level_tiles: rows must be >= 1");
  if (ks > 0 && ks % 16 != 0) throw std::runtime_error("level_tiles_split: segment length must be a multiple of 16");
  if (t_base < 0) t_base = (int)(tiles.size() / 4);
  const int q0 = P.lnoff[l * P.nsys + std::max(sys, 0)], q1 = P.lnoff[sys < 0 ? (l + 1) * P.nsys : l * P.nsys + sys + 1];
  for (int q = q0; q < q1; ++q) {
    const int s = P.lnodes[q];
    const int ns = P.ns[s], ms = P.ms[s];
    const int nr = fwd ? ns + ms : ns;
    for (int r0 = 0; r0 < nr; r0 += rows) {
      const int n = std::min(rows, nr - r0);
      if (ks <= 0) {
        tiles.insert(tiles.end(), {s, r0, n, -1});
        continue;
      }
      const int last = r0 + n - 1;
      // columns the row tile touches: forward [0, longest row), backward [r0, ns + ms)
      const int cbeg = fwd ? 0 : r0;
      const int cend = fwd ? (last < ns ? last + 1 : ns) : ns + ms;
      const int k0 = cbeg / ks, k1 = (cend + ks - 1) / ks;
      if (k1 - k0 > 63) return false;
      const int t0 = (int)(tiles.size() / 4) - t_base;
      for (int k = k0; k < k1; ++k) tiles.insert(tiles.end(), {s, r0, n, k});
      rtiles.insert(rtiles.end(), {s, r0, n, 64 * t0 + (k1 - k0)});
    }
  }
  return true;
}

void rebuild_tiles(PackedFactor& P) {
  P.ftiles.clear();
  P.btiles.clear();
  P.frtiles.clear();
  P.brtiles.clear();
  const int K = P.nsys;
  P.foff.assign(P.nlevels * K + 1, 0);
  P.boff.assign(P.nlevels * K + 1, 0);
  P.froff.assign(P.nlevels * K + 1, 0);
  P.broff.assign(P.nlevels * K + 1, 0);
  if ((int)P.fks.size() != P.nlevels) P.fks.assign(P.nlevels, 0);
  if ((int)P.bks.size() != P.nlevels) P.bks.assign(P.nlevels, 0);
  for (int l = 0; l < P.nlevels; ++l) {
    // lanes per row W > 0: (256 / W) * MAXR rows per tile; W <= 0 (the MFMA
    // sweep): at most 64 * MAXR rows per tile (fewer with its right-hand
    // sides split over waves, W == -1); only the MFMA sweep splits columns
    auto cap = [](int w, int m) { return w > 0 ? (256 / w) * m : 64 * m; };
    if (P.frows[l] > cap(P.fw[l], P.fm[l]) || P.brows[l] > cap(P.bw[l], P.bm[l]))
      throw std::runtime_error("rebuild_tiles: tile height exceeds the rows one workgroup covers");
    if ((P.fks[l] && P.fw[l] > 0) || (P.bks[l] && P.bw[l] > 0))
      throw std::runtime_error("rebuild_tiles: only the MFMA sweep splits columns");
    const int ft = (int)(P.ftiles.size() / 4), bt = (int)(P.btiles.size() / 4);
    for (int k = 0; k < K; ++k) {
      P.foff[l * K + k] = (int)(P.ftiles.size() / 4);
      P.boff[l * K + k] = (int)(P.btiles.size() / 4);
      P.froff[l * K + k] = (int)(P.frtiles.size() / 4);
      P.broff[l * K + k] = (int)(P.brtiles.size() / 4);
      if (!level_tiles_split(P, l, true, P.frows[l], P.fks[l], P.ftiles, P.frtiles, k, ft) ||
          !level_tiles_split(P, l, false, P.brows[l], P.bks[l], P.btiles, P.brtiles, k, bt))
        throw std::runtime_error("rebuild_tiles: too many column segments");
    }
  }
  P.foff[P.nlevels * K] = (int)(P.ftiles.size() / 4);
  P.boff[P.nlevels * K] = (int)(P.btiles.size() / 4);
  P.froff[P.nlevels * K] = (int)(P.frtiles.size() / 4);
  P.broff[P.nlevels * K] = (int)(P.brtiles.size() / 4);
}

}  // namespace pecs
