// semx_tree.cpp -- plan and factorisation of the elimination tree
// (semx_tree.h) on the host.  The condensed boundary system of a mode,
// which semtex factorises as one banded Cholesky (MatrixSys::MatrixSys,
// src/matrix.cpp:139-323), is eliminated region by region instead: for a
// region with eliminated unknowns I and boundary unknowns B,
//   A_II^-1,  X = A_BI A_II^-1,  S = A_BB - X A_IB,
// S going to the region it is merged into.  Cholesky throughout, so an
// indefinite system is reported as dpbtrf would.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <numeric>
#include <thread>

#include "semx_internal.h"

namespace semx {

namespace {

// Recursive bisection of the elements.
struct Bis {
  int lo, hi, depth, l = -1, r = -1;
  int nb = 0, sep = 0, cls = -1;
  int hdep = 0;                 // levels below
};

// Splits elements [lo, hi) of perm: along each coordinate direction, the
// cut near the middle that crosses the fewest shared sides; the better of
// the two directions.  Cuts off the middle are charged for the imbalance.
int best_split(std::vector<int>& perm, int lo, int hi, const std::vector<double>& cx,
               const std::vector<double>& cy, const std::vector<std::vector<int>>& adj,
               std::vector<char>& left) {
  const int n = hi - lo;
  double best = -1.0;
  int bestk = 0;
  std::vector<int> bestp, p(n);
  for (int dir = 0; dir < 2; ++dir) {
    const std::vector<double>& a = dir ? cy : cx;
    const std::vector<double>& b = dir ? cx : cy;
    // coordinates equal to rounding count as equal, so that rows and columns
    // of a regular mesh sort as such
    double mn = 1e300, mx = -1e300;
    for (int i = lo; i < hi; ++i) { mn = std::min(mn, a[perm[i]]); mx = std::max(mx, a[perm[i]]); }
    const double tol = 1e-9 * std::max(mx - mn, 1e-300);
    for (int i = 0; i < n; ++i) p[i] = perm[lo + i];
    std::stable_sort(p.begin(), p.end(), [&](int u, int v) {
      const double ku = std::floor((a[u] - mn) / tol + 0.5), kv = std::floor((a[v] - mn) / tol + 0.5);
      if (std::fabs(ku - kv) > 1.0) return ku < kv;
      return b[u] < b[v];
    });
    for (int i = 0; i < n; ++i) left[p[i]] = 1;
    // walk from all-left down: cut(k) = sides between the first k and the rest
    std::vector<int> cut(n + 1, 0);
    for (int k = n; k > 0; --k) {
      const int e = p[k - 1];
      int in = 0, out = 0;
      for (int q : adj[e]) { in += left[q] == 1; out += left[q] == 2; }
      left[e] = 2;
      cut[k - 1] = cut[k] + in - out;
    }
    for (int i = 0; i < n; ++i) left[p[i]] = 0;
    for (int k = std::max(1, n / 3); k <= std::min(n - 1, n - n / 3); ++k) {
      const double imb = std::fabs(2.0 * k - n) / n;
      const double sc = (cut[k] + 0.5) * (1.0 + imb);
      if (best < 0.0 || sc < best * (1.0 - 1e-12)) { best = sc; bestk = k; bestp = p; }
    }
  }
  std::copy(bestp.begin(), bestp.end(), perm.begin() + lo);
  return lo + bestk;
}

struct VecHash {
  std::map<std::vector<int>, int> m;
  int id(const std::vector<int>& k) {
    auto it = m.find(k);
    if (it != m.end()) return it->second;
    const int v = (int)m.size();
    m.emplace(k, v);
    return v;
  }
};

}  // namespace

void tree_plan(Helm& H) {
  Tree& T = H.tree;
  T = Tree();
  const Mesh& M = *H.M;
  int nd = 0;
  bool pinned = false;
  for (const ModeSys& S : H.modes)
    if (S.kind == SEMX_DIRECT) { ++nd; pinned |= S.singular != 0; }
  if (nd == 0 || M.nsolve < 2) return;
  // The tree is faster than the band sweeps were on the systems measured (the
  // figures in semx_tree.hip), but for small meshes with 64 modes, where both
  // are chains of short launches (8x8 np=5 Nz=128 43 against 40 us, 32x3 np=6
  // Nz=64 46 against 44).  So only the sweeps' own switches and SEMX_TREE=0
  // select them -- and systems with a region too large for a workgroup's LDS
  // (below).
  for (const char* v : {"SEMX_AUTOTUNE", "SEMX_BAND_COOP", "SEMX_BAND_XCOOP", "SEMX_BAND_PARTS"})
    if (getenv(v)) return;
  if (const char* e = getenv("SEMX_TREE")) if (atoi(e) == 0) return;
  const int nel = M.nel, next = M.next, ns = M.nsolve;

  // element centres and neighbours through shared side nodes
  std::vector<double> cx(nel), cy(nel);
  for (int e = 0; e < nel; ++e) {
    cx[e] = cy[e] = 0.0;
    for (int k = 0; k < 4; ++k) { cx[e] += 0.25 * M.vx[4 * e + k]; cy[e] += 0.25 * M.vy[4 * e + k]; }
  }
  std::vector<std::vector<int>> adj(nel);
  {
    std::vector<int> owner(M.nglobal, -1);
    const int nm = M.np - 1;
    for (int e = 0; e < nel; ++e)
      for (int s = 0; s < 4; ++s) {
        const int o = owner[M.btog[e * next + s * nm + 1]];
        if (o >= 0 && o != e) { adj[e].push_back(o); adj[o].push_back(e); }
        for (int i = 1; i < nm; ++i) owner[M.btog[e * next + s * nm + i]] = e;
      }
  }
  std::vector<int> perm(nel), slots(M.nglobal, 0);
  std::iota(perm.begin(), perm.end(), 0);
  for (int i = 0; i < nel * next; ++i) slots[M.btog[i]]++;
  std::vector<Bis> bt;
  bt.push_back({0, nel, 0});
  {
    std::vector<char> left(nel, 0);
    for (size_t i = 0; i < bt.size(); ++i) {
      const int lo = bt[i].lo, hi = bt[i].hi, d = bt[i].depth;
      if (hi - lo < 2) continue;
      const int mid = best_split(perm, lo, hi, cx, cy, adj, left);
      bt[i].l = (int)bt.size();
      bt.push_back({lo, mid, d + 1});
      bt[i].r = (int)bt.size();
      bt.push_back({mid, hi, d + 1});
    }
  }
  const int nbt = (int)bt.size();
  for (int i = nbt - 1; i >= 0; --i)
    if (bt[i].l >= 0) bt[i].hdep = 1 + std::max(bt[bt[i].l].hdep, bt[bt[i].r].hdep);
  const int D = bt[0].hdep;

  // element leaves
  VecHash leafh;
  std::vector<int> leaf_of(nel);
  for (int e = 0; e < nel; ++e) {
    std::vector<int> key{M.eset[e]};
    for (int i = 0; i < next; ++i) if (M.btog[e * next + i] < ns) key.push_back(i);
    leaf_of[e] = leafh.id(key);
    if (leaf_of[e] == (int)T.leaf.size()) {
      TreeLeaf L;
      L.set = key[0];
      L.loc.assign(key.begin() + 1, key.end());
      T.leaf.push_back(L);
    }
  }
  const int pin_gid = pinned ? ns - 1 : -1;

  // boundary size, separator size and class of every bisection node (the
  // class: isomorphic subtrees, whose regions share a type under any merge)
  std::vector<int> seen(ns, 0);
  {
    VecHash clsh;
    std::vector<std::vector<int>> bl(nbt);    // ordered boundary lists
    std::vector<int> pos(ns, -1);
    for (int i = nbt - 1; i >= 0; --i) {
      Bis& b = bt[i];
      std::vector<int> U, key;
      if (b.l < 0) {
        const int e = perm[b.lo];
        key = {-1, leaf_of[e]};
        for (int q : T.leaf[leaf_of[e]].loc) bl[i].push_back(M.btog[e * next + q]);
        // repeated nodes (an element joined to itself) keep their pattern
        for (int g : bl[i]) { if (pos[g] < 0) { pos[g] = (int)U.size(); U.push_back(g); } key.push_back(pos[g]); }
        for (int g : U) pos[g] = -1;
        b.nb = (int)U.size();
        b.cls = clsh.id(key);
        continue;
      }
      for (int q = b.lo; q < b.hi; ++q)
        for (int k = 0; k < next; ++k) {
          const int g = M.btog[perm[q] * next + k];
          if (g < ns) seen[g]++;
        }
      key = {bt[b.l].cls, bt[b.r].cls};
      for (int c : {b.l, b.r})
        for (int g : bl[c]) { if (pos[g] < 0) { pos[g] = (int)U.size(); U.push_back(g); } key.push_back(pos[g]); }
      key.push_back(-2);
      for (int g : U) {
        const bool inner = seen[g] == slots[g];
        key.push_back(inner ? (g == pin_gid ? 2 : 1) : 0);
        if (!inner) bl[i].push_back(g);
        pos[g] = -1;
      }
      b.nb = (int)bl[i].size();
      b.sep = (int)U.size() - b.nb;
      b.cls = clsh.id(key);
      for (int q = b.lo; q < b.hi; ++q)
        for (int k = 0; k < next; ++k) {
          const int g = M.btog[perm[q] * next + k];
          if (g < ns) seen[g] = 0;
        }
      std::vector<int>().swap(bl[b.l]);
      std::vector<int>().swap(bl[b.r]);
    }
  }

  // Which depths to merge at: a region at depth d takes all merges down to
  // the next chosen depth p at once (one forward and one backward launch for
  // many small merges, against larger dense matrices).  Modelled time of a
  // stage: launches and their latency, the matrices' bytes (one copy per
  // type and mode) and the matrix-core time (every region), for two
  // right-hand sides per mode.
  const int R = 2;
  std::vector<std::vector<int>> at(D + 1);
  for (int i = 0; i < nbt; ++i) if (bt[i].l >= 0) at[bt[i].depth].push_back(i);
  auto sep_sum = [&](int i, int p) {          // unknowns eliminated by depths [d, p) under i
    int s = 0;
    std::vector<int> st{i};
    while (!st.empty()) {
      const int q = st.back(); st.pop_back();
      if (bt[q].l < 0 || bt[q].depth >= p) continue;
      s += bt[q].sep;
      st.push_back(bt[q].l); st.push_back(bt[q].r);
    }
    return s;
  };
  constexpr double HBM = 4.0e12, MFMA = 1024.0 * 2.4e9 / 64.0, LAUNCH = 5.0e-6;
  auto stage_cost = [&](int d, int p) {
    std::map<int, std::pair<std::pair<int, int>, int>> cl;   // class -> (ni, nb), count
    for (int i : at[d]) {
      auto& c = cl[bt[i].cls];
      if (c.second == 0) c.first = {sep_sum(i, p), bt[i].nb};
      c.second++;
    }
    double bytes = 0.0, ops = 0.0;
    for (auto& q : cl) {
      const int ni = q.second.first.first, nb = q.second.first.second, cnt = q.second.second;
      if (ni == 0) continue;
      if ((size_t)((ni + nb + 7) / 8 * 8) * 8 * 8 > (size_t)TREE_LDS || ni > 1280) return 1e30;
      const double el = (double)tree_packed(nb, ni) + (double)tree_packed(ni, ni + nb);
      bytes += 8.0 * el;
      ops += el / 64.0 * ((cnt * R + 15) / 16);
    }
    return (d == 0 ? 1.0 : 2.0) * LAUNCH + std::max(nd * bytes / HBM, nd * ops / MFMA);
  };
  std::vector<double> best(D + 2, 1e300);
  std::vector<int> from(D + 2, -1);
  best[D + 1] = 0.0;      // the elements
  for (int d = D; d >= 0; --d) {
    if (at[d].empty() && !(d == 0 && D == 0)) continue;
    for (int p = d + 1; p <= D + 1; ++p) {
      if (best[p] >= 1e29) continue;
      const double c = best[p] + stage_cost(d, p);
      if (c < best[d]) { best[d] = c; from[d] = p; }
    }
  }
  if (best[0] >= 1e29) return;
  std::vector<int> cuts;                 // depths from the deepest to 0
  for (int d = 0; d <= D; d = from[d]) cuts.push_back(d);
  std::reverse(cuts.begin(), cuts.end());

  // Build the regions stage by stage.
  VecHash typeh;
  struct Reg { int type = -1; std::vector<int> bnd; int cslot = 0; };   // per bisection node
  std::vector<Reg> reg(nbt);
  const int L0 = nel * next;
  std::vector<int> pos(ns, -1);
  T.stage_ptr = {0};
  for (size_t k = 0; k < cuts.size(); ++k) {
    const int d = cuts[k], p = k ? cuts[k - 1] : D + 1;
    struct Pend { int bis; int type; std::vector<int> U; std::vector<std::vector<int>> src; };
    std::vector<Pend> pend;
    std::vector<int> tops = at[d];
    if (D == 0) tops = {0};
    for (int t : tops) {
      // children: descendants at depth p, or elements above it; an already
      // passed-through region keeps the child it stands for
      std::vector<int> ch, st{t};
      std::vector<char> merge;
      while (!st.empty()) {
        const int q = st.back(); st.pop_back();
        if (q < 0) { merge.push_back(1); continue; }
        const bool stop = bt[q].l < 0 || (q != t && bt[q].depth >= p);
        if (stop) { ch.push_back(q); merge.push_back(0); continue; }
        st.push_back(-1); st.push_back(bt[q].r); st.push_back(bt[q].l);
      }
      for (int q = bt[t].lo; q < bt[t].hi; ++q)
        for (int i = 0; i < next; ++i) {
          const int g = M.btog[perm[q] * next + i];
          if (g < ns) seen[g]++;
        }
      std::vector<int> U, key{-7};
      std::vector<std::vector<int>> src;
      TreeType ty;
      ty.merge = merge;
      ty.cptr.push_back(0);
      for (int c : ch) {
        const bool leaf = bt[c].l < 0;
        const int e = leaf ? perm[bt[c].lo] : -1;
        const int id = leaf ? -1 - leaf_of[e] : reg[c].type;
        ty.child.push_back(id);
        key.push_back(id);
        std::vector<int> bnd;
        if (leaf) for (int q : T.leaf[leaf_of[e]].loc) bnd.push_back(M.btog[e * next + q]);
        const std::vector<int>& B = leaf ? bnd : reg[c].bnd;
        for (size_t i = 0; i < B.size(); ++i) {
          const int g = B[i];
          if (pos[g] < 0) { pos[g] = (int)U.size(); U.push_back(g); src.emplace_back(); }
          ty.cmap.push_back(pos[g]);
          src[pos[g]].push_back(leaf ? e * next + T.leaf[leaf_of[e]].loc[i]
                                     : L0 + reg[c].cslot + (int)i);
        }
        ty.cptr.push_back((int)ty.cmap.size());
      }
      // eliminated unknowns first
      std::vector<int> ord, newpos(U.size());
      for (int pass = 0; pass < 2; ++pass)
        for (size_t i = 0; i < U.size(); ++i) {
          const bool inner = seen[U[i]] == slots[U[i]];
          if (inner == (pass == 0)) { newpos[i] = (int)ord.size(); ord.push_back((int)i); }
          if (inner && pass == 0) ++ty.ni;
        }
      ty.nb = (int)U.size() - ty.ni;
      for (int& c : ty.cmap) c = newpos[c];
      Pend pe;
      pe.bis = t;
      for (int i : ord) { pe.U.push_back(U[i]); pe.src.push_back(src[i]); }
      for (int i = 0; i < ty.ni; ++i) if (pe.U[i] == pin_gid) ty.pin = i;
      key.push_back(ty.ni); key.push_back(ty.pin);
      key.insert(key.end(), ty.cmap.begin(), ty.cmap.end());
      pe.type = typeh.id(key);
      if (pe.type == (int)T.type.size()) { ty.stage = (int)k; T.type.push_back(ty); }
      for (int g : U) pos[g] = -1;
      for (int q = bt[t].lo; q < bt[t].hi; ++q)
        for (int i = 0; i < next; ++i) {
          const int g = M.btog[perm[q] * next + i];
          if (g < ns) seen[g] = 0;
        }
      pend.push_back(std::move(pe));
    }
    std::stable_sort(pend.begin(), pend.end(), [](const Pend& a, const Pend& b) { return a.type < b.type; });
    for (Pend& pe : pend) {
      const TreeType& ty = T.type[pe.type];
      TreeNode n;
      n.type = pe.type;
      n.uptr = (int)T.gid.size();
      n.cslot = T.nslot_c;
      n.yslot = T.nslot_y;
      T.nslot_c += ty.nb;
      T.nslot_y += ty.ni;
      for (size_t i = 0; i < pe.U.size(); ++i) {
        T.gid.push_back(pe.U[i]);
        T.rowptr.push_back((int)T.src.size());
        T.src.insert(T.src.end(), pe.src[i].begin(), pe.src[i].end());
      }
      reg[pe.bis].type = pe.type;
      reg[pe.bis].cslot = n.cslot;
      reg[pe.bis].bnd.assign(pe.U.begin() + ty.ni, pe.U.end());
      T.node.push_back(n);
    }
    T.stage_ptr.push_back((int)T.node.size());
    // regions that are one element pass through: they stay leaves
  }
  T.rowptr.push_back((int)T.src.size());
  T.nstage = (int)cuts.size();
  long long off = 0;
  for (TreeType& t : T.type) {
    t.off_f = off; off += tree_packed(t.nb, t.ni);
    t.off_b = off; off += tree_packed(t.ni, t.ni + t.nb);
  }
  T.mstride = off;
  T.on = true;
}

// ---------------------------------------------------------------------------
// Dense kernels of the factorisation, row-major, blocked so that the inner
// loops run along rows (cloned by feature for AVX-512 and FMA hosts: a clone by processor name
// left every other model on the baseline code).
// ---------------------------------------------------------------------------

namespace {

constexpr int FB = 48;    // block size of the triangular steps

typedef double v8d __attribute__((vector_size(64)));

// C (m x n) -= A (m x k) B (k x n), in columns of 16 (the last ones through a
// padded copy of B's) so that a column block of B stays in the L1 cache.
__attribute__((target_clones("avx512f", "fma", "default")))
void gemm_sub(int m, int n, int k, const double* __restrict__ A, int lda,
              const double* __restrict__ B, int ldb, double* __restrict__ C, int ldc) {
  for (int j = 0; j < n; j += 16) {
    const int w = std::min(16, n - j);
    const double* b = B + j;
    int sb = ldb;
    static thread_local std::vector<double> pad;
    if (w < 16) {
      pad.assign((size_t)k * 16, 0.0);
      for (int p = 0; p < k; ++p) memcpy(&pad[(size_t)p * 16], b + (size_t)p * ldb, w * sizeof(double));
      b = pad.data();
      sb = 16;
    }
    for (int i = 0; i < m; i += 4) {
      const int h = std::min(4, m - i);
      const double *a0 = A + (size_t)i * lda, *a1 = h > 1 ? a0 + lda : a0,
                   *a2 = h > 2 ? a0 + 2 * (size_t)lda : a0, *a3 = h > 3 ? a0 + 3 * (size_t)lda : a0;
      v8d c00 = {}, c01 = {}, c10 = {}, c11 = {}, c20 = {}, c21 = {}, c30 = {}, c31 = {};
      for (int p = 0; p < k; ++p) {
        v8d b0, b1;
        memcpy(&b0, b + (size_t)p * sb, sizeof b0);
        memcpy(&b1, b + (size_t)p * sb + 8, sizeof b1);
        c00 += a0[p] * b0; c01 += a0[p] * b1;
        c10 += a1[p] * b0; c11 += a1[p] * b1;
        c20 += a2[p] * b0; c21 += a2[p] * b1;
        c30 += a3[p] * b0; c31 += a3[p] * b1;
      }
      const v8d t[4][2] = {{c00, c01}, {c10, c11}, {c20, c21}, {c30, c31}};
      for (int r = 0; r < h; ++r) {
        double* c = C + (size_t)(i + r) * ldc + j;
        if (w == 16) {
          v8d x, y;
          memcpy(&x, c, sizeof x);
          memcpy(&y, c + 8, sizeof y);
          x -= t[r][0];
          y -= t[r][1];
          memcpy(c, &x, sizeof x);
          memcpy(c + 8, &y, sizeof y);
        } else {
          for (int q = 0; q < w; ++q) c[q] -= t[r][q >> 3][q & 7];
        }
      }
    }
  }
}

// A^T block (rows r0.., cols c0..) packed row-major: out (cols x rows)
void pack_t(const double* A, int lda, int rows, int cols, double* out) {
  for (int r = 0; r < rows; ++r)
    for (int c = 0; c < cols; ++c) out[(size_t)c * rows + r] = A[(size_t)r * lda + c];
}

// Rows of T (n x w, row stride w) <- L^-1 T, L the n x n lower triangle at A.
__attribute__((target_clones("avx512f", "fma", "default")))
void panel_forward(int n, int w, const double* A, int ld, double* T) {
  for (int c0 = 0; c0 < w; c0 += 128) {
    const int m = std::min(128, w - c0);
    for (int r = 0; r < n; ++r) {
      double* __restrict__ tr = T + (size_t)r * w + c0;
      for (int k = 0; k < r; ++k) {
        const double l = A[(size_t)r * ld + k];
        const double* tk = T + (size_t)k * w + c0;
        for (int c = 0; c < m; ++c) tr[c] -= l * tk[c];
      }
      const double d = 1.0 / A[(size_t)r * ld + r];
      for (int c = 0; c < m; ++c) tr[c] *= d;
    }
  }
}

// Cholesky of the leading n x n of A (ld), lower triangle in place.
int chol_lower(int n, double* A, int ld, std::vector<double>& tmp) {
  for (int j0 = 0; j0 < n; j0 += FB) {
    const int nb = std::min(FB, n - j0), rest = n - j0 - nb;
    double* P = A + (size_t)j0 * ld + j0;
    for (int j = 0; j < nb; ++j) {
      for (int i = j; i < nb; ++i) {
        double s = P[(size_t)i * ld + j];
        for (int k = 0; k < j; ++k) s -= P[(size_t)i * ld + k] * P[(size_t)j * ld + k];
        if (i == j) {
          if (!(s > 0.0)) return SEMX_E_NOT_SPD;
          P[(size_t)j * ld + j] = std::sqrt(s);
        } else {
          P[(size_t)i * ld + j] = s / P[(size_t)j * ld + j];
        }
      }
    }
    if (rest <= 0) break;
    // the rows below the block, as columns: tmp = L_JJ^-1 A_rest,J^T
    double* B = A + (size_t)(j0 + nb) * ld + j0;
    tmp.resize((size_t)rest * nb);
    pack_t(B, ld, rest, nb, tmp.data());   // nb x rest
    panel_forward(nb, rest, P, ld, tmp.data());
    for (int r = 0; r < rest; ++r)
      for (int c = 0; c < nb; ++c) B[(size_t)r * ld + c] = tmp[(size_t)c * rest + r];
    // trailing update, lower triangle by row blocks
    for (int r0 = 0; r0 < rest; r0 += 64) {
      const int nr = std::min(64, rest - r0);
      gemm_sub(nr, r0 + nr, nb, B + (size_t)r0 * ld, ld, tmp.data(), rest,
               B + (size_t)r0 * ld + nb, ld);
    }
  }
  return SEMX_OK;
}

constexpr int FC = 64;    // columns per chunk of the triangular solves

// Column chunk T (rows i0..ni of n columns, row stride FC) <- L^-1 T.
__attribute__((target_clones("avx512f", "fma", "default")))
void chunk_forward(int ni, int i0, const double* A, int ld, double* T) {
  for (int b0 = i0 / FB * FB; b0 < ni; b0 += FB) {
    const int s = std::max(b0, i0), e = std::min(b0 + FB, ni);
    if (s > i0) gemm_sub(e - s, FC, s - i0, A + (size_t)s * ld + i0, ld, T + (size_t)i0 * FC, FC,
                         T + (size_t)s * FC, FC);
    for (int r = s; r < e; ++r) {
      double* __restrict__ tr = T + (size_t)r * FC;
      for (int k = s; k < r; ++k) {
        const double l = A[(size_t)r * ld + k];
        const double* tk = T + (size_t)k * FC;
        for (int c = 0; c < FC; ++c) tr[c] -= l * tk[c];
      }
      const double d = 1.0 / A[(size_t)r * ld + r];
      for (int c = 0; c < FC; ++c) tr[c] *= d;
    }
  }
}

// Rows i0..ni of the chunk T <- (L^-T T), rows from the last up; LT: L
// transposed (row-major, upper triangle).
__attribute__((target_clones("avx512f", "fma", "default")))
void chunk_backward(int ni, int i0, const double* LT, double* T) {
  for (int b0 = (ni - 1) / FB * FB; b0 + FB > i0; b0 -= FB) {
    const int s = std::max(b0, i0), e = std::min(b0 + FB, ni);
    if (e < ni) gemm_sub(e - s, FC, ni - e, LT + (size_t)s * ni + e, ni, T + (size_t)e * FC, FC,
                         T + (size_t)s * FC, FC);
    for (int r = e - 1; r >= s; --r) {
      double* __restrict__ tr = T + (size_t)r * FC;
      for (int k = r + 1; k < e; ++k) {
        const double l = LT[(size_t)r * ni + k];
        const double* tk = T + (size_t)k * FC;
        for (int c = 0; c < FC; ++c) tr[c] -= l * tk[c];
      }
      const double d = 1.0 / LT[(size_t)r * ni + r];
      for (int c = 0; c < FC; ++c) tr[c] *= d;
    }
  }
}

struct ElimWork { std::vector<double> U, W, LT, tmp; RawDoubles XE, G, Z; };

// fn(i) for i < n on up to nth threads
template <class F>
void spread(int n, int nth, F fn) {
  nth = std::min(n, nth);
  if (nth <= 1) { for (int i = 0; i < n; ++i) fn(i); return; }
  std::atomic<int> next{0};
  std::vector<std::thread> pool;
  for (int t = 0; t < nth; ++t)
    pool.emplace_back([&]() { for (int i; (i = next++) < n;) fn(i); });
  for (auto& th : pool) th.join();
}

// A region's dense matrices: U (nu x nu, eliminated unknowns first) ->
// W = [A_II^-1 A_IB | A_II^-1] (ni x (nb + ni)) and S = A_BB - A_BI A_II^-1
// A_IB in U's last block, on nth threads (column chunks are independent).
int eliminate(int ni, int nb, ElimWork& E, int nth) {
  const int nu = ni + nb, ldw = nu;
  double* A = E.U.data();
  if (int st = chol_lower(ni, A, nu, E.tmp)) return st;
  E.W.resize((size_t)ni * ldw);
  E.LT.assign((size_t)ni * ni, 0.0);
  double* W = E.W.data();
  for (int r = 0; r < ni; ++r)
    for (int c = 0; c <= r; ++c) E.LT[(size_t)c * ni + r] = A[(size_t)r * nu + c];
  const int cb = (nb + FC - 1) / FC, ci = (ni + FC - 1) / FC;
  if ((long long)ni * ni * nu < 4000000) nth = 1;
  // boundary columns forward
  spread(cb, nth, [&](int j) {
    const int c0 = j * FC, n = std::min(FC, nb - c0);
    std::vector<double> T((size_t)ni * FC, 0.0);
    for (int r = 0; r < ni; ++r) memcpy(&T[(size_t)r * FC], A + (size_t)r * nu + ni + c0, n * sizeof(double));
    chunk_forward(ni, 0, A, nu, T.data());
    for (int r = 0; r < ni; ++r) memcpy(W + (size_t)r * ldw + c0, &T[(size_t)r * FC], n * sizeof(double));
  });
  // S, by row blocks of the upper triangle, mirrored
  spread(cb, nth, [&](int j) {
    const int r0 = j * FC, n = std::min(FC, nb - r0);
    std::vector<double> t((size_t)ni * FC);
    pack_t(W + r0, ldw, ni, n, t.data());      // n x ni
    gemm_sub(n, nb - r0, ni, t.data(), ni, W + r0, ldw, A + (size_t)(ni + r0) * nu + ni + r0, nu);
  });
  for (int r = 0; r < nb; ++r)
    for (int c = 0; c < r; ++c)
      A[(size_t)(ni + r) * nu + ni + c] = A[(size_t)(ni + c) * nu + ni + r];
  // boundary columns backward; identity columns both ways, their rows from
  // the chunk's own on (the inverse's lower triangle, mirrored)
  spread(cb + ci, nth, [&](int j) {
    std::vector<double> T((size_t)ni * FC, 0.0);
    if (j < cb) {
      const int c0 = j * FC, n = std::min(FC, nb - c0);
      for (int r = 0; r < ni; ++r) memcpy(&T[(size_t)r * FC], W + (size_t)r * ldw + c0, n * sizeof(double));
      chunk_backward(ni, 0, E.LT.data(), T.data());
      for (int r = 0; r < ni; ++r) memcpy(W + (size_t)r * ldw + c0, &T[(size_t)r * FC], n * sizeof(double));
      return;
    }
    const int c0 = (j - cb) * FC, n = std::min(FC, ni - c0);
    for (int c = 0; c < n; ++c) T[(size_t)(c0 + c) * FC + c] = 1.0;
    chunk_forward(ni, c0, A, nu, T.data());
    chunk_backward(ni, c0, E.LT.data(), T.data());
    for (int r = c0; r < ni; ++r)
      for (int c = 0; c < n && c0 + c <= r; ++c) {
        W[(size_t)r * ldw + nb + c0 + c] = T[(size_t)r * FC + c];
        W[(size_t)(c0 + c) * ldw + nb + r] = T[(size_t)r * FC + c];
      }
  });
  return SEMX_OK;
}

// A part of a region: its eliminated unknowns I and boundary unknowns B (the
// region's numbers; cnt: how many of the region's child entries each of B
// stands for), A_II^-1, X = A_II^-1 A_IB and the Schur complement on B.
struct Part {
  std::vector<int> I, B, cnt;
  RawDoubles inv, X;
  std::vector<double> S;
};

// Two parts (or one alone) merged: the unknowns that no other part holds are
// eliminated.  With e of them, n eliminated before and the parts' matrices,
//   A_EE^-1, Y = A_EE^-1 A_EB, S = A_BB - A_BE Y          (eliminate)
//   X   = [X_B - X_E Y; Y]
//   inv = [blockdiag(inv) + X_E A_EE^-1 X_E^T, -X_E A_EE^-1; sym., A_EE^-1]
// which is n^2 e / 2 multiply-adds for the inverse where a factorisation of
// the whole region takes (n + e)^3 / 2.  total: entries of each unknown; pin:
// the unknown to drop (-1: none); pos: scratch, -1 everywhere.
int merge_parts(Part* a, Part* b, int nelim, const std::vector<int>& total, int pin,
                std::vector<int>& pos, ElimWork& E, int nth, Part& out) {
  Part* parts[2] = {a, b};
  const int np = b ? 2 : 1;
  std::vector<int> U, cnt;
  for (int k = 0; k < np; ++k)
    for (size_t i = 0; i < parts[k]->B.size(); ++i) {
      const int u = parts[k]->B[i];
      if (pos[u] < 0) { pos[u] = (int)U.size(); U.push_back(u); cnt.push_back(0); }
      cnt[pos[u]] += parts[k]->cnt[i];
    }
  std::vector<int> el;
  for (size_t i = 0; i < U.size(); ++i) {
    if (U[i] < nelim && cnt[i] == total[U[i]]) el.push_back(U[i]);
    else { out.B.push_back(U[i]); out.cnt.push_back(cnt[i]); }
  }
  const int e = (int)el.size(), nb = (int)out.B.size(), nu = e + nb;
  for (int i = 0; i < e; ++i) pos[el[i]] = i;
  for (int i = 0; i < nb; ++i) pos[out.B[i]] = e + i;
  E.U.assign((size_t)nu * nu, 0.0);
  for (int k = 0; k < np; ++k) {
    const Part& q = *parts[k];
    const int m = (int)q.B.size();
    for (int i = 0; i < m; ++i) {
      double* row = &E.U[(size_t)pos[q.B[i]] * nu];
      for (int j = 0; j < m; ++j) row[pos[q.B[j]]] += q.S[(size_t)i * m + j];
    }
  }
  // the pinned node of a singular mode is dropped (src/matrix.cpp:167-169):
  // decoupled here, its rows and columns of the results zeroed below
  const int ip = pin >= 0 && pos[pin] >= 0 && pos[pin] < e ? pos[pin] : -1;
  if (ip >= 0) {
    for (int k = 0; k < nu; ++k) E.U[(size_t)ip * nu + k] = E.U[(size_t)k * nu + ip] = 0.0;
    E.U[(size_t)ip * nu + ip] = 1.0;
  }
  if (e)
    if (const int st = eliminate(e, nb, E, nth)) return st;
  const double* W = E.W.data();
  if (ip >= 0) {
    for (int k = 0; k < nu; ++k) E.W[(size_t)ip * nu + k] = 0.0;
    for (int r = 0; r < e; ++r) E.W[(size_t)r * nu + nb + ip] = 0.0;
  }
  out.S.resize((size_t)nb * nb);
  for (int r = 0; r < nb; ++r)
    std::copy_n(&E.U[(size_t)(e + r) * nu + e], nb, &out.S[(size_t)r * nb]);
  int n = 0;
  for (int k = 0; k < np; ++k) n += (int)parts[k]->I.size();
  const int ni = n + e;
  out.inv.resize((size_t)ni * ni);
  out.X.resize((size_t)ni * nb);
  E.XE.resize((size_t)n * e);
  if ((long long)n * (ni + e) < 200000) nth = 1;
  const int split = np > 1 ? (int)a->I.size() : n;
  for (int k = 0; k < np; ++k) out.I.insert(out.I.end(), parts[k]->I.begin(), parts[k]->I.end());
  out.I.insert(out.I.end(), el.begin(), el.end());
  std::vector<int> col[2];
  for (int k = 0; k < np; ++k)
    for (int u : parts[k]->B) col[k].push_back(pos[u]);
  for (int u : U) pos[u] = -1;
  // the parts' rows: their inverses with zeros to their right, their X split
  // into the eliminated and the other columns
  const int nblk = (n + FC - 1) / FC;
  spread(nblk, nth, [&](int j) {
    for (int r = j * FC; r < std::min((j + 1) * FC, n); ++r) {
      const int k = r >= split, r0 = k ? split : 0;
      const Part& q = *parts[k];
      const int m = (int)q.I.size(), mb = (int)q.B.size();
      double* v = &out.inv[(size_t)r * ni];
      std::copy_n(&q.inv[(size_t)(r - r0) * m], m, v + r0);
      std::fill(v + r0 + m, v + n, 0.0);
      const double* x = q.X.data() + (size_t)(r - r0) * mb;
      double *xe = E.XE.data() + (size_t)r * e, *xb = out.X.data() + (size_t)r * nb;
      std::fill_n(xe, e, 0.0);
      std::fill_n(xb, nb, 0.0);
      for (int c = 0; c < mb; ++c) {
        const int at = col[k][c];
        (at < e ? xe[at] : xb[at - e]) = x[c];
      }
    }
  });
  if (e) {
    E.G.resize((size_t)n * e);
    E.Z.resize((size_t)n * e);
    pack_t(E.XE.data(), e, n, e, E.Z.data());      // e x n
    spread(nblk, nth, [&](int j) {
      const int s = j * FC, m = std::min(FC, n - s);
      const double* x = &E.XE[(size_t)s * e];
      double* g = &E.G[(size_t)s * e];
      std::fill_n(g, (size_t)m * e, 0.0);
      gemm_sub(m, nb, e, x, e, W, nu, out.X.data() + (size_t)s * nb, nb);
      gemm_sub(m, e, e, x, e, W + nb, nu, g, e);
      gemm_sub(m, n - s, e, g, e, &E.Z[s], n, &out.inv[(size_t)s * ni + s], ni);
      for (int r = s; r < s + m; ++r) std::copy_n(&E.G[(size_t)r * e], e, &out.inv[(size_t)r * ni + n]);
    });
    for (int r = 0; r < e; ++r) {
      std::copy_n(W + (size_t)r * nu, nb, out.X.data() + (size_t)(n + r) * nb);
      std::copy_n(W + (size_t)r * nu + nb, e, &out.inv[(size_t)(n + r) * ni + n]);
    }
  }
  // the rows below the diagonal: mirrored, by blocks
  spread((ni + 31) / 32, nth, [&](int b) {
    const int i = 32 * b;
    for (int j = 0; j <= i; j += 32)
      for (int r = i; r < std::min(i + 32, ni); ++r)
        for (int c = j; c < std::min(j + 32, r); ++c)
          out.inv[(size_t)r * ni + c] = out.inv[(size_t)c * ni + r];
  });
  return SEMX_OK;
}

// Packs a matrix of which row(r, buf) writes row r.
template <class F>
void pack_matrix(int rows, int cols, double* out, int nth, F row) {
  const int mt = tree_mt(rows), kp = tree_kp(cols);
  if ((long long)rows * cols < 100000) nth = 1;
  spread(mt, nth, [&](int t) {
    std::vector<double> buf((size_t)16 * kp * 8, 0.0);
    for (int r = 16 * t; r < std::min(16 * t + 16, rows); ++r) row(r, &buf[(size_t)(r - 16 * t) * kp * 8]);
    double* o = out + (size_t)t * kp * 128;
    for (int k = 0; k < kp; ++k, o += 128)
      for (int l = 0; l < 64; ++l) {
        const double* b = &buf[(size_t)(l & 15) * kp * 8 + 8 * k + (l >> 4)];
        o[2 * l] = b[0];
        o[2 * l + 1] = b[4];
      }
  });
}

}  // namespace

int tree_factor(Helm& H) {
  Tree& T = H.tree;
  const Mesh& M = *H.M;
  const int next = M.next, nset = M.nset;
  std::vector<int> dm;
  for (int m = 0; m < H.nmodes; ++m) if (H.modes[m].kind == SEMX_DIRECT) dm.push_back(m);
  const int nd = (int)dm.size(), nt = (int)T.type.size();
  T.mat.resize((size_t)nd * T.mstride);   // packed whole below
  std::vector<std::vector<double>> S((size_t)nd * nt);
  // how many types of later stages still read a type's S
  std::vector<std::atomic<int>> uses((size_t)nd * nt);
  for (auto& u : uses) u = 0;
  for (int t = 0; t < nt; ++t)
    for (int c : T.type[t].child)
      if (c >= 0) for (int i = 0; i < nd; ++i) uses[(size_t)i * nt + c]++;
  std::atomic<int> status{SEMX_OK};
  auto work = [&](int im, int t, ElimWork& E, int nth) {
    const TreeType& ty = T.type[t];
    const int m = dm[im], ni = ty.ni, nb = ty.nb, nu = ni + nb;
    std::vector<int> total(nu, 0), pos(nu, -1);
    for (int u : ty.cmap) total[u]++;
    const int pin = H.modes[m].singular ? ty.pin : -1;
    // merge by merge, as the bisection did: parts in the order the children
    // come in, the halves of a large region on threads of their own
    struct Half { int child, l, r, size; };
    std::vector<Half> half;
    {
      std::vector<int> st;
      int c = 0;
      for (char op : ty.merge) {
        if (!op) {
          half.push_back({c++, -1, -1, 1});
        } else {
          const int r = st.back(), l = st[st.size() - 2];
          st.resize(st.size() - 2);
          half.push_back({-1, l, r, half[l].size + half[r].size});
        }
        st.push_back((int)half.size() - 1);
      }
    }
    std::function<int(int, int, ElimWork&, std::vector<int>&, Part&)> build =
        [&](int h, int threads, ElimWork& W, std::vector<int>& pos, Part& out) {
      const Half& q = half[h];
      if (q.child >= 0) {
        const int id = ty.child[q.child], n = ty.cptr[q.child + 1] - ty.cptr[q.child];
        const int* mp = &ty.cmap[ty.cptr[q.child]];
        out.B.assign(mp, mp + n);
        out.cnt.assign(n, 1);
        if (id < 0) {
          const TreeLeaf& L = T.leaf[-1 - id];
          const double* hbb = &H.hbb[((size_t)m * nset + L.set) * next * next];
          out.S.resize((size_t)n * n);
          for (int i = 0; i < n; ++i)
            for (int k = 0; k < n; ++k) out.S[(size_t)i * n + k] = hbb[(size_t)L.loc[i] * next + L.loc[k]];
        } else {
          std::vector<double>& s = S[(size_t)im * nt + id];
          out.S = s;
          if (--uses[(size_t)im * nt + id] == 0) std::vector<double>().swap(s);
        }
        return SEMX_OK;
      }
      Part l, r;
      int sl = SEMX_OK, sr;
      if (threads > 1 && q.size >= 16) {
        std::thread left([&]() {
          ElimWork Wl;
          std::vector<int> pl(nu, -1);
          sl = build(q.l, threads / 2, Wl, pl, l);
        });
        sr = build(q.r, threads - threads / 2, W, pos, r);
        left.join();
      } else {
        sl = build(q.l, threads, W, pos, l);
        sr = build(q.r, threads, W, pos, r);
      }
      if (sl || sr) return sl ? sl : sr;
      return merge_parts(&l, &r, ni, total, pin, pos, W, threads, out);
    };
    Part R;
    int fail = build((int)half.size() - 1, nth, E, pos, R);
    if (!fail && half.size() == 1) {
      Part one;
      std::swap(one, R);
      fail = merge_parts(&one, nullptr, ni, total, pin, pos, E, nth, R);
    }
    if (fail) { status = SEMX_E_NOT_SPD; return; }
    std::vector<int> pi(ni), pb(nb);        // the region's numbers -> rows and columns
    for (int i = 0; i < ni; ++i) pi[R.I[i]] = i;
    for (int i = 0; i < nb; ++i) pb[R.B[i] - ni] = i;
    // forward: -X^T (nb x ni); backward: [inv | -X] (ni x (ni + nb))
    double* out = &T.mat[(size_t)im * T.mstride];
    pack_matrix(nb, ni, out + ty.off_f, nth, [&](int r, double* o) {
      for (int q = 0; q < ni; ++q) o[q] = -R.X[(size_t)pi[q] * nb + pb[r]];
    });
    pack_matrix(ni, nu, out + ty.off_b, nth, [&](int r, double* o) {
      const double *v = &R.inv[(size_t)pi[r] * ni], *x = R.X.data() + (size_t)pi[r] * nb;
      for (int q = 0; q < ni; ++q) o[q] = v[pi[q]];
      for (int q = 0; q < nb; ++q) o[ni + q] = -x[pb[q]];
    });
    if (nb) {
      std::vector<double>& s = S[(size_t)im * nt + t];
      s.resize((size_t)nb * nb);
      for (int r = 0; r < nb; ++r)
        for (int k = 0; k < nb; ++k) s[(size_t)r * nb + k] = R.S[(size_t)pb[r] * nb + pb[k]];
    }
  };
  // types of a stage are independent of each other
  const int nth = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  for (int st = 0; st < T.nstage && status == SEMX_OK; ++st) {
    std::vector<int> list;
    for (int t = 0; t < nt; ++t) if (T.type[t].stage == st) list.push_back(t);
    const int total = (int)list.size() * nd;
    std::atomic<int> nextj{0};
    // one worker per region and mode at a time; the last of them share the threads
    spread(std::min(nth, total), nth, [&](int) {
      ElimWork E;
      for (int j; (j = nextj++) < total && status == SEMX_OK;)
        work(j % nd, list[j / nd], E, std::max(1, nth / (total - j)));
    });
  }
  return status;
}

}  // namespace semx
