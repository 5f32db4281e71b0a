// semx_tree.hip -- the direct solve's boundary systems through the
// elimination tree (semx_tree.h) on CDNA4: one launch per stage up the tree
// (regions reduce their right-hand sides to their boundaries) and one per
// stage down (regions recover their eliminated unknowns), in the place of
// LAPACK's banded triangular solves (dpbtrs, src/field.cpp:609).
//
// Why a tree: the band sweeps walk a mode's factor block by block, a serial
// chain of nsolve/32 steps on few workgroups, and read nsolve x nband
// doubles twice.  The tree's matrices are 2.5-8 times fewer bytes (fill
// grows with the separators, not with the band), are shared by translated
// copies of a region, and every region of a stage and every mode is
// independent.  Measured, whole solves, us (band sweeps with the element
// kernels of semx_elem.hip -> tree with them): 16x16 quads np=9 Nz=64 267 ->
// 113 (matrices 110 MB against 444 MB of factor; 156 MB of HBM traffic a
// solve); 32x32 np=11 Nz=16 4124 -> 180; three fields on 20x12 np=8 Nz=32
// periodic in x 305 -> 128; 8x8 np=8 one plane 47 -> 25; 11x7 np=6 Nz=36 all
// elements distinct 45 -> 38.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "semx_hip.h"

namespace semx {

typedef double tree_d4 __attribute__((ext_vector_type(4)));

// A region type's sizes and matrices, and a region.
struct TreeTypeDev { int ni, nb; long long off_f, off_b; };
struct TreeTask { int node, count, mt, pad; };   // regions of one type, first row tile

struct TreeList {               // launch list of one direction and stage
  size_t first = 0;             // of its tasks
  int ntask = 0, wk = 1, ct = 1, ldn = 16;
  size_t lds = 0;
};

struct TreeDev {
  double* mat = nullptr;
  TreeTypeDev* type = nullptr;
  int4* node = nullptr;         // type, uptr, cslot, yslot
  int* gid = nullptr;
  int* rowptr = nullptr;
  int* src = nullptr;
  double* C = nullptr;          // boundary contributions, per field and plane
  double* Y = nullptr;          // assembled right-hand sides of eliminated unknowns
  int nf_cap = 0;
  // launch lists per field count: forward stages, then backward stages
  std::vector<TreeList> list[SEMX_MAX_FIELDS + 1];
  TreeTask* task = nullptr;     // their tasks
};

namespace {

constexpr int TT = 512;         // threads per workgroup
constexpr int TW = TT / 64;

struct TreeArgs {
  const TreeTask* task;
  const TreeTypeDev* type;
  const int4* node;
  const int* gid;
  const int* rowptr;
  const int* src;
  const double* mat;
  long long mstride;
  const int* dmode;
  const int* mode_plane;
  const double* Fb;
  double* C;
  double* Y;
  double* sol;
  long long fbF, cF, yF, solF;   // strides between fields
  int fbS, cS, yS, solS;         // strides between planes
  int npl, nrhs, wk, ldn;
};

// The right-hand-side tile of a workgroup, K rows by its (region, plane)
// columns: ldn = 16: 16-column tiles of K rows one after the other; ldn <
// 16: one tile of ldn columns, which the lanes of a matrix instruction
// read modulo ldn (columns past the last one compute values nobody stores).
//
// A workgroup multiplies wm = TW / wk row tiles of the type's matrix by
// that tile: wave (t, q) takes row tile mt + t and the q-th of wk shares of
// the K steps, its matrix operands streamed from memory in the packed order
// (16 bytes per lane and step, four steps ahead), the partial products
// added through LDS.  What bounds it: on a mesh of one geometric set the
// few types' matrices come from L2 and the matrix cores do the work; where
// every region is its own type, streaming the matrices from HBM.
template <int CT>
__device__ inline void tree_product(const double* __restrict__ mat, int mt, int mtn, int K,
                                    int wk, int ldn, const double* vs, double* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int t = wave / wk, q = wave - t * wk;
  const int KP = (K + 7) >> 3, Kr = KP * 8;
  const bool live = mt + t < mtn && KP > 0;
  tree_d4 acc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) acc[c] = tree_d4{0.0, 0.0, 0.0, 0.0};
  if (live) {
    const int k0 = (KP * q) / wk, k1 = (KP * (q + 1)) / wk;
    const double2* A = reinterpret_cast<const double2*>(mat) + (size_t)(mt + t) * KP * 64 + lane;
    const int col = CT > 1 ? li : (li & (ldn - 1));
    const int ld = CT > 1 ? 16 : ldn;
    double2 a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = A[(size_t)min(k0 + u, KP - 1) * 64];
    for (int k = k0; k < k1; k += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double2 av = a[u];
        a[u] = A[(size_t)min(k + u + 4, KP - 1) * 64];
        if (k + u < k1) {
          const double* v = vs + (size_t)(8 * (k + u) + lk) * ld + col;
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, v[(size_t)c * Kr * 16], acc[c], 0, 0, 0);
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, v[(size_t)c * Kr * 16 + 4 * ld],
                                                          acc[c], 0, 0, 0);
          }
        }
      }
    }
  }
  __syncthreads();     // the right-hand-side tile is no longer read: red takes its place
  // red[wave][column][row], rows padded to 17
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      red[((size_t)wave * 16 * CT + c * 16 + li) * 17 + 4 * r + lk] = acc[c][r];
  __syncthreads();
}

struct TreeCol { int fld, p, node; };

// column n of a task: region n / nrhs, field and plane from n % nrhs
// (p < 0: a mode without a second plane)
__device__ inline TreeCol tree_col(const TreeArgs& a, int m, int node0, int n) {
  TreeCol c;
  const int q = n / a.nrhs, r = n - q * a.nrhs;
  c.node = node0 + q;
  c.fld = r / a.npl;
  c.p = a.mode_plane[2 * m + (r - c.fld * a.npl)];
  return c;
}

// sum of the contributions to unknown u of a region
__device__ inline double tree_gather(const TreeArgs& a, const TreeCol& c, int u, int nleaf) {
  const double* fb = a.Fb + c.fld * a.fbF + (size_t)c.p * a.fbS;
  const double* cc = a.C + c.fld * a.cF + (size_t)c.p * a.cS;
  double v = 0.0;
  for (int k = a.rowptr[u]; k < a.rowptr[u + 1]; ++k) {
    const int s = a.src[k];
    v += s < nleaf ? fb[s] : cc[s - nleaf];
  }
  return v;
}

__device__ inline size_t tree_at(int ldn, int Kr, int k, int n) {
  return ldn < 16 ? (size_t)k * ldn + n : ((size_t)(n >> 4) * Kr + k) * 16 + (n & 15);
}

// Up the tree: c = F_B - X F_I per region, F_I kept for the way down.
template <int CT>
__global__ __launch_bounds__(TT) void k_tree_up(TreeArgs a, int nleaf) {
  extern __shared__ double lds[];
  const TreeTask tk = a.task[blockIdx.x];
  const int im = blockIdx.y, m = a.dmode[im];
  const int4 n0 = a.node[tk.node];
  const TreeTypeDev ty = a.type[n0.x];
  const int K = ty.ni, N = tk.count * a.nrhs, Kr = (K + 7) & ~7;
  const int tid = threadIdx.x, wm = TW / a.wk;
  for (int i = tid; i < N * Kr; i += TT) {
    const int n = i / Kr, k = i - n * Kr;
    double v = 0.0;
    const TreeCol c = tree_col(a, m, tk.node, n);
    if (k < K && c.p >= 0) {
      const int4 nd = a.node[c.node];
      v = tree_gather(a, c, nd.y + k, nleaf);
      if (tk.mt == 0) a.Y[c.fld * a.yF + (size_t)c.p * a.yS + nd.w + k] = v;
    }
    lds[tree_at(a.ldn, Kr, k, n)] = v;
  }
  __syncthreads();
  const int mtn = (ty.nb + 15) >> 4;
  tree_product<CT>(a.mat + (size_t)im * a.mstride + ty.off_f, tk.mt, mtn, K, a.wk, a.ldn, lds, lds);
  const int rows = min(wm * 16, ty.nb - tk.mt * 16);
  for (int i = tid; i < N * wm * 16; i += TT) {
    const int n = i / (wm * 16), r = i - n * (wm * 16);
    if (r >= rows) continue;
    const TreeCol c = tree_col(a, m, tk.node, n);
    if (c.p < 0) continue;
    const int4 nd = a.node[c.node];
    const int b = tk.mt * 16 + r;
    double v = tree_gather(a, c, nd.y + K + b, nleaf);
    for (int q = 0; q < a.wk; ++q)
      v += lds[((size_t)((r >> 4) * a.wk + q) * 16 * CT + n) * 17 + (r & 15)];
    a.C[c.fld * a.cF + (size_t)c.p * a.cS + nd.z + b] = v;
  }
}

// Down the tree: u_I = A_II^-1 F_I - X^T u_B per region.  ROOT: the last
// stage, which has no boundary and gathers its right-hand side itself.
template <int CT, bool ROOT>
__global__ __launch_bounds__(TT) void k_tree_down(TreeArgs a, int nleaf) {
  extern __shared__ double lds[];
  const TreeTask tk = a.task[blockIdx.x];
  const int im = blockIdx.y, m = a.dmode[im];
  const int4 n0 = a.node[tk.node];
  const TreeTypeDev ty = a.type[n0.x];
  const int K = ty.ni + ty.nb, N = tk.count * a.nrhs, Kr = (K + 7) & ~7;
  const int tid = threadIdx.x, wm = TW / a.wk;
  for (int i = tid; i < N * Kr; i += TT) {
    const int n = i / Kr, k = i - n * Kr;
    double v = 0.0;
    const TreeCol c = tree_col(a, m, tk.node, n);
    if (k < K && c.p >= 0) {
      const int4 nd = a.node[c.node];
      if (ROOT)
        v = tree_gather(a, c, nd.y + k, nleaf);
      else if (k < ty.ni)
        v = a.Y[c.fld * a.yF + (size_t)c.p * a.yS + nd.w + k];
      else
        v = a.sol[c.fld * a.solF + (size_t)c.p * a.solS + a.gid[nd.y + k]];
    }
    lds[tree_at(a.ldn, Kr, k, n)] = v;
  }
  __syncthreads();
  const int mtn = (ty.ni + 15) >> 4;
  tree_product<CT>(a.mat + (size_t)im * a.mstride + ty.off_b, tk.mt, mtn, K, a.wk, a.ldn, lds, lds);
  const int rows = min(wm * 16, ty.ni - tk.mt * 16);
  for (int i = tid; i < N * wm * 16; i += TT) {
    const int n = i / (wm * 16), r = i - n * (wm * 16);
    if (r >= rows) continue;
    const TreeCol c = tree_col(a, m, tk.node, n);
    if (c.p < 0) continue;
    const int4 nd = a.node[c.node];
    double v = 0.0;
    for (int q = 0; q < a.wk; ++q)
      v += lds[((size_t)((r >> 4) * a.wk + q) * 16 * CT + n) * 17 + (r & 15)];
    a.sol[c.fld * a.solF + (size_t)c.p * a.solS + a.gid[nd.y + tk.mt * 16 + r]] = v;
  }
}

// K shares of a stage: enough waves on the long products, whole products
// per wave on the short ones (independent of the field count, so that a
// field's sums do not depend on the fields solved with it).
int share(int K) { return K >= 256 ? 8 : K >= 128 ? 4 : K >= 48 ? 2 : 1; }

}  // namespace

int tree_upload(Helm& H) {
  Tree& T = H.tree;
  if (!T.on || H.d.tree) return SEMX_OK;
  TreeDev* D = new TreeDev();
  H.d.tree = D;
  std::vector<TreeTypeDev> ty;
  for (const TreeType& t : T.type) ty.push_back({t.ni, t.nb, t.off_f, t.off_b});
  std::vector<int4> nd;
  for (const TreeNode& n : T.node) nd.push_back(make_int4(n.type, n.uptr, n.cslot, n.yslot));
  int st;
  if ((st = dev_upload(&D->mat, T.mat.data(), T.mat.size()))) return st;
  if ((st = dev_upload(&D->type, ty.data(), ty.size()))) return st;
  if ((st = dev_upload(&D->node, nd.data(), nd.size()))) return st;
  if ((st = dev_upload(&D->gid, T.gid.data(), T.gid.size()))) return st;
  if ((st = dev_upload(&D->rowptr, T.rowptr.data(), T.rowptr.size()))) return st;
  if ((st = dev_upload(&D->src, T.src.data(), T.src.size()))) return st;
  RawDoubles().swap(T.mat);
  return SEMX_OK;
}

// Launch lists for nrhs right-hand sides a mode, without their device
// addresses: up to TREE_GROUP regions of one type per workgroup, as many as
// the right-hand-side tile's LDS holds.  Every workgroup of a stage reads as
// many column tiles as its widest one, so the stage's longest regions limit
// the columns of all: a duct's short regions beside a large section's long
// ones are taken in smaller groups (nrhs <= 6 columns of the at most 2048
// rows that tree_plan allows always fit).
static int tree_lists(const Tree& T, int nrhs, std::vector<TreeList>& out,
                      std::vector<TreeTask>& tasks) {
  for (int dir = 0; dir < 2; ++dir)
    for (int s = 0; s < T.nstage; ++s) {
      TreeList L;
      int Kmax = 0;
      for (int i = T.stage_ptr[s]; i < T.stage_ptr[s + 1]; ++i) {
        const TreeType& t = T.type[T.node[i].type];
        Kmax = std::max(Kmax, dir && t.ni ? t.ni + t.nb : t.ni);
      }
      L.wk = share(Kmax);
      const int wm = TW / L.wk, kl = (Kmax + 7) / 8 * 8;
      int cols = 48;            // three column tiles
      while (cols > 16 && (size_t)kl * cols * 8 > 160 * 1024) cols -= 16;
      if ((size_t)kl * cols * 8 > 160 * 1024) cols = 8;
      const size_t first = tasks.size();
      int nmax = 1;
      for (int i = T.stage_ptr[s]; i < T.stage_ptr[s + 1];) {
        const TreeType& t = T.type[T.node[i].type];
        const int K = dir ? t.ni + t.nb : t.ni, rows = dir ? t.ni : t.nb;
        int run = 1;
        while (i + run < T.stage_ptr[s + 1] && T.node[i + run].type == T.node[i].type) ++run;
        if (dir && rows == 0) { i += run; continue; }    // nothing to recover
        int g = std::min({run, TREE_GROUP, std::max(1, cols / nrhs)});
        while (g > 1 && (size_t)((K + 7) / 8 * 8) * ((g * nrhs + 15) / 16 * 16) * 8 > 64 * 1024) --g;
        // even groups
        g = (run + (run + g - 1) / g - 1) / ((run + g - 1) / g);
        for (int j = 0; j < run; j += g)
          for (int mt = 0; mt < tree_mt(rows) || (mt == 0 && rows == 0); mt += wm)
            tasks.push_back({i + j, std::min(g, run - j), mt, 0});
        nmax = std::max(nmax, g * nrhs);
        i += run;
      }
      L.ct = (nmax + 15) / 16;
      L.ldn = 16;
      if (L.ct == 1) { L.ldn = 1; while (L.ldn < nmax) L.ldn *= 2; }
      size_t v = 0;
      for (size_t k = first; k < tasks.size(); ++k) {
        const TreeType& t = T.type[T.node[tasks[k].node].type];
        const size_t Kr = ((dir ? t.ni + t.nb : t.ni) + 7) / 8 * 8;
        v = std::max(v, Kr * (L.ct == 1 ? (size_t)L.ldn : (size_t)(tasks[k].count * nrhs + 15) / 16 * 16));
      }
      // the product reads every column tile of its width
      if (L.ct > 1) v = std::max(v, (size_t)kl * 16 * L.ct);
      L.lds = std::max(v, (size_t)TW * 16 * L.ct * 17) * sizeof(double);
      if (L.ct > 3 || L.lds > 160 * 1024) return SEMX_E_UNSUPPORTED;
      L.first = first;
      L.ntask = (int)(tasks.size() - first);
      out.push_back(L);
    }
  return SEMX_OK;
}

// Contribution scratch for nf fields and the launch lists of every field
// count up to that (their tasks in one allocation): a solve of fewer fields
// may be captured into a graph without a call of its own before it.
int tree_scratch(Helm& H, int nf) {
  Tree& T = H.tree;
  TreeDev* D = H.d.tree;
  int st;
  if (nf <= D->nf_cap) return SEMX_OK;
  retire(H, D->C); retire(H, D->Y);
  D->nf_cap = 0;
  const size_t np = (size_t)H.nplanes * nf;
  if ((st = dev_upload<double>(&D->C, nullptr, np * T.nslot_c))) return st;
  if ((st = dev_upload<double>(&D->Y, nullptr, np * T.nslot_y))) return st;
  int npl = 1;
  for (int m : H.dmode) if (H.mode_plane[2 * m + 1] >= 0) npl = 2;
  retire(H, D->task);
  std::vector<TreeTask> tasks;
  for (int f = 1; f <= nf; ++f) {
    D->list[f].clear();
    if ((st = tree_lists(T, npl * f, D->list[f], tasks))) return st;
  }
  if ((st = dev_upload(&D->task, tasks.data(), tasks.size()))) return st;
  D->nf_cap = nf;
  return SEMX_OK;
}

void tree_release(Helm& H) {
  TreeDev* D = H.d.tree;
  if (!D) return;
  dev_free(D->mat); dev_free(D->type); dev_free(D->node); dev_free(D->gid);
  dev_free(D->rowptr); dev_free(D->src); dev_free(D->C); dev_free(D->Y);
  dev_free(D->task);
  delete D;
  H.d.tree = nullptr;
}

// The boundary systems of every direct mode for nf fields: Fb (condensed
// element-boundary right-hand sides) in, sol (solved unknowns) out.
int tree_solve(Helm& H, int nf, size_t pFb, size_t psol, hipStream_t s) {
  Tree& T = H.tree;
  TreeDev* D = H.d.tree;
  const Mesh& M = *H.M;
  TreeArgs a;
  a.type = D->type; a.node = D->node; a.gid = D->gid; a.rowptr = D->rowptr; a.src = D->src;
  a.mat = D->mat; a.mstride = T.mstride; a.dmode = H.d.dmode; a.mode_plane = H.d.mode_plane;
  a.Fb = H.d.Fb; a.C = D->C; a.Y = D->Y; a.sol = H.d.sol;
  a.fbS = M.nel * M.next; a.cS = T.nslot_c; a.yS = T.nslot_y; a.solS = H.solstride;
  a.fbF = (long long)pFb; a.solF = (long long)psol;
  a.cF = (long long)H.nplanes * T.nslot_c; a.yF = (long long)H.nplanes * T.nslot_y;
  a.npl = 1;
  for (int m : H.dmode) if (H.mode_plane[2 * m + 1] >= 0) a.npl = 2;
  a.nrhs = a.npl * nf;
  int nleaf = a.fbS;
  const std::vector<TreeList>& L = D->list[nf];
  hipEvent_t ev;
  prof_begin(s, &ev);
  for (int k = 0; k < 2 * T.nstage - 1; ++k) {
    const bool up = k < T.nstage - 1, root = k == T.nstage - 1;
    const TreeList& l = up ? L[k] : L[T.nstage + (2 * T.nstage - 2 - k)];
    const void* fn = nullptr;
    if (up)
      fn = l.ct == 1 ? (const void*)k_tree_up<1> : l.ct == 2 ? (const void*)k_tree_up<2>
                                                             : (const void*)k_tree_up<3>;
    else if (root)
      fn = l.ct == 1 ? (const void*)k_tree_down<1, true>
                     : l.ct == 2 ? (const void*)k_tree_down<2, true> : (const void*)k_tree_down<3, true>;
    else
      fn = l.ct == 1 ? (const void*)k_tree_down<1, false>
                     : l.ct == 2 ? (const void*)k_tree_down<2, false> : (const void*)k_tree_down<3, false>;
    if (!l.ntask) continue;
    a.task = D->task + l.first; a.wk = l.wk; a.ldn = l.ldn;
    if (l.lds > 64 * 1024)
      HIPCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds));
    void* kargs[] = {&a, &nleaf};
    HIPCHK(hipLaunchKernel(fn, dim3((unsigned)l.ntask, (unsigned)H.dmode.size()), dim3(TT), kargs,
                           l.lds, s));
  }
  prof_end(s, "k_tree", ev);
  return SEMX_OK;
}

}  // namespace semx
