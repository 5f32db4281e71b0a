// semx_elem.hip -- the element ends of Field::solve on CDNA4: every
// element's right-hand side before the boundary systems and its solution
// after them.
//
//   k_lift   boundary terms of the elements that have any: -H g for the
//            essential values g (Field::constrain, src/field.cpp:728-768)
//            plus <h, w> (Natural::sum, src/condition.cpp:192-219)
//   k_cond   direct modes: F = -(M f) + those terms, F_b - hbi F_i
//            (Element::local2globalSumSC, src/element.cpp:356-395)
//   k_back   direct modes: u_i = hii F_i - hbi^T u_b, essential values
//            re-imposed (Element::global2localSC, src/element.cpp:398-438)
//   k_force  PCG modes: F alone, boundary and interior parts
//   k_end3   k_cond and k_back for np = 3
//
// Condensation and recovery are products of one small matrix per mode and
// geometric set with as many columns as there are elements of that set,
// planes and fields, so they run on the FP64 matrix cores.  A workgroup
// takes a group of elements of one set with all right-hand sides of a mode:
// their values come in as whole contiguous elements, sit in LDS one column
// each (boundary first, then interior: emap order), and leave as whole
// elements.  The interior recovery is hii (-M f)_i - hbi^T u_b over ALL
// boundary values: H_ib g = hii^-1 hbi^T g, so essential ones need no
// lifting there, and the forcing is read again in place of an interior part
// kept in memory.
//
// What bounds them: memory traffic (f in, F_b out; f and the solved
// unknowns in, u out) and, on small systems, one round of memory latency.
// Measured, condensation + recovery, us (before: one thread per row, one
// launch per field, the lifting inside): 16x16 quads np=9 Nz=64 34 + 26 ->
// 9 + 19 and k_lift 10; 32x32 np=11 Nz=16 63 + 47 -> 12 + 24 and 8; three
// fields on 20x12 np=8 Nz=32 38 + 35 -> 10 + 15 and 6; 24x24 np=9 Nz=96 68 +
// 73 -> 20 + 42; 11x7 np=6 Nz=36 of elements each with its own matrices 12 +
// 8 -> 6 + 6 and 5.  k_back at 24x24 moves 100 MB: 2.4 TB/s, its gather of
// solved unknowns and three barriers with 12 waves a CU in the way of more.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <numeric>
#include <vector>

#include "semx_hip.h"

namespace semx {

typedef double elem_d4 __attribute__((ext_vector_type(4)));

struct ElemList {               // element groups for one field count
  size_t first = 0;             // of its groups
  int ngrp = 0, ncol = 1;
};

struct ElemDev {
  double* cond = nullptr;       // per direct mode and set: hbi, packed
  double* back = nullptr;       // [-hbi^T | hii], packed
  int* elist = nullptr;         // elements ordered by geometric set
  int* bidx = nullptr;          // per element: entry of blist, or -1
  int4* blist = nullptr;        // elements with essential or natural sides: number,
                                // set, whether any node is essential
  int4* bsrc = nullptr;         // per blist entry and boundary position: BC-line
                                // indices of its essential value and of its
                                // natural terms (-1: none)
  int nbe = 0;
  double* L = nullptr;          // their boundary terms: field, plane, entry, node
  int nf_cap = 0;
  int4* grp = nullptr;          // groups: first entry of elist, elements, set
  ElemList list[SEMX_MAX_FIELDS + 1];
};

namespace {

constexpr int ET = 256;         // threads per workgroup
constexpr int EW = ET / 64;
// columns a wavefront loads together, by nodes per lane
constexpr int end_cols(int nj) { return nj <= 2 ? 8 : 4; }
constexpr int END_FEW = 2;      // the same for groups of at most 2 columns a wavefront

struct EndArgs {
  int np, npnp, next, nint, nel, planeSize, nline, nsolve, nplanes, nset, nbe, ld, npl, nrhs;
  int solstride, ngrp, lds;         // lds: doubles of a group (W = 1)
  const int4* grp;
  const int* elist;
  const int* bidx;
  const int* eset;
  const int* pmap;
  const int* btog;
  const int* ess_src;
  const double* G;
  const double* L;
  const double* mat;
  const int* dmode;
  const int* mode_plane;
  const int* plane_of;
  const int* mode_n;
  double* Fb;
  double* Fi;
  const double* sol;
  long long FbF, FiF, solF, LF;   // strides between fields
  const double* f[SEMX_MAX_FIELDS];
  const double* bc[SEMX_MAX_FIELDS];
  double* u[SEMX_MAX_FIELDS];
};

// The columns of a group, N = elements x right-hand sides <= 64: lane c
// looks up column c once, and the wavefront that works on a column takes
// its scalars from that lane (a chain of scalar loads per column cost more
// than the products).
struct EndCols {
  int e, fld, p, k, ib;
  __device__ EndCols(const EndArgs& a, int m, int4 g) {
    const int c = min((int)(threadIdx.x & 63), g.y * a.nrhs - 1);
    const int r = c / g.y;
    e = a.elist[g.x + c - r * g.y];
    fld = a.npl == 2 ? r >> 1 : r;
    p = a.mode_plane[2 * m + (a.npl == 2 ? r & 1 : 0)];   // < 0: no second plane
    k = p >= 0 ? a.plane_of[p] : 0;
    ib = a.bidx[e];
  }
  struct Col { int e, fld, p, k, ib; };
  __device__ Col col(int c) const {
    return {__builtin_amdgcn_readlane(e, c), __builtin_amdgcn_readlane(fld, c),
            __builtin_amdgcn_readlane(p, c), __builtin_amdgcn_readlane(k, c),
            __builtin_amdgcn_readlane(ib, c)};
  }
};

// LDS order within a group of W wavefronts
template <int W>
__device__ inline void end_sync() {
  if constexpr (W > 1) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Row tile rt of the packed matrix times CT column tiles of the LDS
// columns at vs (K rows, column stride ld), matrix operands four steps
// ahead.  Lanes past the last column repeat it (never stored).
template <int CT>
__device__ inline void end_product(const double* __restrict__ mat, int rt, int KP, const double* vs,
                                   int ld, int c0, int ncol, elem_d4 (&acc)[CT]) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const double* v[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    acc[c] = elem_d4{0.0, 0.0, 0.0, 0.0};
    v[c] = vs + (size_t)min(c0 + 16 * c + li, ncol - 1) * ld + lk;
  }
  const double2* A = reinterpret_cast<const double2*>(mat) + (size_t)rt * KP * 64 + lane;
  double2 q[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) q[u] = A[(size_t)min(u, KP - 1) * 64];
  for (int k = 0; k < KP; k += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double2 av = q[u];
      q[u] = A[(size_t)min(k + u + 4, KP - 1) * 64];
      if (k + u < KP) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, v[c][8 * (k + u)], acc[c], 0, 0, 0);
          acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, v[c][8 * (k + u) + 4], acc[c], 0, 0, 0);
        }
      }
    }
  }
}

// One wavefront per (boundary element, plane, field), NJ nodes per lane;
// everything the products need is loaded ahead of the first barrier.
template <int NJ>
__global__ __launch_bounds__(ET) void k_lift(EndArgs a, const int4* __restrict__ blist,
                                             const int4* __restrict__ bsrc,
                                             const double* __restrict__ ops,
                                             const double* __restrict__ hcon,
                                             const double* __restrict__ mq,
                                             const double* __restrict__ barea, int svv,
                                             double* __restrict__ L) {
  extern __shared__ double lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int np = a.np, npnp = a.npnp, next = a.next;
  double* sD = lds;
  double* sT = sD + npnp;
  double* sU = sT + npnp + (size_t)wave * 3 * npnp;
  double* sR = sU + npnp;
  double* sS = sR + npnp;
  const int ib = min(blockIdx.x * EW + wave, a.nbe - 1), p = blockIdx.y, fld = blockIdx.z;
  const bool live = blockIdx.x * EW + wave < a.nbe;
  const int4 be = blist[ib];                      // element, set, essential
  const int k = a.plane_of[p], m = k >> 1, set = be.y;
  const bool em = be.z != 0;                      // uniform over the wavefront
  const double* bc = a.bc[fld] + (size_t)k * a.nline;
  const double* g = a.G + (size_t)set * G_N * npnp;
  const double* q4 = mq ? mq + ((size_t)m * a.nset + set) * npnp : g + G_Q4 * npnp;
  const double hc = hcon[m];
  double nat[NJ], f1[NJ], f2[NJ], f3[NJ], f4[NJ];
  int pos[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int i = min(lane + 64 * j, npnp - 1);
    pos[j] = a.pmap[i];
    f1[j] = g[G_Q1 * npnp + i];
    f2[j] = g[G_Q2 * npnp + i];
    f3[j] = g[G_Q3 * npnp + i];
    f4[j] = q4[i] * hc;
    nat[j] = 0.0;
    double v = 0.0;
    if (pos[j] < next) {
      const int4 src = bsrc[ib * next + pos[j]];
      if (src.x >= 0) v = bc[src.x];
      if (src.y >= 0) nat[j] += bc[src.y] * barea[src.y];
      if (src.z >= 0) nat[j] += bc[src.z] * barea[src.z];
    }
    sU[i] = v;
  }
  for (int i = tid; i < npnp; i += ET) {
    sD[i] = ops[(svv ? 2 : 0) * npnp + i];
    sT[i] = ops[(svv ? 3 : 1) * npnp + i];
  }
  __syncthreads();
  double F[NJ];
#pragma unroll
  for (int n = 0; n < NJ; ++n) {
    const int pt = min(lane + 64 * n, npnp - 1), i = pt / np, j = pt - i * np;
    F[n] = f4[n] * sU[pt];
    double r = 0.0, s = 0.0;
    if (em) {
      for (int q = 0; q < np; ++q) {
        r += sU[i * np + q] * sT[q * np + j];
        s += sD[i * np + q] * sU[q * np + j];
      }
      sR[pt] = f1[n] * r + f3[n] * s;
      sS[pt] = f2[n] * s + f3[n] * r;
    }
  }
  __syncthreads();
  if (!live) return;
  double* out = L + fld * a.LF + ((size_t)p * a.nbe + ib) * npnp;
#pragma unroll
  for (int n = 0; n < NJ; ++n) {
    const int pt = lane + 64 * n, i = pt / np, j = pt - i * np;
    if (pt >= npnp) continue;
    double T = 0.0;
    if (em) {
      double s1 = 0.0, s3 = 0.0;
      for (int q = 0; q < np; ++q) {
        s1 += sT[i * np + q] * sS[q * np + j];
        s3 += sR[i * np + q] * sD[q * np + j];
      }
      T = F[n] + s1;
      T += s3;
    }
    out[pos[n]] = nat[n] - T;
  }
}

__global__ __launch_bounds__(ET) void k_force(EndArgs a, const int* __restrict__ pcg_plane) {
  const int idx = blockIdx.x * ET + threadIdx.x;
  if (idx >= a.nel * a.npnp) return;
  const int e = idx / a.npnp, q = idx - e * a.npnp, b = a.pmap[q];
  const int p = pcg_plane[blockIdx.y], fld = blockIdx.z, ib = a.bidx[e];
  double v = -(a.G[((size_t)a.eset[e] * G_N + G_Q4) * a.npnp + q] *
               a.f[fld][(size_t)a.plane_of[p] * a.planeSize + idx]);
  if (ib >= 0) v += a.L[fld * a.LF + ((size_t)p * a.nbe + ib) * a.npnp + b];
  const size_t pe = (size_t)p * a.nel + e;
  if (b < a.next) a.Fb[fld * a.FbF + pe * a.next + b] = v;
  else a.Fi[fld * a.FiF + pe * a.nint + (b - a.next)] = v;
}

// A wavefront brings in whole columns (NJ nodes per lane, EU columns in
// flight; the column's field, plane and element sit in scalar registers).
// A group is worked on by W wavefronts: the workgroup's, or one of them (see
// end_launch).
template <int CT, int NJ, int EU, int W>
__global__ __launch_bounds__(ET) void k_cond(EndArgs a) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, wave = W > 1 ? wave_id() : 0;
  const int gi = W > 1 ? blockIdx.x : blockIdx.x * EW + wave_id();
  if (W == 1 && gi >= a.ngrp) return;
  double* vs = lds + (W > 1 ? 0 : wave_id() * a.lds);
  const int4 g = a.grp[gi];
  const int im = blockIdx.y, m = a.dmode[im];
  const EndCols cols(a, m, g);
  const int npnp = a.npnp, next = a.next, ld = a.ld, N = g.y * a.nrhs;
  const int set = g.z;
  const int MT = (next + 15) >> 4, KP = (a.nint + 7) >> 3, ctn = (N + 15) >> 4;
  const double* mat = a.mat + ((size_t)im * a.nset + set) * ((size_t)MT * KP * 128);
  const int npair = (ctn + CT - 1) / CT;
  double q4[NJ];
  int b[NJ], pt[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    pt[j] = min(lane + 64 * j, npnp - 1);
    q4[j] = -a.G[((size_t)set * G_N + G_Q4) * npnp + pt[j]];
    b[j] = a.pmap[pt[j]];
  }
  for (int c0 = wave; c0 < N; c0 += W * EU) {
    // loads without a condition (lanes past the last node repeat it), so
    // that all of them are in flight together
    double f[EU][NJ], l[EU][NJ];
#pragma unroll
    for (int u = 0; u < EU; ++u) {
      const EndCols::Col q = cols.col(min(c0 + u * W, N - 1));
      const double* fp = a.f[q.fld] + (size_t)q.k * a.planeSize + (size_t)q.e * npnp;
#pragma unroll
      for (int j = 0; j < NJ; ++j) f[u][j] = fp[pt[j]];
    }
#pragma unroll
    for (int u = 0; u < EU; ++u) {
      const EndCols::Col q = cols.col(min(c0 + u * W, N - 1));
      const double* lp = a.L + q.fld * a.LF + ((size_t)q.p * a.nbe + q.ib) * npnp;
#pragma unroll
      for (int j = 0; j < NJ; ++j) l[u][j] = 0.0;
      if (q.ib >= 0 && q.p >= 0)
#pragma unroll
        for (int j = 0; j < NJ; ++j) l[u][j] = lp[b[j]];
    }
#pragma unroll
    for (int u = 0; u < EU; ++u)
      if (c0 + u * W < N) {
        const bool on = cols.col(c0 + u * W).p >= 0;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          if (lane + 64 * j < npnp)
            vs[(c0 + u * W) * ld + b[j]] = on ? q4[j] * f[u][j] + l[u][j] : 0.0;
        if (lane < ld - npnp) vs[(c0 + u * W) * ld + npnp + lane] = 0.0;
      }
  }
  end_sync<W>();
  for (int t = wave; t < MT * npair; t += W) {
    const int rt = t / npair, c0 = (t - rt * npair) * CT * 16;
    elem_d4 acc[CT];
    end_product<CT>(mat, rt, KP, vs + next, ld, c0, N, acc);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = c0 + 16 * c + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rt * 16 + 4 * r + (lane >> 4);
        // boundary rows: no product reads them
        if (row < next && col < N) vs[col * ld + row] -= acc[c][r];
      }
    }
  }
  end_sync<W>();
  for (int c = wave; c < N; c += W) {
    const EndCols::Col q = cols.col(c);
    if (q.p >= 0 && lane < next)
      a.Fb[q.fld * a.FbF + ((size_t)q.p * a.nel + q.e) * next + lane] = vs[c * ld + lane];
  }
}

template <int CT, int NJ, int EU, int W>
__global__ __launch_bounds__(ET) void k_back(EndArgs a) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, wave = W > 1 ? wave_id() : 0;
  const int gi = W > 1 ? blockIdx.x : blockIdx.x * EW + wave_id();
  if (W == 1 && gi >= a.ngrp) return;
  double* vs = lds + (W > 1 ? 0 : wave_id() * a.lds);
  const int4 g = a.grp[gi];
  const int im = blockIdx.y, m = a.dmode[im], n = a.mode_n[m];
  const EndCols cols(a, m, g);
  const int npnp = a.npnp, next = a.next, ld = a.ld, N = g.y * a.nrhs;
  const int set = g.z;
  const int MT = (a.nint + 15) >> 4, KP = (npnp + 7) >> 3, ctn = (N + 15) >> 4;
  const double* mat = a.mat + ((size_t)im * a.nset + set) * ((size_t)MT * KP * 128);
  const int npair = (ctn + CT - 1) / CT;
  double q4[NJ];
  int b[NJ], pt[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    pt[j] = min(lane + 64 * j, npnp - 1);
    q4[j] = -a.G[((size_t)set * G_N + G_Q4) * npnp + pt[j]];
    b[j] = a.pmap[pt[j]];
  }
  for (int c0 = wave; c0 < N; c0 += W * EU) {
    double f[EU][NJ], v[EU][NJ];
    int gid[EU][NJ];
    // forcing and node numbers, then the solved values of boundary nodes (a
    // pinned node holds zero); loads without a condition, see k_cond
#pragma unroll
    for (int u = 0; u < EU; ++u) {
      const EndCols::Col q = cols.col(min(c0 + u * W, N - 1));
      const double* fp = a.f[q.fld] + (size_t)q.k * a.planeSize + (size_t)q.e * npnp;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        gid[u][j] = a.btog[q.e * next + min(b[j], next - 1)];
        f[u][j] = fp[pt[j]];
      }
    }
#pragma unroll
    for (int u = 0; u < EU; ++u) {
      const EndCols::Col q = cols.col(min(c0 + u * W, N - 1));
      const double* sp = a.sol + q.fld * a.solF + (size_t)max(q.p, 0) * a.solstride;
#pragma unroll
      for (int j = 0; j < NJ; ++j) v[u][j] = sp[gid[u][j] < n ? gid[u][j] : 0];
    }
#pragma unroll
    for (int u = 0; u < EU; ++u)
      if (c0 + u * W < N) {
        const EndCols::Col q = cols.col(c0 + u * W);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          if (gid[u][j] >= n) v[u][j] = 0.0;
          if (q.ib >= 0 && gid[u][j] >= a.nsolve)
            v[u][j] = a.bc[q.fld][(size_t)q.k * a.nline + a.ess_src[gid[u][j] - a.nsolve]];
          if (b[j] >= next) v[u][j] = q4[j] * f[u][j];
          if (lane + 64 * j < npnp) vs[(c0 + u * W) * ld + b[j]] = q.p >= 0 ? v[u][j] : 0.0;
        }
        if (lane < ld - npnp) vs[(c0 + u * W) * ld + npnp + lane] = 0.0;
      }
  }
  end_sync<W>();
  const int lo = a.nint | 1;
  // the products read the interior values of every row tile: results go to
  // the part of LDS after the columns
  double* out = vs + (size_t)N * ld;
  for (int t = wave; t < MT * npair; t += W) {
    const int rt = t / npair, c0 = (t - rt * npair) * CT * 16;
    elem_d4 acc[CT];
    end_product<CT>(mat, rt, KP, vs, ld, c0, N, acc);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = c0 + 16 * c + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rt * 16 + 4 * r + (lane >> 4);
        if (row < a.nint && col < N) out[col * lo + row] = acc[c][r];
      }
    }
  }
  end_sync<W>();
  for (int c = wave; c < N; c += W) {
    const EndCols::Col q = cols.col(c);
    if (q.p < 0) continue;
    double* up = a.u[q.fld] + (size_t)q.k * a.planeSize + (size_t)q.e * npnp;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (lane + 64 * j < npnp)
        up[lane + 64 * j] = b[j] < next ? vs[c * ld + b[j]] : out[c * lo + (b[j] - next)];
  }
}

// np = 3: eight boundary nodes and one interior one, a thread per node and
// right-hand side; the same matrices.
template <bool BACK>
__global__ __launch_bounds__(ET) void k_end3(EndArgs a) {
  const int idx = blockIdx.x * ET + threadIdx.x;
  if (idx >= a.nel * 9) return;
  const int e = idx / 9, pt = idx - 9 * e, im = blockIdx.y, m = a.dmode[im];
  const int fld = blockIdx.z / a.npl, p = a.mode_plane[2 * m + blockIdx.z % a.npl];
  if (p < 0) return;
  const int k = a.plane_of[p], b = a.pmap[pt], set = a.eset[e], ib = a.bidx[e];
  const double* q4 = a.G + ((size_t)set * G_N + G_Q4) * 9;
  const double* f = a.f[fld] + (size_t)k * a.planeSize + (size_t)e * 9;
  const double fi = -(q4[4] * f[4]);               // the interior node
  if constexpr (!BACK) {
    if (b == 8) return;
    const double* L = a.L + fld * a.LF + ((size_t)p * a.nbe + max(ib, 0)) * 9;
    const double lb = ib >= 0 ? L[b] : 0.0, li = ib >= 0 ? L[8] : 0.0;
    const double h = a.mat[((size_t)im * a.nset + set) * 128 + 2 * b];
    a.Fb[fld * a.FbF + ((size_t)p * a.nel + e) * 8 + b] = (lb - q4[pt] * f[pt]) - h * (fi + li);
  } else {
    const int n = a.mode_n[m];
    const double* sol = a.sol + fld * a.solF + (size_t)p * a.solstride;
    const double* bc = a.bc[fld] + (size_t)k * a.nline;
    auto node = [&](int c) {                       // a pinned one holds zero
      const int gid = a.btog[e * 8 + c];
      return gid < n ? sol[gid] : gid >= a.nsolve ? bc[a.ess_src[gid - a.nsolve]] : 0.0;
    };
    double v = 0.0;
    if (b < 8) {
      v = node(b);
    } else {
      const double* A = a.mat + ((size_t)im * a.nset + set) * 256;
#pragma unroll
      for (int c = 0; c < 8; ++c) v += A[32 * (c & 3) + (c >> 2)] * node(c);
      v += A[128] * fi;
    }
    a.u[fld][(size_t)k * a.planeSize + (size_t)e * 9 + pt] = v;
  }
}

// hbi (next x nint) and [-hbi^T | hii] (nint x npnp) of one mode's sets in
// the order the matrix cores take them (tree_packed)
__global__ void k_end_pack(const double* __restrict__ hbi, const double* __restrict__ hii, int next,
                           int nint, double* __restrict__ cond, double* __restrict__ back) {
  const int set = blockIdx.y, npnp = next + nint;
  const double* bi = hbi + (size_t)set * next * nint;
  const double* ii = hii + (size_t)set * nint * nint;
  const int kc = (nint + 7) / 8, kb = (npnp + 7) / 8;
  const int nc = (next + 15) / 16 * kc * 128, nb = (nint + 15) / 16 * kb * 128;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nc + nb; i += gridDim.x * blockDim.x) {
    const bool b = i >= nc;
    const int j = b ? i - nc : i, kp = b ? kb : kc;
    const int tile = j >> 7, lane = (j >> 1) & 63;
    const int row = tile / kp * 16 + (lane & 15);
    const int col = (tile % kp) * 8 + (j & 1) * 4 + (lane >> 4);
    double v = 0.0;
    if (!b) {
      if (row < next && col < nint) v = bi[row * nint + col];
      cond[(size_t)set * nc + j] = v;
    } else {
      if (row < nint && col < npnp) v = col < next ? -bi[col * nint + row] : ii[row * nint + col - next];
      back[(size_t)set * nb + j] = v;
    }
  }
}

// k_cond or k_back for npnp nodes, groups of ncol columns and a matrix of mt
// row tiles.  Two column tiles per product (each matrix operand used twice)
// where that leaves no wavefront with more work than single tiles would; few
// columns (elements of their own geometry) load no repeats of them.
const void* end_kernel(bool back, int ncol, int mt, int npnp) {
  int ct = ncol > 16 ? 2 : 1;
  if (2 * ((mt + EW - 1) / EW) > (2 * mt + EW - 1) / EW) ct = 1;
  const void* fn = nullptr;
#define SEMX_END_PICK(K_, NJ_)                                                              \
  (ncol <= EW * END_FEW ? (const void*)K_<1, NJ_, END_FEW, EW>                              \
   : ct == 1            ? (const void*)K_<1, NJ_, end_cols(NJ_), EW>                        \
                        : (const void*)K_<2, NJ_, end_cols(NJ_), EW>)
#define SEMX_END(NJ_)                                                                       \
  if ((npnp + 63) / 64 == NJ_) fn = back ? SEMX_END_PICK(k_back, NJ_) : SEMX_END_PICK(k_cond, NJ_)
  SEMX_END(1); SEMX_END(2); SEMX_END(3); SEMX_END(4);
#undef SEMX_END
#undef SEMX_END_PICK
  return fn;
}

// Condensation or recovery of every group and direct mode.  np = 3 takes a
// thread per node: nine of a wavefront's lanes would work.  np = 4 and 5 with
// geometries of their own take one wavefront per group, four groups per
// workgroup: both matrices are one row tile, so three of the workgroup's
// wavefronts would only load.  Measured, whole solves, us, a workgroup per
// group -> this (the band sweeps' element kernels, a thread per row): 32x32
// distorted np=3 Nz=128 420 -> 187 (204), Nz=32 119 -> 72 (98); 16x16
// distorted np=4 Nz=64 69 -> 54 (64), np=5 82 -> 66 (97); 16x16 uniform np=3
// Nz=128 59 -> 47 (55).
int end_launch(bool back, EndArgs& a, const Mesh& M, const ElemList& l, unsigned nd, hipStream_t s) {
  void* kargs[] = {&a};
  if (M.np == 3) {
    const dim3 grid((M.nel * 9 + ET - 1) / ET, nd, a.nrhs);
    HIPCHK(hipLaunchKernel(back ? (const void*)k_end3<true> : (const void*)k_end3<false>, grid,
                           dim3(ET), kargs, 0, s));
    return SEMX_OK;
  }
  const bool one = tree_mt(M.next) == 1 && tree_mt(M.nint) == 1 && l.ncol <= 2 * SEMX_MAX_FIELDS;
  const void* fn = one ? back ? (const void*)k_back<1, 1, END_FEW, 1> : (const void*)k_cond<1, 1, END_FEW, 1>
                       : end_kernel(back, l.ncol, tree_mt(back ? M.nint : M.next), M.npnp);
  a.ngrp = l.ngrp;
  a.lds = l.ncol * (a.ld + (back ? M.nint | 1 : 0));
  const size_t lds = (size_t)a.lds * (one ? EW : 1) * sizeof(double);
  if (lds > 64 * 1024)
    HIPCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  HIPCHK(hipLaunchKernel(fn, dim3(one ? (l.ngrp + EW - 1) / EW : l.ngrp, nd), dim3(ET), kargs, lds, s));
  return SEMX_OK;
}

}  // namespace

int elem_upload(Helm& H) {
  if (H.d.elem) return SEMX_OK;
  Mesh& M = *H.M;
  ElemDev* D = new ElemDev();
  H.d.elem = D;
  std::vector<int> el(M.nel), bidx(M.nel, -1);
  std::vector<int4> bl;
  std::iota(el.begin(), el.end(), 0);
  std::stable_sort(el.begin(), el.end(), [&](int x, int y) { return M.eset[x] < M.eset[y]; });
  for (int e = 0; e < M.nel; ++e)
    if (M.emask[e] || M.nat_ptr[e + 1] > M.nat_ptr[e]) {
      bidx[e] = (int)bl.size();
      bl.push_back(make_int4(e, M.eset[e], M.emask[e], 0));
    }
  D->nbe = (int)bl.size();
  std::vector<int4> src((size_t)D->nbe * M.next, make_int4(-1, -1, -1, 0));
  for (int i = 0; i < D->nbe; ++i) {
    const int e = bl[i].x;
    int4* r = &src[(size_t)i * M.next];
    for (int b = 0; b < M.next; ++b) {
      const int gid = M.btog[e * M.next + b];
      if (gid >= M.nsolve) r[b].x = M.ess_src[gid - M.nsolve];
    }
    for (int c = M.nat_ptr[e]; c < M.nat_ptr[e + 1]; ++c)
      for (int q = 0; q < M.np; ++q) {      // a corner lies on two sides at most
        const int bb = M.nat_b[c], b = (M.bside[bb] * (M.np - 1) + q) % M.next;
        (r[b].y < 0 ? r[b].y : r[b].z) = bb * M.np + q;
      }
  }
  int st;
  if ((st = dev_upload(&D->elist, el.data(), el.size()))) return st;
  if ((st = dev_upload(&D->bidx, bidx.data(), bidx.size()))) return st;
  if ((st = dev_upload(&D->blist, bl.data(), bl.size()))) return st;
  if ((st = dev_upload(&D->bsrc, src.data(), src.size()))) return st;
  if (H.dmode.empty()) return SEMX_OK;
  const size_t nbi = (size_t)M.nset * M.next * M.nint, nii = (size_t)M.nset * M.nint * M.nint;
  const size_t sc = (size_t)M.nset * tree_packed(M.next, M.nint);
  const size_t sb = (size_t)M.nset * tree_packed(M.nint, M.npnp);
  double *bi = nullptr, *ii = nullptr;
  if ((st = dev_upload<double>(&D->cond, nullptr, sc * H.dmode.size()))) return st;
  if ((st = dev_upload<double>(&D->back, nullptr, sb * H.dmode.size()))) return st;
  st = dev_upload<double>(&bi, nullptr, nbi);
  if (!st) st = dev_upload<double>(&ii, nullptr, nii);
  for (size_t k = 0; k < H.dmode.size() && !st; ++k) {
    const int m = H.dmode[k];
    // blocking copies, ordered after the previous mode's packing
    if (hipMemcpy(bi, &H.hbi[m * nbi], nbi * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(ii, &H.hii[m * nii], nii * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
      st = SEMX_E_HIP;
      break;
    }
    const int nb = (int)std::min<long long>(64, (long long)(tree_packed(M.next, M.nint) +
                                                             tree_packed(M.nint, M.npnp) + 255) / 256);
    hipLaunchKernelGGL(k_end_pack, dim3(nb, M.nset), dim3(256), 0, nullptr, bi, ii, M.next, M.nint,
                       D->cond + k * sc, D->back + k * sb);
    if (hipGetLastError() != hipSuccess) st = SEMX_E_HIP;
  }
  if (hipStreamSynchronize(nullptr) != hipSuccess && !st) st = SEMX_E_HIP;
  dev_free(bi);
  dev_free(ii);
  return st;
}

void elem_release(Helm& H) {
  ElemDev* D = H.d.elem;
  if (!D) return;
  dev_free(D->cond); dev_free(D->back); dev_free(D->elist); dev_free(D->bidx); dev_free(D->blist);
  dev_free(D->bsrc); dev_free(D->L);
  dev_free(D->grp);
  delete D;
  H.d.elem = nullptr;
}

// Column stride of the LDS tile: every matrix step's rows, odd so that the
// 16 columns a matrix operand reads fall in distinct banks.
static int end_ld(const Mesh& M) {
  return std::max(M.next + (M.nint + 7) / 8 * 8, (M.npnp + 7) / 8 * 8) | 1;
}

// The element groups of nf fields: two column tiles (32 columns) per
// workgroup, or one where two would leave fewer than 512 workgroups (two per
// CU).
static void elem_list(const Helm& H, int nf, ElemList& l, std::vector<int4>& groups) {
  const Mesh& M = *H.M;
  int npl = 1;
  for (int m : H.dmode) if (H.mode_plane[2 * m + 1] >= 0) npl = 2;
  const int nrhs = npl * nf;
  const size_t col = ((size_t)end_ld(M) + (M.nint | 1)) * sizeof(double);
  int ge = std::max(1, 32 / nrhs);
  while (ge > 1 && ge * nrhs * col > 64 * 1024) --ge;
  std::vector<int> order(M.eset);       // the sets along D->elist
  std::sort(order.begin(), order.end());
  auto split = [&](int w) {
    std::vector<int4> g;
    for (int i = 0; i < M.nel;) {
      int run = 0;
      while (i + run < M.nel && order[i + run] == order[i]) ++run;
      const int parts = (run + w - 1) / w;
      for (int k = 0; k < parts; ++k) {
        const int a = (int)((long long)run * k / parts), b = (int)((long long)run * (k + 1) / parts);
        g.push_back(make_int4(i + a, b - a, order[i], 0));
      }
      i += run;
    }
    return g;
  };
  std::vector<int4> g = split(ge);
  if (g.size() * H.dmode.size() < 512 && ge * nrhs > 16) g = split(std::max(1, 16 / nrhs));
  int nmax = 1;
  for (const int4& q : g) nmax = std::max(nmax, q.y * nrhs);
  l.ncol = nmax;                        // np <= 16: at most 32 x 4 KB
  l.ngrp = (int)g.size();
  l.first = groups.size();
  groups.insert(groups.end(), g.begin(), g.end());
}

// Boundary-term scratch for nf fields and the element groups of every field
// count up to that (see tree_scratch).
int elem_scratch(Helm& H, int nf) {
  ElemDev* D = H.d.elem;
  int st;
  if (nf <= D->nf_cap) return SEMX_OK;
  retire(H, D->L);
  D->nf_cap = 0;
  if ((st = dev_upload<double>(&D->L, nullptr, (size_t)H.nplanes * nf * D->nbe * H.M->npnp))) return st;
  if (!H.dmode.empty()) {
    retire(H, D->grp);
    std::vector<int4> groups;
    for (int f = 1; f <= nf; ++f) elem_list(H, f, D->list[f], groups);
    if ((st = dev_upload(&D->grp, groups.data(), groups.size()))) return st;
  }
  D->nf_cap = nf;
  return SEMX_OK;
}

static EndArgs end_args(Helm& H, int nf, double* const* fs, const double* const* bcs,
                        double* const* us, size_t pFb, size_t pFi, size_t psol) {
  Mesh& M = *H.M;
  const ElemDev& D = *H.d.elem;
  EndArgs a{};
  a.np = M.np; a.npnp = M.npnp; a.next = M.next; a.nint = M.nint; a.nel = M.nel;
  a.planeSize = M.planeSize; a.nline = M.nbound * M.np; a.nsolve = M.nsolve;
  a.nplanes = H.nplanes; a.nset = M.nset; a.nbe = D.nbe; a.ld = end_ld(M);
  a.npl = 1;
  for (int m : H.dmode) if (H.mode_plane[2 * m + 1] >= 0) a.npl = 2;
  a.nrhs = a.npl * nf;
  a.solstride = H.solstride;
  a.grp = D.grp + D.list[nf].first; a.elist = D.elist; a.bidx = D.bidx;
  a.eset = M.d.eset; a.pmap = M.d.pmap; a.btog = M.d.btog;
  a.ess_src = M.d.ess_src; a.G = M.d.G; a.L = D.L;
  a.dmode = H.d.dmode; a.mode_plane = H.d.mode_plane; a.plane_of = H.d.plane_of;
  a.mode_n = H.d.mode_n;
  a.Fb = H.d.Fb; a.Fi = H.d.Fi; a.sol = H.d.sol;
  a.FbF = (long long)pFb; a.FiF = (long long)pFi; a.solF = (long long)psol;
  a.LF = (long long)H.nplanes * D.nbe * M.npnp;
  for (int i = 0; i < nf; ++i) {
    a.f[i] = fs[i];
    a.bc[i] = bcs ? bcs[i] : nullptr;
    a.u[i] = us[i];
  }
  return a;
}

// Element right-hand sides of every mode: d.Fb (condensed for the direct
// ones) and, for PCG planes, d.Fi.
int elem_condense(Helm& H, int nf, double* const* fs, const double* const* bcs, double* const* us,
                  size_t pFb, size_t pFi, size_t psol, hipStream_t s) {
  Mesh& M = *H.M;
  const ElemDev& D = *H.d.elem;
  EndArgs a = end_args(H, nf, fs, bcs, us, pFb, pFi, psol);
  hipEvent_t ev;
  if (D.nbe) {
    const size_t lds = (2 + 3 * (size_t)EW) * M.npnp * sizeof(double);   // 28 KB at np = 16
    prof_begin(s, &ev);
    const dim3 grid((D.nbe + EW - 1) / EW, H.nplanes, nf);
    const int svv = H.lambda2 > EPSDP ? 1 : 0;
#define SEMX_LIFT(NJ_)                                                                     \
  if ((M.npnp + 63) / 64 == NJ_)                                                           \
    hipLaunchKernelGGL(k_lift<NJ_>, grid, dim3(ET), lds, s, a, D.blist, D.bsrc, M.d.ops,   \
                       H.d.hcon, H.d.mq, M.d.barea, svv, D.L)
    SEMX_LIFT(1); SEMX_LIFT(2); SEMX_LIFT(3); SEMX_LIFT(4);
#undef SEMX_LIFT
    prof_end(s, "k_lift", ev);
  }
  if (!H.dmode.empty()) {
    const ElemList& l = D.list[nf];
    a.mat = D.cond;
    prof_begin(s, &ev);
    if (const int st = end_launch(false, a, M, l, (unsigned)H.dmode.size(), s)) return st;
    prof_end(s, "k_condense", ev);
  }
  if (!H.pcg_plane.empty()) {
    prof_begin(s, &ev);
    hipLaunchKernelGGL(k_force, dim3((M.nel * M.npnp + ET - 1) / ET, (unsigned)H.pcg_plane.size(), nf),
                       dim3(ET), 0, s, a, H.d.pcg_plane);
    prof_end(s, "k_condense", ev);
  }
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

// Solutions of the direct modes from d.sol.
int elem_backsub(Helm& H, int nf, double* const* fs, const double* const* bcs, double* const* us,
                 size_t pFb, size_t pFi, size_t psol, hipStream_t s) {
  const Mesh& M = *H.M;
  const ElemDev& D = *H.d.elem;
  EndArgs a = end_args(H, nf, fs, bcs, us, pFb, pFi, psol);
  const ElemList& l = D.list[nf];
  a.mat = D.back;
  hipEvent_t ev;
  prof_begin(s, &ev);
  if (const int st = end_launch(true, a, M, l, (unsigned)H.dmode.size(), s)) return st;
  prof_end(s, "k_backsub", ev);
  return SEMX_OK;
}

}  // namespace semx
