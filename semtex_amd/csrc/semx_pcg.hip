// semx_pcg.hip -- Jacobi-preconditioned CG with a plane's vectors held on
// chip: semtex's JACPCG branch of Field::solve (src/field.cpp:627-720) with
// the global operator of Field::HelmholtzOperator (src/field.cpp:771-856).
//
// A plane's elements are split over the fewest workgroups whose registers
// and LDS hold them; thread (element, column j) keeps the element's column j
// of x, r, p and the preconditioner in registers, nodes shared by elements
// repeated in each (the same bits in every copy), and nothing of the
// iteration but the results at nodes shared by two workgroups goes through
// memory.  Per iteration: the element operator inside each wavefront (whole
// elements per wavefront, so no block barrier), the direct-stiffness sum of
// the element-boundary results through LDS, and two sums over the plane.
//
// What bounds it: the two exchanges between a plane's workgroups (one way
// through the memory-side cache each) and the operator's FP64 arithmetic; the
// kernel it stands in for (k_pcg) reads and writes every vector in global
// memory each iteration and meets at four grid barriers whose fences write
// back the L2.
//
// Eight wavefronts of 256 registers, not twelve of 168: those spilled up to
// 291 registers (np = 11, FP64) inside the iteration, whose traffic was most
// of its time.  us a solve, twelve wavefronts with shuffle sums -> eight with
// row shifts -> boundary slots at constant offsets, awaited values two at a
// time, general factors and preconditioner in registers up to np = 7, one
// kernel per np: 32x32 np=11 Nz=128 MIXED 72200 -> 40500 -> 32700; 512 mixed
// 2D problems FP32 refined 25900 -> 15700 -> 12900; 9x6 np=7 one distorted
// plane 2480 -> 1754 -> 1343; 16x16 np=9 Nz=64 FP32 refined 633 -> 621 -> 550.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "semx_chip.h"

namespace semx {

namespace {

constexpr int CT = 512;                 // threads: 8 wavefronts, 256 registers each
constexpr int CWV = CT / 64;
constexpr int CHIP_WMAX = 48;           // workgroups of one problem at most
constexpr int CHIP_NPMIN = 4, CHIP_NPMAX = 12;
constexpr int CHIP_NPREG = 7;         // at 8 they spill
constexpr long CHIP_SPIN = 1L << 22;    // polls before a wait gives up
constexpr unsigned long long CHIP_SENT = 0x7FF4DEADBEEF0001ull;   // signalling NaN
constexpr int CHIP_RED = 4 * CWV + CWV + 8 + CHIP_WMAX;   // LDS doubles of the sums

constexpr int chip_epw(int np) { return 64 / np; }
constexpr int chip_ldr(int np) { return np | 1; }

__device__ inline double ch_ld(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void ch_st(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void ch_reset(double* p) {
  ch_st(p, __longlong_as_double((long long)CHIP_SENT));
}
// Waits (bounded) for a slot's value.  A slot holds a signalling NaN, which
// arithmetic never produces, until its producer stores the value, so a
// consumer needs no separate flag.
__device__ inline double ch_take(const double* p, bool& dead) {
  double v = ch_ld(p);
  long it = 0;
  while ((unsigned long long)__double_as_longlong(v) == CHIP_SENT) {
    if (dead || ++it > CHIP_SPIN) { dead = true; return 0.0; }
    __builtin_amdgcn_s_sleep(1);
    v = ch_ld(p);
  }
  return v;
}

__device__ inline void ch_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// a block barrier that also waits for this wavefront's global stores: what
// a thread contributes after it is seen after what it stored before it
__device__ inline void ch_barrier_mem() {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
}

template <typename T> struct ConstPtr { typedef const __attribute__((address_space(4))) T* type; };
template <typename T>
__device__ inline typename ConstPtr<T>::type ch_const(const T* p) {   // a workgroup-uniform pointer
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
  return (typename ConstPtr<T>::type)(((unsigned long long)hi << 32) | lo);
}

// The state of a workgroup.
struct Wg {
  int W, w, ne, nslot, nrem, npub;
  bool dead;
  int kA, kB;                  // exchanges and sums done
  double* exch;                // ring of 4 x nif
  double* red;                 // ring of 4 x 3 W
  int nif;
  const int* rem;              // LDS
  const int2* pub;             // LDS
  double* lb;                  // LDS: boundary results (T), received ones, a zero
  double* lb2;                 // LDS: their sums (T)
  const ushort4* tab;          // LDS
  double* rd;                  // LDS: reduction scratch
  int* err;
};

// Sum over the wavefront by row shifts and broadcasts (the data-parallel
// paths: a step costs two moves and an add, where a shuffle through LDS costs
// its latency), the same bits in all lanes.
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double wave_add(double v) {
  v = dpp_add<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Sums of (u, v) over every thread of the problem's workgroups, the same
// bits in all of them: within a workgroup through LDS, then the workgroups'
// partial sums in a fixed order.  Ring of 4 slots per workgroup: the slot
// two sums ahead is reset here, when all have read what it held (they
// contributed to the sum in between after that), and the reset is complete
// before this workgroup's next contribution (ch_barrier_mem).
__device__ inline double2 plane_sum2(Wg& G, double u, double v) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  u = wave_add(u);
  v = wave_add(v);
  double* rb = G.rd + (G.kB & 1) * 2 * CWV;
  if (lane == 0) { rb[2 * wave] = u; rb[2 * wave + 1] = v; }
  ch_barrier_mem();
  double2 t = make_double2(0.0, 0.0);
#pragma unroll
  for (int q = 0; q < CWV; ++q) { t.x += rb[2 * q]; t.y += rb[2 * q + 1]; }
  if (G.W > 1) {
    double* out = G.rd + 5 * CWV + (G.kB & 1) * 2;
    if (wave == 0) {
      double* s = G.red + (size_t)(G.kB & 3) * 3 * G.W;
      double* z = G.red + (size_t)((G.kB + 2) & 3) * 3 * G.W;
      if (lane < 2) {
        ch_st(s + 3 * G.w + 1 + lane, lane ? t.y : t.x);
        ch_reset(z + 3 * G.w + 1 + lane);
      }
      double a = 0.0, b = 0.0;
      if (lane < G.W) {
        a = ch_take(s + 3 * lane + 1, G.dead);
        b = ch_take(s + 3 * lane + 2, G.dead);
      }
      a = wave_add(a);
      b = wave_add(b);
      if (lane == 0) { out[0] = a; out[1] = b; }
    }
    __syncthreads();
    t = make_double2(out[0], out[1]);
  }
  ++G.kB;
  return t;
}

// The boundary results in G.lb summed at every node (the sums in G.lb2),
// with the results of other workgroups, and pq summed over the problem.
// Every copy of a node adds the same terms in the same order.
template <typename T>
__device__ inline double plane_assemble(Wg& G, double pq) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  T* lb = (T*)G.lb;
  T* lb2 = (T*)G.lb2;
  pq = wave_add(pq);
  double* rb = G.rd + 4 * CWV;
  if (lane == 0) rb[wave] = pq;
  if (tid == 0) lb[G.nslot + G.nrem] = 0;
  ch_barrier_mem();
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < CWV; ++q) t += rb[q];
  if (G.W > 1) {
    double* ex = G.exch + (size_t)(G.kA & 3) * G.nif;
    double* zx = G.exch + (size_t)((G.kA + 2) & 3) * G.nif;
    double* xs = G.rd + 5 * CWV + 8;
    double* s = G.red + (size_t)(G.kA & 3) * 3 * G.W;
    for (int i = tid; i < G.npub; i += CT) {
      const int2 p = G.pub[i];
      ch_st(ex + p.y, (double)lb[p.x]);
      ch_reset(zx + p.y);
    }
    if (tid == CT - 1) {
      ch_st(s + 3 * G.w, t);
      ch_reset(G.red + (size_t)((G.kA + 2) & 3) * 3 * G.W + 3 * G.w);
    }
    // received results and the workgroups' partial sums, two per thread asked
    // for before either is waited for
    const int n = G.nrem + G.W;
    for (int i = tid; i < n; i += 2 * CT) {
      const int k = min(i + CT, n - 1);
      const double* p = i < G.nrem ? ex + G.rem[i] : s + 3 * (i - G.nrem);
      const double* q = k < G.nrem ? ex + G.rem[k] : s + 3 * (k - G.nrem);
      double u = ch_ld(p), v = ch_ld(q);
      if ((unsigned long long)__double_as_longlong(u) == CHIP_SENT) u = ch_take(p, G.dead);
      if ((unsigned long long)__double_as_longlong(v) == CHIP_SENT) v = ch_take(q, G.dead);
      if (i < G.nrem) lb[G.nslot + i] = (T)u;
      else xs[i - G.nrem] = u;
      if (k < G.nrem) lb[G.nslot + k] = (T)v;
      else xs[k - G.nrem] = v;
    }
    __syncthreads();
    t = wave_add(lane < G.W ? xs[lane] : 0.0);
  }
  // two slots at a time and without conditions, so that their reads are in
  // flight together: absent terms read the zero, threads past the last slot
  // sum zeros into the spare one
  for (int i = tid; i < G.nslot; i += 2 * CT) {
    const int k = min(i + CT, G.nslot);
    const ushort4 a = G.tab[i], b = G.tab[k];
    const T u = lb[a.x], v = lb[b.x], u1 = lb[a.y], v1 = lb[b.y], u2 = lb[a.z], v2 = lb[b.z],
            u3 = lb[a.w], v3 = lb[b.w];
    lb2[i] = ((u + u1) + u2) + u3;
    lb2[k] = ((v + v1) + v2) + v3;
  }
  __syncthreads();
  ++G.kA;
  return t;
}

// Boundary position (emap order) of node (i, j), -1 inside.
template <int NP>
__device__ inline int bpos(int i, int j) {
  constexpr int nm = NP - 1;
  if (i == 0) return j;
  if (j == nm) return nm + i;
  if (i == nm) return 2 * nm + (nm - j);
  if (j == 0) return 3 * nm + (nm - i);
  return -1;
}
template <int NP>
__device__ inline int bnode(int b) {   // node i * NP + j of boundary position b
  constexpr int nm = NP - 1;
  if (b < nm) return b;
  if (b < 2 * nm) return (b - nm) * NP + nm;
  if (b < 3 * nm) return nm * NP + (3 * nm - b);
  return (4 * nm - b) * NP;
}

// What a thread needs for its column of one element's operator.
template <typename TT, int NP, bool GREG>
struct ElemFac {
  typedef TT T;
  static constexpr bool greg = GREG;
  bool aff;
  T f1, f2, f3, f4;              // parallelograms: Q1..Q4 = f (this column) x weight (row)
  typename ConstPtr<T>::type w;
  const double* g;               // else the set's factors, and the mass factors
  const double* m;
  T q[4][GREG ? NP : 1];         // GREG: these in registers, the last times hcon
  T hcon;
  typename ConstPtr<T>::type D, DT;
};

// a uniform address the compiler takes as new: loads through it stay where
// they are written instead of moving ahead of everything (the scalar
// registers hold two rows of a matrix, not all of it)
template <typename T>
__device__ inline typename ConstPtr<T>::type fresh_ptr(typename ConstPtr<T>::type p) {
  unsigned long long v = (unsigned long long)p;
  asm volatile("" : "+s"(v));
  return ch_const((const T*)v);
}

// fn(q, i, A[q][i]) over a matrix in scalar registers, one row loaded while
// the previous one is used.
template <typename T, int NP, class F>
__device__ inline void scalar_rows(typename ConstPtr<T>::type A, F fn) {
  T t[2][NP];
  {
    const auto a = fresh_ptr<T>(A);
#pragma unroll
    for (int i = 0; i < NP; ++i) t[0][i] = a[i];
  }
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    if (q + 1 < NP) {
      const auto a = fresh_ptr<T>(A);
#pragma unroll
      for (int i = 0; i < NP; ++i) t[(q + 1) & 1][i] = a[(q + 1) * NP + i];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NP; ++i) fn(q, i, t[q & 1][i]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// out = (K + hcon M) p on the thread's element (Element::HelmholtzOp,
// src/element.cpp:1621-1650), columns in registers.  The row products go
// through the element's LDS tile; the operator matrices come as scalars,
// one load serving the row and the column product of a step.
template <typename T, int NP, class Fac>
__device__ inline void elem_apply(const Fac& F, const T (&p)[NP], T (&out)[NP], T* buf, int j) {
  constexpr int LD = chip_ldr(NP), NN = NP * NP;
#pragma unroll
  for (int i = 0; i < NP; ++i) buf[i * LD + j] = p[i];
  ch_wave_sync();
  T R[NP], S[NP], u[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q) u[q] = buf[j * LD + q];
#pragma unroll
  for (int i = 0; i < NP; ++i) R[i] = S[i] = 0;
  scalar_rows<T, NP>(F.DT, [&](int q, int i, T t) {
    R[i] += u[q] * t;            // row j of U D^T
    S[i] += p[q] * t;            // column j of D U
  });
  ch_wave_sync();
#pragma unroll
  for (int i = 0; i < NP; ++i) buf[j * LD + i] = R[i];
  ch_wave_sync();
#pragma unroll
  for (int i = 0; i < NP; ++i) R[i] = buf[i * LD + j];
  // R' = Q1 R + Q3 S, S' = Q2 S + Q3 R, mass term
  if (F.aff) {
    const auto w = fresh_ptr<T>(F.w);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const T wi = w[i], r = R[i], s = S[i];
      R[i] = wi * (F.f1 * r + F.f3 * s);
      S[i] = wi * (F.f2 * s + F.f3 * r);
      out[i] = wi * F.f4 * p[i];
    }
  } else if constexpr (Fac::greg) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const T r = R[i], s = S[i];
      R[i] = F.q[0][i] * r + F.q[2][i] * s;
      S[i] = F.q[1][i] * s + F.q[2][i] * r;
      out[i] = F.q[3][i] * p[i];
    }
  } else {
    const double *g = F.g + j, *m = F.m + j;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const T q1 = (T)g[G_Q1 * NN + i * NP], q2 = (T)g[G_Q2 * NN + i * NP],
              q3 = (T)g[G_Q3 * NN + i * NP], r = R[i], s = S[i];
      R[i] = q1 * r + q3 * s;
      S[i] = q2 * s + q3 * r;
      out[i] = (T)m[i * NP] * F.hcon * p[i];
    }
  }
  ch_wave_sync();
#pragma unroll
  for (int i = 0; i < NP; ++i) buf[i * LD + j] = R[i];
  ch_wave_sync();
#pragma unroll
  for (int q = 0; q < NP; ++q) u[q] = buf[j * LD + q];
#pragma unroll
  for (int i = 0; i < NP; ++i) R[i] = 0;
  scalar_rows<T, NP>(F.D, [&](int q, int i, T t) {
    R[i] += u[q] * t;            // row j of R' D
    out[i] += S[q] * t;          // column j of D^T S'
  });
  ch_wave_sync();
#pragma unroll
  for (int i = 0; i < NP; ++i) buf[j * LD + i] = R[i];
  ch_wave_sync();
#pragma unroll
  for (int i = 0; i < NP; ++i) out[i] += buf[i * LD + j];
  ch_wave_sync();
}

// A thread's column: its element, and the roles of its nodes as bit masks
// over the rows -- solved, counted in dot products (the first copy of a
// node).
struct Place { int e, el, j, slot0; bool act; unsigned msk, own; };

template <typename T, int NP, bool GREG>
__device__ inline ElemFac<T, NP, GREG> elem_fac(const ChipMesh& M, const ChipInst& I, const Place& P) {
  constexpr int NN = NP * NP;
  ElemFac<T, NP, GREG> F;
  const int set = M.nset == 1 ? 0 : M.eset[P.e];
  F.g = M.G + (size_t)set * G_N * NN;
  F.m = I.mq ? I.mq + (size_t)set * NN : F.g + G_Q4 * NN;
  F.hcon = (T)I.hcon;
  F.aff = M.aff != nullptr && I.mq == nullptr;
  F.f1 = F.f2 = F.f3 = F.f4 = 0;
  if (F.aff) {
    const double* c = M.aff + 4 * (size_t)set;
    const double wj = M.wq[P.j];
    F.f1 = (T)(c[0] * wj); F.f2 = (T)(c[1] * wj); F.f3 = (T)(c[2] * wj);
    F.f4 = (T)(c[3] * wj * I.hcon);
  }
  if constexpr (GREG) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int n = i * NP + P.j;
      for (int k = 0; k < 3; ++k) F.q[k][i] = (T)F.g[(G_Q1 + k) * NN + n];
      F.q[3][i] = (T)F.m[n] * F.hcon;
    }
  }
  const int o = I.svv ? 2 * NN : 0;
  if constexpr (sizeof(T) == 8) {
    F.w = ch_const(M.wq);
    F.D = ch_const(M.ops + o);
    F.DT = ch_const(M.ops + o + NN);
  } else {
    F.w = ch_const(M.wqf);
    F.D = ch_const(M.opsf + o);
    F.DT = ch_const(M.opsf + o + NN);
  }
  return F;
}

// a value the compiler takes as new, so that what is tested on it is not
// kept in scalar registers across the iteration
__device__ inline unsigned fresh(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

// The column's element-boundary entries into / out of their LDS slots: the
// first and last row of every column, the others of the first and last.  The
// slots of the last column ascend and those of the first descend; each has
// its own branch with constant offsets (a common one with a step of +-1 kept
// an address register per row, spilled and reloaded one after the other).
template <typename T, int NP>
__device__ inline void to_boundary(T* lb, const Place& P, const T (&q)[NP]) {
  constexpr int nm = NP - 1;
  T* s = lb + fresh((unsigned)P.slot0);
  s[P.j] = q[0];
  s[3 * nm - P.j] = q[nm];
  if (P.j == nm) {
#pragma unroll
    for (int i = 1; i < nm; ++i) s[nm + i] = q[i];
  } else if (P.j == 0) {
#pragma unroll
    for (int i = 1; i < nm; ++i) s[4 * nm - i] = q[i];
  }
}
template <typename T, int NP>
__device__ inline void from_boundary(const T* lb, const Place& P, T (&q)[NP]) {
  constexpr int nm = NP - 1;
  const T* s = lb + fresh((unsigned)P.slot0);
  q[0] = s[P.j];
  q[nm] = s[3 * nm - P.j];
  if (P.j == nm) {
#pragma unroll
    for (int i = 1; i < nm; ++i) q[i] = s[nm + i];
  } else if (P.j == 0) {
#pragma unroll
    for (int i = 1; i < nm; ++i) q[i] = s[4 * nm - i];
  }
}

// q = A p for the thread's column, summed over elements, rows not solved
// zero; returns p . q over the problem (each element's own part of it, which
// counts a shared node once).
template <typename T, int NP, class Fac>
__device__ inline double plane_apply(Wg& G, const Place& P, const Fac& F, const T (&p)[NP],
                                     T (&q)[NP], T* buf) {
  elem_apply<T, NP>(F, p, q, buf, P.j);
  double pq = 0.0;
  if (P.act) {
#pragma unroll
    for (int i = 0; i < NP; ++i) pq += (double)p[i] * (double)q[i];
    to_boundary<T, NP>((T*)G.lb, P, q);
  }
  pq = plane_assemble<T>(G, pq);
  from_boundary<T, NP>((const T*)G.lb2, P, q);
  const unsigned msk = fresh(P.msk);
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (!(msk >> i & 1)) q[i] = 0;
  return pq;
}

// PCG iterations on A d = r from d = x, semtex's loop (src/field.cpp:
// 665-712): pc holds the preconditioner's column in registers, or (null
// pcr) the thread reads its entries from element-ordered memory.
template <typename T, int NP, bool PCREG, class Fac>
__device__ inline int chip_core(Wg& G, const Place& P, const Fac& F, T (&x)[NP], T (&r)[NP],
                                const T (&pcr)[NP], const double* pcm, double epsb2, int step_max,
                                T* buf) {
  T p[NP], q[NP];
  double r2 = 0.0, rho1 = 0.0, rho2 = 1.0;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const T c = PCREG ? pcr[i] : (T)(P.act ? pcm[i * NP] : 0.0);
    const T z = c * r[i];
    p[i] = 0;
    q[i] = z;
    if (P.own >> i & 1) {
      r2 += (double)r[i] * (double)r[i];
      rho1 += (double)r[i] * (double)c * (double)r[i];
    }
  }
  {
    const double2 t = plane_sum2(G, r2, rho1);
    r2 = t.x;
    rho1 = t.y;
  }
  int it = 0;
  while (r2 > epsb2 && ++it < step_max) {
    const T beta = (it == 1) ? (T)0 : (T)(rho1 / rho2);
#pragma unroll
    for (int i = 0; i < NP; ++i) p[i] = q[i] + beta * p[i];
    const double pq = plane_apply<T, NP>(G, P, F, p, q, buf);
    const T alpha = (T)(rho1 / pq);
    double nr2 = 0.0, nrho = 0.0;
    const unsigned own = fresh(P.own);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const T c = PCREG ? pcr[i] : (T)(P.act ? pcm[i * NP] : 0.0);
      x[i] += alpha * p[i];
      r[i] -= alpha * q[i];
      q[i] = c * r[i];
      if (own >> i & 1) {
        nr2 += (double)r[i] * (double)r[i];
        nrho += (double)r[i] * (double)c * (double)r[i];
      }
    }
    rho2 = rho1;
    const double2 t = plane_sum2(G, nr2, nrho);
    r2 = t.x;
    rho1 = t.y;
  }
  return (it == step_max) ? -it : it;
}

template <bool REFINE, int NP>
__device__ __forceinline__ void chip_solve(const ChipArgs& a, const ChipInst& I, const ChipMesh& M, int fld,
                                  int pid, const ChipPart& pt, Wg& G, double* bufd) {
  constexpr int NN = NP * NP, NX = 4 * (NP - 1), NI = (NP - 2) * (NP - 2);
  constexpr int EPW = chip_epw(NP), LD = chip_ldr(NP);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  Place P;
  P.el = wave * EPW + lane / NP;
  P.j = lane - (lane / NP) * NP;
  P.act = lane < EPW * NP && P.el < pt.ne;
  if (!P.act) P.el = 0;
  P.e = pt.elo + P.el;
  P.slot0 = P.el * NX;
  P.msk = P.own = 0;
  if (P.act)
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int b = bpos<NP>(i, P.j);
      if (b < 0) {
        P.msk |= 1u << i;
        P.own |= 1u << i;
      } else {
        if (M.btog[P.e * NX + b] < I.n) {
          P.msk |= 1u << i;
          if (G.tab[P.slot0 + b].x == P.slot0 + b) P.own |= 1u << i;
        }
      }
    }
  // inactive lanes share one more tile, which nobody else reads
  const int ecap = (pt.ne + EPW - 1) / EPW * EPW;
  double* tile = bufd + (size_t)(P.act ? P.el : ecap) * NP * LD;
  // FP64 iterations, small np: general factors and the preconditioner fit in
  // the registers beside the vectors
  constexpr bool REGS = !REFINE && NP <= CHIP_NPREG;
  const auto F = elem_fac<double, NP, REGS>(M, I, P);
  double x[NP], r[NP], q[NP];
  const double* bc = a.bbc ? a.bbc[pid] : nullptr;
  // right-hand side of the element: -(M f + H g) + <h,w>
  if (a.bf) {
    const double* f = a.bf[pid];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      x[i] = 0.0;
      const int b = bpos<NP>(i, P.j);
      if (P.act && b >= 0) {
        const int gid = M.btog[P.e * NX + b];
        if (gid >= M.nsolve) x[i] = bc[M.ess_src[gid - M.nsolve]];
      }
    }
    elem_apply<double, NP>(F, x, q, tile, P.j);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      r[i] = 0.0;
      if (!P.act) continue;
      r[i] = -(F.g[G_Q4 * NN + i * NP + P.j] * f[(size_t)P.e * NN + i * NP + P.j]) - q[i];
      const int b = bpos<NP>(i, P.j);
      if (b >= 0)
        for (int cc = M.nat_ptr[P.e]; cc < M.nat_ptr[P.e + 1]; ++cc) {
          const int bs = M.nat_b[cc];
          const int ii = (b - M.bside[bs] * (NP - 1) + NX) % NX;
          if (ii <= NP - 1) r[i] += bc[bs * NP + ii] * M.barea[bs * NP + ii];
        }
    }
  } else {
    const double* fb = a.Fb + fld * a.FbF + ((size_t)I.pidx * M.nel + P.e) * NX;
    const double* fi = a.Fi + fld * a.FiF + ((size_t)I.pidx * M.nel + P.e) * NI;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int b = bpos<NP>(i, P.j);
      r[i] = !P.act ? 0.0 : b >= 0 ? fb[b] : fi[(i - 1) * (NP - 2) + P.j - 1];
    }
  }
  // assembled: b, its norm
  if (P.act) to_boundary<double, NP>(G.lb, P, r);
  plane_assemble<double>(G, 0.0);
  from_boundary<double, NP>(G.lb2, P, r);
  double bb = 0.0;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if (!(P.msk >> i & 1)) r[i] = 0.0;
    if (P.own >> i & 1) bb += r[i] * r[i];
  }
  const double epsb = a.tol * sqrt(plane_sum2(G, bb, 0.0).x);
  const double epsb2 = epsb * epsb;
  // x0: the current field; the copy written last wins where copies differ
  // (Field::local2global, src/field.cpp:928-947)
  double* uk = a.bu ? a.bu[pid] : a.u[fld] + (size_t)I.plane * a.planeSize;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    x[i] = 0.0;
    if (!(P.msk >> i & 1)) continue;
    const int b = bpos<NP>(i, P.j);
    if (b < 0) {
      x[i] = uk[(size_t)P.e * NN + i * NP + P.j];
    } else {
      const int4 g = M.gsrc[P.e * NX + b];
      const int s = g.w >= 0 ? g.w : g.z >= 0 ? g.z : g.y >= 0 ? g.y : g.x;
      const int e2 = s / NX;
      x[i] = uk[(size_t)e2 * NN + bnode<NP>(s - e2 * NX)];
    }
  }
  double* wk = I.work + fld * a.workF + (size_t)P.e * NN + P.j;   // this column, rows NP apart
  if constexpr (REFINE) {
    if (P.act)
#pragma unroll
      for (int i = 0; i < NP; ++i) wk[i * NP] = r[i];     // b, for the residuals
  }
  plane_apply<double, NP>(G, P, F, x, q, tile);
#pragma unroll
  for (int i = 0; i < NP; ++i) r[i] -= q[i];
  int its = 0;
  if constexpr (!REFINE) {
    if (P.act)
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int b = bpos<NP>(i, P.j);
        wk[i * NP] = !(P.msk >> i & 1) ? 0.0
                     : b >= 0 ? I.pc[M.btog[P.e * NX + b]]
                              : I.pc[M.nglobal + P.e * NI + (i - 1) * (NP - 2) + P.j - 1];
      }
    if constexpr (REGS) {
      double pc[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) pc[i] = P.act ? wk[i * NP] : 0.0;
      its = chip_core<double, NP, true>(G, P, F, x, r, pc, wk, epsb2, a.step_max, tile);
    } else {
      its = chip_core<double, NP, false>(G, P, F, x, r, q, wk, epsb2, a.step_max, tile);
    }
  } else {
    const auto Ff = elem_fac<float, NP, false>(M, I, P);
    float pc[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int b = bpos<NP>(i, P.j);
      pc[i] = !(P.msk >> i & 1) ? 0.0f
              : b >= 0 ? I.pc32[M.btog[P.e * NX + b]]
                       : I.pc32[M.nglobal + P.e * NI + (i - 1) * (NP - 2) + P.j - 1];
    }
    float* tilef = (float*)tile;
    for (int outer = 0;; ++outer) {
      double rn = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (P.own >> i & 1) rn += r[i] * r[i];
      rn = plane_sum2(G, rn, 0.0).x;
      if (rn <= epsb2) break;
      if (outer == a.max_outer) { its = -its; break; }
      float d[NP], rr[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) { d[i] = 0.0f; rr[i] = (float)r[i]; }
      const int it = chip_core<float, NP, true>(G, P, Ff, d, rr, pc, nullptr,
                                                a.inner_tol * a.inner_tol * rn, a.step_max, tilef);
      its += it < 0 ? -it : it;
#pragma unroll
      for (int i = 0; i < NP; ++i) x[i] += (double)d[i];
      plane_apply<double, NP>(G, P, F, x, q, tile);
#pragma unroll
      for (int i = 0; i < NP; ++i) r[i] = (P.act && (P.msk >> i & 1)) ? wk[i * NP] - q[i] : 0.0;
    }
  }
  // solution and essential values (Field::global2local + setEssential); the
  // initial guess is read by other workgroups' first copies of shared nodes:
  // every workgroup passed a sum after reading it
  const double* gp = a.bf ? nullptr : a.g + fld * a.gF + (size_t)I.pidx * a.nzero;
  if (P.act)
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int b = bpos<NP>(i, P.j);
      double v = x[i];
      if (b >= 0 && !(P.msk >> i & 1)) {
        const int gid = M.btog[P.e * NX + b];
        v = gid < M.nsolve ? 0.0 : a.bf ? bc[M.ess_src[gid - M.nsolve]] : gp[gid - M.nsolve];
      }
      uk[(size_t)P.e * NN + i * NP + P.j] = v;
    }
  if (threadIdx.x == 0 && G.w == 0) a.iters[(size_t)fld * a.count + pid] = its;
  if (G.dead) __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One workgroup takes the next (problem, part) of the order.  Workgroups of
// one problem are consecutive there and wait for each other; the ticket
// makes the order of taking the order of starting, so the problem taken
// first among the unfinished ones always has all its workgroups running,
// or the next free ones: the grid drains whatever the dispatch order.
// SNP: the np of every problem (planes of one system: the compiler then
// allocates the registers for that np alone), or 0 (a batch of any).
template <bool REFINE, int SNP>
__global__ __launch_bounds__(CT) void k_pcg_chip(ChipArgs a) {
  extern __shared__ double lds[];
  __shared__ int s_t;
  if (threadIdx.x == 0) s_t = (int)atomicAdd(a.ticket, 1u);
  __syncthreads();
  int2 job = a.order[__builtin_amdgcn_readfirstlane(s_t)];
  job.x = __builtin_amdgcn_readfirstlane(job.x);
  job.y = __builtin_amdgcn_readfirstlane(job.y);
  const int fld = job.x / a.count, pid = job.x - fld * a.count;
  const ChipInst& I = a.inst[pid];
  const ChipMesh& M = *I.mesh;
  const ChipPart pt = M.part[job.y];
  Wg G;
  G.W = M.W; G.w = job.y; G.ne = pt.ne; G.nslot = pt.ne * M.next;
  G.nrem = pt.nrem; G.npub = pt.npub;
  G.dead = a.no_wait;
  G.kA = G.kB = 0;
  G.nif = M.nif;
  G.exch = a.exch + fld * a.exchF + I.exch;
  G.red = a.red + fld * a.redF + I.red;
  G.err = a.err;
  const int np = M.np, ldr = chip_ldr(np), epw = chip_epw(np);
  const int ecap = (pt.ne + epw - 1) / epw * epw;
  G.rd = lds;
  double* buf = lds + CHIP_RED;
  G.lb = buf + (size_t)(ecap + 1) * np * ldr;
  G.lb2 = G.lb + G.nslot + G.nrem + 1;          // the zero behind
  ushort4* tab = reinterpret_cast<ushort4*>(G.lb2 + G.nslot + 1);
  G.tab = tab;
  int2* pub = reinterpret_cast<int2*>(tab + G.nslot + 1);
  int* rem = reinterpret_cast<int*>(pub + G.npub);
  G.pub = pub;
  G.rem = rem;
  for (int i = threadIdx.x; i < G.npub; i += CT) pub[i] = M.pub[pt.pub0 + i];
  for (int i = threadIdx.x; i < G.nrem; i += CT) rem[i] = M.rem[pt.rem0 + i];
  const unsigned short zero = (unsigned short)(G.nslot + G.nrem);
  for (int i = threadIdx.x; i <= G.nslot; i += CT) {
    ushort4 q = ushort4{zero, zero, zero, zero};
    if (i < G.nslot) q = M.tab[(size_t)pt.elo * M.next + i];
    tab[i] = ushort4{q.x, q.y == 0xFFFF ? zero : q.y, q.z == 0xFFFF ? zero : q.z,
                     q.w == 0xFFFF ? zero : q.w};
  }
  __syncthreads();
  if constexpr (SNP > 0) {
    chip_solve<REFINE, SNP>(a, I, M, fld, pid, pt, G, buf);
    return;
  } else switch (np) {
#define CHIP_CASE(N) case N: chip_solve<REFINE, N>(a, I, M, fld, pid, pt, G, buf); break;
    CHIP_CASE(4) CHIP_CASE(5) CHIP_CASE(6) CHIP_CASE(7) CHIP_CASE(8) CHIP_CASE(9)
    CHIP_CASE(10) CHIP_CASE(11) CHIP_CASE(12)
#undef CHIP_CASE
    default: break;
  }
}

// exchange and partial-sum slots to the sentinel, the ticket to zero
__global__ void k_chip_reset(double* ex, long long nex, double* red, long long nred,
                             unsigned* ticket) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const double z = __longlong_as_double((long long)CHIP_SENT);
  if (i < nex) ex[i] = z;
  if (i < nred) red[i] = z;
  if (i == 0) *ticket = 0;
}

int elems_per_wg(int np) { return CWV * chip_epw(np); }

}  // namespace

int chip_workgroups(const Mesh& M) {
  if (M.np < CHIP_NPMIN || M.np > CHIP_NPMAX) return 0;
  for (int g = 0; g < M.nglobal; ++g)
    if (M.asm_ptr[g + 1] - M.asm_ptr[g] > 4) return 0;
  const int W = (M.nel + elems_per_wg(M.np) - 1) / elems_per_wg(M.np);
  // a problem's workgroups wait for each other, each on a CU of its own: all of
  // them have to be resident (fewer than 256 CUs on a partitioned device)
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return W <= std::min(CHIP_WMAX, cus) ? W : 0;
}

int chip_plan(Mesh& M, ChipPlan& P, const ChipMesh** dev) {
  P = ChipPlan();
  *dev = nullptr;
  const int W = chip_workgroups(M);
  if (!W) return SEMX_OK;
  const int next = M.next, nel = M.nel, npnp = M.npnp;
  std::vector<ChipPart> part(W);
  std::vector<int> owner(nel);
  for (int w = 0; w < W; ++w) {
    part[w].elo = (int)((long long)nel * w / W);
    part[w].ne = (int)((long long)nel * (w + 1) / W) - part[w].elo;
    for (int e = part[w].elo; e < part[w].elo + part[w].ne; ++e) owner[e] = w;
  }
  // exchange position of every slot that another workgroup adds
  std::vector<int> pos((size_t)nel * next, -1), rem;
  std::vector<int4> gsrc((size_t)nel * next);
  int nif = 0;
  for (int g = 0; g < M.nglobal; ++g) {
    const int c0 = M.asm_ptr[g], c1 = M.asm_ptr[g + 1];
    bool shared = false;
    for (int c = c0; c < c1; ++c) shared |= owner[M.asm_idx[c] / next] != owner[M.asm_idx[c0] / next];
    int s4[4] = {-1, -1, -1, -1};
    for (int c = c0; c < c1; ++c) {
      s4[c - c0] = M.asm_idx[c];
      if (shared) pos[M.asm_idx[c]] = 0;
    }
    for (int c = c0; c < c1; ++c) gsrc[M.asm_idx[c]] = make_int4(s4[0], s4[1], s4[2], s4[3]);
  }
  // in slot order: what a workgroup sends lies together (whole cache lines)
  for (int& q : pos)
    if (q == 0) q = nif++;
  std::vector<ushort4> tab((size_t)nel * next);
  std::vector<int2> pub;
  size_t lds = 0;
  const int epw = chip_epw(M.np), ldr = chip_ldr(M.np);
  for (int w = 0; w < W; ++w) {
    ChipPart& p = part[w];
    const int s0 = p.elo * next, ns = p.ne * next;
    p.rem0 = (int)rem.size();
    p.pub0 = (int)pub.size();
    std::vector<int> at((size_t)nel * next, -1);
    for (int s = s0; s < s0 + ns; ++s) {
      if (pos[s] >= 0) pub.push_back(make_int2(s - s0, pos[s]));
      const int4 g = gsrc[s];
      const int src[4] = {g.x, g.y, g.z, g.w};
      unsigned short q[4];
      for (int k = 0; k < 4; ++k) {
        q[k] = 0xFFFF;
        const int t = src[k];
        if (t < 0) continue;
        int idx = t - s0;
        if (idx < 0 || idx >= ns) {
          if (at[t] < 0) { at[t] = ns + (int)rem.size() - p.rem0; rem.push_back(pos[t]); }
          idx = at[t];
        }
        if (idx >= 0xFFFF) return SEMX_OK;
        q[k] = (unsigned short)idx;
      }
      tab[s] = ushort4{q[0], q[1], q[2], q[3]};
    }
    p.nrem = (int)rem.size() - p.rem0;
    p.npub = (int)pub.size() - p.pub0;
    const size_t ecap = (size_t)(p.ne + epw - 1) / epw * epw;
    lds = std::max(lds, (CHIP_RED + (ecap + 1) * M.np * ldr + (size_t)(ns + 1) * 3 + p.nrem + p.npub +
                         (p.nrem + 1) / 2) * sizeof(double));
  }
  if (lds > 160 * 1024 - 1024) return SEMX_OK;
  // parallelograms: factors proportional to the products of the weights, to the
  // last places of the stored ones.  Rectangles, sheared and rotated meshes
  // deviate by at most 4.4e-16 (np 4 to 12); against long double the stored
  // factors are off by up to 3.1e-16 and constant x weight x weight by 3.1e-16.
  // In FP32 the latter rounds twice where the stored factor rounds once; only
  // the refined solves' inner iterations do.
  std::vector<double> aff;
  bool isaff = !M.cyl;
  const int np = M.np;
  const std::vector<double>& w = M.ops.w;
  for (int s = 0; s < M.nset && isaff; ++s) {
    const double* g = &M.G[(size_t)s * G_N * npnp];
    double c[4], big = 0.0;
    const int mid = (np / 2) * np + np / 2;
    const double wm = w[np / 2] * w[np / 2];
    for (int k = 0; k < 4; ++k) { c[k] = g[(G_Q1 + k) * npnp + mid] / wm; }
    for (int k = 0; k < 4; ++k) {
      big = k == 3 ? std::fabs(c[3]) : std::max(std::fabs(c[0]), std::fabs(c[1]));
      for (int i = 0; i < np; ++i)
        for (int j = 0; j < np; ++j)
          isaff &= std::fabs(g[(G_Q1 + k) * npnp + i * np + j] - c[k] * w[i] * w[j]) <=
                   1e-15 * big * w[i] * w[j];
    }
    for (int k = 0; k < 4; ++k) aff.push_back(c[k]);
  }
  if (!isaff) aff.clear();
  std::vector<float> opsf;
  for (const auto* v : {&M.ops.DV, &M.ops.DT, &M.ops.SDV, &M.ops.SDT})
    opsf.insert(opsf.end(), v->begin(), v->end());
  std::vector<float> wf(w.begin(), w.end());
  // one allocation: descriptor, then the arrays, each on 256 bytes
  std::vector<char> blob(256 * ((sizeof(ChipMesh) + 255) / 256));
  auto put = [&](const void* src, size_t bytes) {
    const size_t off = blob.size();
    blob.resize(off + (bytes + 255) / 256 * 256);
    if (bytes) memcpy(&blob[off], src, bytes);
    return off;
  };
  const size_t o_part = put(part.data(), part.size() * sizeof(ChipPart));
  const size_t o_tab = put(tab.data(), tab.size() * sizeof(ushort4));
  const size_t o_src = put(gsrc.data(), gsrc.size() * sizeof(int4));
  const size_t o_rem = put(rem.data(), rem.size() * sizeof(int));
  const size_t o_pub = put(pub.data(), pub.size() * sizeof(int2));
  const size_t o_aff = put(aff.data(), aff.size() * sizeof(double));
  const size_t o_wq = put(w.data(), w.size() * sizeof(double));
  const size_t o_wf = put(wf.data(), wf.size() * sizeof(float));
  const size_t o_of = put(opsf.data(), opsf.size() * sizeof(float));
  char* d = nullptr;
  if (int st = dev_upload<char>(&d, nullptr, blob.size())) return st;
  P.store = d;
  ChipMesh& m = P.m;
  m.np = np; m.npnp = npnp; m.next = next; m.nint = M.nint; m.nel = nel; m.nglobal = M.nglobal;
  m.nsolve = M.nsolve; m.nset = M.nset; m.W = W; m.nif = nif;
  m.part = (const ChipPart*)(d + o_part);
  m.tab = (const ushort4*)(d + o_tab);
  m.gsrc = (const int4*)(d + o_src);
  m.rem = (const int*)(d + o_rem);
  m.pub = (const int2*)(d + o_pub);
  m.G = M.d.G; m.eset = M.d.eset; m.btog = M.d.btog;
  m.aff = aff.empty() ? nullptr : (const double*)(d + o_aff);
  m.wq = (const double*)(d + o_wq);
  m.wqf = (const float*)(d + o_wf);
  m.ops = M.d.ops;
  m.opsf = (const float*)(d + o_of);
  m.ess_src = M.d.ess_src; m.nat_ptr = M.d.nat_ptr; m.nat_b = M.d.nat_b;
  m.bside = M.d.bside; m.barea = M.d.barea;
  memcpy(&blob[0], &m, sizeof m);
  HIPCHK(hipMemcpy(d, blob.data(), blob.size(), hipMemcpyHostToDevice));
  P.W = W; P.nif = nif; P.lds64 = lds; P.ok = true;
  *dev = (const ChipMesh*)d;
  return SEMX_OK;
}

void chip_release(ChipPlan& P) {
  if (P.store) (void)hipFree(P.store);
  P = ChipPlan();
}

int chip_launch(const ChipArgs& a, int np, bool refine, int groups, size_t lds, long long nexch,
                long long nred, hipStream_t s) {
  const void* fn = nullptr;
  switch (np) {
#define CHIP_FN(N)                                                                      \
  case N:                                                                               \
    fn = refine ? (const void*)k_pcg_chip<true, N> : (const void*)k_pcg_chip<false, N>; \
    break;
    CHIP_FN(0) CHIP_FN(4) CHIP_FN(5) CHIP_FN(6) CHIP_FN(7) CHIP_FN(8) CHIP_FN(9) CHIP_FN(10)
    CHIP_FN(11) CHIP_FN(12)
#undef CHIP_FN
    default: return SEMX_E_UNSUPPORTED;
  }
  HIPCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const long long n = std::max(std::max(nexch, nred), 1LL);
  hipLaunchKernelGGL(k_chip_reset, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a.exch,
                     nexch, a.red, nred, a.ticket);
  // SEMX_PCG_NOWAIT=1, for tests of an expired wait: no value is waited for
  // (a limit on the polls as an argument of the kernel cost the batch 3%)
  ChipArgs b = a;
  b.no_wait = getenv("SEMX_PCG_NOWAIT") && atoi(getenv("SEMX_PCG_NOWAIT")) != 0;
  hipEvent_t ev;
  prof_begin(s, &ev);
  void* kargs[] = {&b};
  HIPCHK(hipLaunchKernel(fn, dim3((unsigned)groups), dim3(CT), kargs, lds, s));
  prof_end(s, a.bf ? "k_pcg_batch" : "k_pcg", ev);
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

}  // namespace semx
