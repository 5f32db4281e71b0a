// semx_dns.hip -- field operators and the 3D3C Navier-Stokes time step of
// semtex's dns solver on CDNA4 (gfx950):
//
//   k_fft        dDFTr along z, femlib/fourier.c:47-171: every column of a
//                field (ntrn columns, z-stride ntrn), semtex's packing
//                [Re0, Re_N/2, Re1, Im1, ...] and 1/N forward scaling
//   k_dft_z      the same as one dense real N x N product (odd lengths and
//                the allocation-free entry point)
//   k_grad_xy    AuxField::gradient x/y, src/auxfield.cpp:514-665 with
//                Element::grad, src/element.cpp:552-597
//   k_grad_z     AuxField::gradient z in Fourier space, auxfield.cpp:636-657
//   k_smooth     Field::smooth, src/field.cpp:190-236 (mass-weighted DSS)
//   k_nl         the nonlinear terms of all components
//   k_wave_div   waveProp and setPForce
//   k_project    project
//
//   k_hopbc      BCmgr::maintainFourier and evaluateCNBCp (src/bcmgr.cpp:
//                1039-1337): the computed high-order pressure flux on the
//                boundary sides of a bounded mesh
//
// and the host driver of integrate (dns/integrate.cpp:79-221) with
// waveProp, setPForce, project and the velocity/pressure solves of
// Field::solve (semx_solve.hip), on a periodic mesh or on a bounded one
// (velocity BC lines given, pressure flux computed).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

#include "semx_hip.h"

using namespace semx;

namespace {

constexpr int DFT_KB = 16;          // padding of the transform matrix columns

// The same product on the FP64 matrix cores (v_mfma_f64_16x16x4: A 16x4,
// B 4x16, D 16x16; lane l holds A[l%16][l/16], B[l/16][l%16] and, in
// register r, D[4r + l/16][l%16]).  W (MT 16-row tiles by K padded to 4) is
// staged in LDS with an odd row stride, so the 16 rows an A operand reads
// fall in distinct banks; each wave owns DFT_MCT 16-column tiles of the
// block's columns and all MT row tiles, and takes its B operands (four input
// rows by 16 columns per k step) straight from memory, DFT_MPF steps ahead
// in a register ring.  Input rows at or beyond N are clamped (their W
// columns are zero), as are columns beyond ntrn (not stored).  For N <= 128.
constexpr int DFT_MCT = 2;                       // column tiles per wave
constexpr int DFT_MPF = 4;                       // k steps of B prefetch
constexpr int DFT_MCOLS = 4 * 16 * DFT_MCT;      // columns per block
typedef double dft_d4 __attribute__((ext_vector_type(4)));

template <int MT>
__global__ __launch_bounds__(256) void k_dft_mfma(const double* __restrict__ in,
                                                  double* __restrict__ out,
                                                  const double* __restrict__ W, int N, int ldw,
                                                  int ntrn, long long ld) {
  extern __shared__ double sWm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int KP = (N + 3) & ~3;
  const int ldk = KP + 1;
  const int li = lane & 15, lk = lane >> 4;
  int col[DFT_MCT];
#pragma unroll
  for (int ct = 0; ct < DFT_MCT; ++ct)
    col[ct] = min(blockIdx.x * DFT_MCOLS + (wave * DFT_MCT + ct) * 16 + li, ntrn - 1);
  // B operands DFT_MPF k steps ahead in a register ring (rows clamped)
  const int KS = KP / 4;
  auto load_b = [&](int ks, double (&b)[DFT_MCT]) {
    const size_t row = (size_t)min(4 * ks + lk, N - 1) * ld;
#pragma unroll
    for (int ct = 0; ct < DFT_MCT; ++ct) b[ct] = in[row + col[ct]];
  };
  double bq[DFT_MPF][DFT_MCT];
#pragma unroll
  for (int u = 0; u < DFT_MPF; ++u) load_b(u, bq[u]);
  for (int r = tid >> 6; r < MT * 16; r += 4)
    for (int k = lane; k < KP; k += 64) sWm[r * ldk + k] = W[(size_t)r * ldw + k];
  __syncthreads();
  dft_d4 acc[MT][DFT_MCT];
#pragma unroll
  for (int rt = 0; rt < MT; ++rt)
#pragma unroll
    for (int ct = 0; ct < DFT_MCT; ++ct) acc[rt][ct] = dft_d4{0.0, 0.0, 0.0, 0.0};
  const double* wa = sWm + li * ldk + lk;
  for (int k0 = 0; k0 < KS; k0 += DFT_MPF) {
#pragma unroll
    for (int u = 0; u < DFT_MPF; ++u) {
      const int ks = k0 + u;
      if (ks < KS) {
#pragma unroll
        for (int rt = 0; rt < MT; ++rt) {
          const double a = wa[rt * 16 * ldk + 4 * ks];
#pragma unroll
          for (int ct = 0; ct < DFT_MCT; ++ct)
            acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bq[u][ct], acc[rt][ct], 0, 0, 0);
        }
      }
      load_b(ks + DFT_MPF, bq[u]);
    }
  }
#pragma unroll
  for (int ct = 0; ct < DFT_MCT; ++ct) {
    const int c = blockIdx.x * DFT_MCOLS + (wave * DFT_MCT + ct) * 16 + li;
    if (c >= ntrn) continue;
#pragma unroll
    for (int rt = 0; rt < MT; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rt * 16 + 4 * r + lk;
        if (row < N) out[(size_t)row * ld + c] = acc[rt][ct][r];
      }
  }
}

// out[r][col] = sum_k W[r][k] in[k][col], r < N: a register-blocked
// product of the (padded) N x N transform matrix with a 64-column tile of
// the field.  Threads form 16 row groups x 16 column groups; each computes
// RP rows x 4 columns, with the k dimension staged through LDS 16 rows at a
// time.  W has rows padded to 16*RP and columns to a multiple of 16 (zero
// entries), so loads of rows >= N are clamped without a branch.
constexpr int DFT_COLS = 64;
constexpr int DFT_KC = 16;

template <int RP>
__global__ __launch_bounds__(256) void k_dft_z(const double* __restrict__ in,
                                               double* __restrict__ out,
                                               const double* __restrict__ W, int N, int ldw,
                                               int ncol, long long stride) {
  __shared__ double sX[DFT_KC][DFT_COLS];
  __shared__ double sW[16 * RP][DFT_KC + 1];
  const int tid = threadIdx.x;
  const int cg = tid & 15, rg = tid >> 4;
  const int col0 = blockIdx.x * DFT_COLS;
  double acc[RP][4];
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0;
  for (int k0 = 0; k0 < N; k0 += DFT_KC) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < DFT_KC * DFT_COLS / 256; ++q) {
      const int idx = tid + q * 256;
      const int kk = idx / DFT_COLS, c = idx - (idx / DFT_COLS) * DFT_COLS;
      sX[kk][c] = in[(size_t)min(k0 + kk, N - 1) * stride + min(col0 + c, ncol - 1)];
    }
#pragma unroll
    for (int q = 0; q < RP; ++q) {
      const int idx = tid + q * 256;            // 16*RP rows x 16 k
      const int r = idx / DFT_KC, kk = idx - (idx / DFT_KC) * DFT_KC;
      sW[r][kk] = W[(size_t)r * ldw + k0 + kk];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < DFT_KC; ++kk) {
      double xv[4], wv[RP];
#pragma unroll
      for (int j = 0; j < 4; ++j) xv[j] = sX[kk][cg * 4 + j];
#pragma unroll
      for (int i = 0; i < RP; ++i) wv[i] = sW[rg * RP + i][kk];
#pragma unroll
      for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += wv[i] * xv[j];
    }
  }
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    const int r = rg * RP + i;
    if (r >= N) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = col0 + cg * 4 + j;
      if (c < ncol) out[(size_t)r * stride + c] = acc[i][j];
    }
  }
}

// Transforms of even length N <= 256 = 2 M along z: the real sequence of a
// column taken as M complex values, a Stockham FFT of radix 5, 4, 3 and 2
// passes over them, and the split into (or, inverse, the join from) the
// spectrum of length N.  A workgroup holds CT columns in LDS, twice (a pass
// reads one copy and writes the other), [row][column], so that every access
// of a wavefront is to whole rows of columns; it reads all rows of its
// columns before it writes any, so input and output may be one buffer.
//
// What bounds it: memory, one read and one write of the field.  The dense
// product on the matrix cores that took even lengths before did 2 N^2
// operations a column (11 us at the FP64 peak on 96 x 46656 values, 40 us
// measured with its operands' latencies); it stays for odd lengths.
// Measured, N = 96: 38880 columns 39 us and 10 us for the copy back -> 19 us
// (3.1 TB/s); three components of 46656, the transforms with their
// derivatives: 85 us inverse (3.8 TB/s), 87 us forward, for 24 and 24 us of
// z derivatives, 240 us and 160 us of products and 64 us of elementwise passes.
//
// Kinds, with c the column's component (blockIdx.y):
//   FORWARD     out = F(in), semtex's packing, 1/N
//   INVERSE     out = F^-1(in)
//   INVERSE_DZ  out = F^-1(in), out2 = F^-1(d(in)/dz): a convective term's
//               two operands from one read of the spectrum
//   FORWARD_DZ  out = sc (F(in) - d/dz F(b1 b2)): the transform of a
//               nonlinear term with its conservative z part formed there
enum { FFT_FORWARD, FFT_INVERSE, FFT_INVERSE_DZ, FFT_FORWARD_DZ };

struct FftArgs {
  const double* in[3];
  double* out[3];
  double* out2[3];
  const double* b1[3];
  const double* b2;
  const double2* tw;      // cos, sin of 2 pi j / N, j < N
  int N, ntrn, nrad;
  int rad[8];
  double beta, sc;
};

template <int R, bool INV>
__device__ __forceinline__ void fft_butterfly(double (&x)[R], double (&y)[R]) {
  constexpr double sg = INV ? 1.0 : -1.0;
  if constexpr (R == 2) {
    const double a = x[1], b = y[1];
    x[1] = x[0] - a; y[1] = y[0] - b;
    x[0] += a; y[0] += b;
  } else if constexpr (R == 3) {
    constexpr double s3 = 0.86602540378443864676;
    const double ax = x[1] + x[2], ay = y[1] + y[2];
    const double bx = sg * s3 * (x[1] - x[2]), by = sg * s3 * (y[1] - y[2]);
    const double mx = x[0] - 0.5 * ax, my = y[0] - 0.5 * ay;
    x[0] += ax; y[0] += ay;
    x[1] = mx - by; y[1] = my + bx;
    x[2] = mx + by; y[2] = my - bx;
  } else if constexpr (R == 4) {
    const double ax = x[0] + x[2], ay = y[0] + y[2], bx = x[0] - x[2], by = y[0] - y[2];
    const double cx = x[1] + x[3], cy = y[1] + y[3];
    const double dx = sg * (x[1] - x[3]), dy = sg * (y[1] - y[3]);
    x[0] = ax + cx; y[0] = ay + cy;
    x[2] = ax - cx; y[2] = ay - cy;
    x[1] = bx - dy; y[1] = by + dx;
    x[3] = bx + dy; y[3] = by - dx;
  } else {
    constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    const double ax = x[1] + x[4], ay = y[1] + y[4], bx = x[2] + x[3], by = y[2] + y[3];
    const double cx = sg * (x[1] - x[4]), cy = sg * (y[1] - y[4]);
    const double dx = sg * (x[2] - x[3]), dy = sg * (y[2] - y[3]);
    const double px = x[0] + c1 * ax + c2 * bx, py = y[0] + c1 * ay + c2 * by;
    const double qx = x[0] + c2 * ax + c1 * bx, qy = y[0] + c2 * ay + c1 * by;
    const double ux = s1 * cx + s2 * dx, uy = s1 * cy + s2 * dy;
    const double vx = s2 * cx - s1 * dx, vy = s2 * cy - s1 * dy;
    x[0] += ax + bx; y[0] += ay + by;
    x[1] = px - uy; y[1] = py + ux;
    x[4] = px + uy; y[4] = py - ux;
    x[2] = qx - vy; y[2] = qy + vx;
    x[3] = qx + vy; y[3] = qy - vx;
  }
}

// One pass of radix R over S sets of M complex values (rows 2 j, 2 j + 1):
// l values of each transform are done.
template <int R, bool INV, int S, int CT>
__device__ __forceinline__ void fft_pass(const double* src, double* dst, const double2* tw, int N,
                                         int l) {
  constexpr int NG = 256 / CT;
  const int col = threadIdx.x % CT, M = N / 2, nb = M / R, step = N / (l * R);
  const float il = 1.0f / (float)l;
  for (int it = threadIdx.x / CT; it < S * nb; it += NG) {
    const int s = S > 1 && it >= nb ? 1 : 0, b = it - s * nb;
    const int k = b - (int)(((float)b + 0.5f) * il) * l;
    const double* in = src + (size_t)s * N * CT + col;
    double* out = dst + (size_t)s * N * CT + col;
    double x[R], y[R];
#pragma unroll
    for (int t = 0; t < R; ++t) {
      x[t] = in[2 * (b + t * nb) * CT];
      y[t] = in[(2 * (b + t * nb) + 1) * CT];
    }
#pragma unroll
    for (int t = 1; t < R; ++t) {
      const double2 w = tw[t * k * step];
      const double wi = INV ? w.y : -w.y, a = x[t];
      x[t] = a * w.x - y[t] * wi;
      y[t] = a * wi + y[t] * w.x;
    }
    fft_butterfly<R, INV>(x, y);
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const int r = (b - k) * R + k + t * l;
      out[2 * r * CT] = x[t];
      out[(2 * r + 1) * CT] = y[t];
    }
  }
}

template <int KIND, int CT>
__global__ __launch_bounds__(256) void k_fft(FftArgs a) {
  constexpr bool INV = KIND == FFT_INVERSE || KIND == FFT_INVERSE_DZ;
  constexpr int S = KIND == FFT_INVERSE_DZ || KIND == FFT_FORWARD_DZ ? 2 : 1;
  constexpr int NG = 256 / CT, U = 4;
  extern __shared__ double fft_lds[];
  const int tid = threadIdx.x, col = tid % CT, g = tid / CT, N = a.N, M = N / 2, c = blockIdx.y;
  double2* tw = reinterpret_cast<double2*>(fft_lds);
  double* src = fft_lds + 2 * N;
  double* dst = src + (size_t)S * N * CT;
  const size_t ld = a.ntrn;
  const int gc = blockIdx.x * CT + col;
  const bool on = gc < a.ntrn;
  const size_t cc = on ? gc : a.ntrn - 1;       // columns past the last are not stored
  for (int i = tid; i < N; i += 256) tw[i] = a.tw[i];
  const double* in = a.in[c] + cc;
  if (!INV) {
    for (int n0 = g; n0 < N; n0 += U * NG) {
      double v[U], w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const size_t r = (size_t)min(n0 + u * NG, N - 1) * ld;
        v[u] = in[r];
        if (S > 1) w[u] = a.b1[c][cc + r] * a.b2[cc + r];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (n0 + u * NG < N) {
          src[(n0 + u * NG) * CT + col] = v[u];
          if (S > 1) src[(size_t)(N + n0 + u * NG) * CT + col] = w[u];
        }
    }
    __syncthreads();
  } else {
    __syncthreads();
    for (int k0 = g; k0 <= M / 2; k0 += 2 * NG) {
      double v[2][4];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k = min(k0 + u * NG, M / 2), q = k ? M - k : 0;
        v[u][0] = in[(size_t)(2 * k) * ld];
        v[u][1] = in[(size_t)(2 * k + 1) * ld];
        v[u][2] = in[(size_t)(2 * q) * ld];
        v[u][3] = in[(size_t)(2 * q + 1) * ld];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k = k0 + u * NG, q = M - k;
        if (k > M / 2) continue;
        if (k == 0) {
          src[col] = v[u][0] + v[u][1];
          src[CT + col] = v[u][0] - v[u][1];
          if (S > 1) src[(size_t)N * CT + col] = src[(size_t)(N + 1) * CT + col] = 0.0;
          continue;
        }
        const double2 w = tw[k];
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const double bk = s ? a.beta * k : 1.0, bq = s ? a.beta * q : 1.0;
          const double xr = s ? -bk * v[u][1] : v[u][0], xi = s ? bk * v[u][0] : v[u][1];
          const double yr = s ? -bq * v[u][3] : v[u][2], yi = s ? bq * v[u][2] : v[u][3];
          const double pr = xr + yr, pi = xi - yi, dr = xr - yr, di = xi + yi;
          const double e = w.x * di + w.y * dr, f = w.x * dr - w.y * di;
          double* z = src + (size_t)s * N * CT + col;
          z[2 * k * CT] = pr - e;
          z[(2 * k + 1) * CT] = pi + f;
          if (q != k) {
            z[2 * q * CT] = pr + e;
            z[(2 * q + 1) * CT] = f - pi;
          }
        }
      }
    }
    __syncthreads();
  }
  for (int i = 0, l = 1; i < a.nrad; ++i) {
    const int r = a.rad[i];
    if (r == 4) fft_pass<4, INV, S, CT>(src, dst, tw, N, l);
    else if (r == 3) fft_pass<3, INV, S, CT>(src, dst, tw, N, l);
    else if (r == 5) fft_pass<5, INV, S, CT>(src, dst, tw, N, l);
    else fft_pass<2, INV, S, CT>(src, dst, tw, N, l);
    __syncthreads();
    double* t = src; src = dst; dst = t;
    l *= r;
  }
  if (!on) return;
  double* out = a.out[c] + cc;
  if (INV) {
    for (int n = g; n < N; n += NG) {
      out[(size_t)n * ld] = src[n * CT + col];
      if (S > 1) a.out2[c][cc + (size_t)n * ld] = src[(size_t)(N + n) * CT + col];
    }
    return;
  }
  const double sc = (KIND == FFT_FORWARD_DZ ? a.sc : 1.0) / N;
  for (int k = g; k <= M / 2; k += NG) {
    const double* z = src + col;
    if (k == 0) {
      out[0] = sc * (z[0] + z[CT]);
      out[ld] = sc * (z[0] - z[CT]);
      continue;
    }
    const int q = M - k;
    const double2 w = tw[k];
    double x[S][4];             // X_k, X_{M-k}
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const double* zs = z + (size_t)s * N * CT;
      const double zr = zs[2 * k * CT], zi = zs[(2 * k + 1) * CT];
      const double yr = zs[2 * q * CT], yi = zs[(2 * q + 1) * CT];
      const double er = 0.5 * (zr + yr), ei = 0.5 * (zi - yi);
      const double pr = 0.5 * (zi + yi), pi = 0.5 * (yr - zr);
      const double tr = w.x * pr + w.y * pi, ti = w.x * pi - w.y * pr;
      x[s][0] = er + tr; x[s][1] = ei + ti;
      x[s][2] = er - tr; x[s][3] = ti - ei;
    }
    if (S > 1) {                // - i beta k
      const double bk = a.beta * k, bq = a.beta * q;
      x[0][0] += bk * x[S - 1][1]; x[0][1] -= bk * x[S - 1][0];
      x[0][2] += bq * x[S - 1][3]; x[0][3] -= bq * x[S - 1][2];
    }
    out[(size_t)(2 * k) * ld] = sc * x[0][0];
    out[(size_t)(2 * k + 1) * ld] = sc * x[0][1];
    if (q != k) {
      out[(size_t)(2 * q) * ld] = sc * x[0][2];
      out[(size_t)(2 * q + 1) * ld] = sc * x[0][3];
    }
  }
}

// d/dx (dir 0) or d/dy (dir 1) on every element, PB planes per workgroup:
// tgt = (D_s u) * ds/dx_i + (u D_r^T) * dr/dx_i, plain (non-SVV) D.  The
// planes share the element's factors and put PB loads per thread in flight.
// Measured, 24x20 quads np=9, 96 planes: 27 -> 20 us (3.0 TB/s).
template <int PB>
__global__ __launch_bounds__(256) void k_grad_xy(double* __restrict__ data,
                                                 const double* __restrict__ G,
                                                 const int* __restrict__ eset,
                                                 const double* __restrict__ ops, int np,
                                                 int nel, int planeSize, int nz, int dir) {
  extern __shared__ double gsh[];
  const int npnp = np * np, ce = 256 / npnp, t = threadIdx.x;
  const int el = t / npnp, pt = t - el * npnp;
  const int e = blockIdx.x * ce + el;
  const bool act = el < ce && e < nel;
  double* sD = gsh;
  double* sT = sD + npnp;
  double* sU = sT + npnp;                 // PB x ce * npnp
  if (t < npnp) {
    sD[t] = ops[t];
    sT[t] = ops[npnp + t];
  }
  const int k0 = blockIdx.y * PB;
  double* u = data + (size_t)k0 * planeSize + (size_t)e * npnp + pt;
  if (act) {
    double v[PB];
#pragma unroll
    for (int p = 0; p < PB; ++p) v[p] = u[(size_t)min(p, nz - 1 - k0) * planeSize];
#pragma unroll
    for (int p = 0; p < PB; ++p) sU[p * ce * npnp + t] = v[p];
  }
  __syncthreads();
  if (!act) return;
  const int i = pt / np, j = pt - i * np;
  const double* su = sU + el * npnp;
  double A[PB], B[PB];
#pragma unroll
  for (int p = 0; p < PB; ++p) A[p] = B[p] = 0.0;
  for (int q = 0; q < np; ++q) {
    const double dt = sT[q * np + j], ds = sD[i * np + q];
#pragma unroll
    for (int p = 0; p < PB; ++p) {
      A[p] += su[p * ce * npnp + i * np + q] * dt;
      B[p] += ds * su[p * ce * npnp + q * np + j];
    }
  }
  const double* g = G + (size_t)eset[e] * G_N * npnp;
  const double rx = g[(dir ? G_DRDY : G_DRDX) * npnp + pt];
  const double sx = g[(dir ? G_DSDY : G_DSDX) * npnp + pt];
#pragma unroll
  for (int p = 0; p < PB; ++p)
    if (k0 + p < nz) u[(size_t)p * planeSize] = fma(B[p], sx, A[p] * rx);   // one order for every PB
}

// Computed pressure boundary conditions (KIO91; BCmgr::maintainFourier,
// src/bcmgr.cpp:1039-1298, and evaluateCNBCp, :1301-1337), Cartesian.  One
// workgroup per (boundary side, Fourier mode); at each node of the side and
// each plane of the mode (the Nyquist plane is left alone):
//   un   = u.n
//   hop  = -(1/dt) (a0 un + sum_{l<Jd} a_{l+1} un_l)      (Jd > 0 only)
//          + n.N(u) - nu n.curlCurl(u)
//   un_l, hop_l shift down one level (level 0 the new value)
//   bcp  = sum_{l<Je} b_l hop_l on the pressure's natural sides, else 0
// with u the Fourier velocity at the start of the step and N(u) its
// nonlinear terms.  curlCurl (Edge::curlCurl, src/edge.cpp:98-258) takes
// the z vorticity w = dv/dx - du/dy on the whole element and its gradient
// at the side: (dw/dy, -dw/dx), plus for mode k > 0 (beta k) the
// semi-Fourier terms of w-velocity and (beta k)^2 (u, v).  Each thread owns
// one (plane, side node) entry of every level array, so the in-place level
// shift has no hazards, and the level arrays never move (one HIP graph of
// the step stays valid).
struct HopArgs {
  const double* U[3];     // Fourier velocity, nz*planeSize each (W unused in 2D)
  const double* N[2];     // Fourier nonlinear terms, x and y
  double* un;             // nord levels of u.n, nz*nline each
  double* hop;            // nord levels of the flux terms
  double* bcp;            // pressure BC lines, nz*nline
  const int* bel;         // nbound: element
  const int* bsd;         // nbound: side 0-3
  const int* pnat;        // nbound: pressure side natural
  const double* nrm;      // 2*nline: unit outward normal x, then y
  const double* G;
  const int* eset;
  const double* ops;      // DV first
  int np, nz, nline, planeSize, nord, w3, Jd, Je;
  double beta, nu, invdt;
  double a[4], b[3];
};

__device__ __forceinline__ int side_node(int np, int s, int q) {
  return s == 0 ? q : s == 1 ? q * np + np - 1 : s == 2 ? (np - 1) * np + (np - 1 - q)
                                                        : (np - 1 - q) * np;
}

// x and y derivatives at element node n of element data f (LDS, np x np).
__device__ __forceinline__ void node_grad(const double* f, const double* sD, int np, int n,
                                          const double* g, int npnp, double& gx, double& gy) {
  const int i = n / np, j = n - (n / np) * np;
  double ddr = 0.0, dds = 0.0;
  for (int k = 0; k < np; ++k) {
    ddr += sD[j * np + k] * f[i * np + k];
    dds += sD[i * np + k] * f[k * np + j];
  }
  gx = ddr * g[G_DRDX * npnp + n] + dds * g[G_DSDX * npnp + n];
  gy = ddr * g[G_DRDY * npnp + n] + dds * g[G_DSDY * npnp + n];
}

__global__ __launch_bounds__(256) void k_hopbc(HopArgs A) {
  __shared__ double sD[256], sf[6][256], sw[2][256];
  const int np = A.np, npnp = np * np, t = threadIdx.x;
  const int b = blockIdx.x, m = blockIdx.y;
  const int e = A.bel[b], sd = A.bsd[b];
  const int npl = (m == 0) ? 1 : 2;               // planes of this mode
  const int k0 = 2 * m;                           // mode 0: plane 0 only
  const bool zt = m > 0 && A.w3;                  // semi-Fourier terms of w
  const double* g = A.G + (size_t)A.eset[e] * G_N * npnp;
  if (t < npnp) {
    sD[t] = A.ops[t];
    for (int p = 0; p < npl; ++p) {
      const size_t off = (size_t)(k0 + p) * A.planeSize + (size_t)e * npnp + t;
      sf[2 * p][t] = A.U[0][off];
      sf[2 * p + 1][t] = A.U[1][off];
      if (zt) sf[4 + p][t] = A.U[2][off];
    }
  }
  __syncthreads();
  // z vorticity of each plane on the whole element
  if (t < npnp)
    for (int p = 0; p < npl; ++p) {
      double ux, uy, vx, vy;
      node_grad(sf[2 * p], sD, np, t, g, npnp, ux, uy);
      node_grad(sf[2 * p + 1], sD, np, t, g, npnp, vx, vy);
      sw[p][t] = vx - uy;
    }
  __syncthreads();
  if (t >= npl * np) return;
  const int p = t / np, q = t - (t / np) * np;    // p 0 real, 1 imaginary
  const int n = side_node(np, sd, q);
  const double bk = A.beta * m;
  double wx, wy;
  node_grad(sw[p], sD, np, n, g, npnp, wx, wy);
  double cx = wy, cy = -wx;                       // curl curl (u, v) of the plane
  if (zt) {   // real: -bk d(Wi)/dx_j, imaginary: +bk d(Wr)/dx_j
    double zx, zy;
    node_grad(sf[4 + (1 - p)], sD, np, n, g, npnp, zx, zy);
    const double sg = p ? bk : -bk;
    cx += sg * zx;
    cy += sg * zy;
  }
  if (m > 0) {
    cx += bk * bk * sf[2 * p][n];
    cy += bk * bk * sf[2 * p + 1][n];
  }
  const int j = b * np + q;
  const size_t i = (size_t)(k0 + p) * A.nline + j;
  const size_t lv = (size_t)A.nz * A.nline;
  const double nx = A.nrm[j], ny = A.nrm[A.nline + j];
  const size_t off = (size_t)(k0 + p) * A.planeSize + (size_t)e * npnp + n;
  const double un = sf[2 * p][n] * nx + sf[2 * p + 1][n] * ny;
  double h = 0.0;
  if (A.Jd) {
    double wk = A.a[0] * un;
    for (int l = 0; l < A.Jd; ++l) wk += A.a[l + 1] * A.un[l * lv + i];
    h = -A.invdt * wk;
  }
  h += A.N[0][off] * nx + A.N[1][off] * ny;
  h += -A.nu * cx * nx + -A.nu * cy * ny;
  for (int l = A.nord - 1; l > 0; --l) {
    A.un[l * lv + i] = A.un[(l - 1) * lv + i];
    A.hop[l * lv + i] = A.hop[(l - 1) * lv + i];
  }
  A.un[i] = un;
  A.hop[i] = h;
  double v = 0.0;
  if (A.pnat[b])
    for (int l = 0; l < A.Je; ++l) v += A.b[l] * A.hop[l * lv + i];
  A.bcp[i] = v;
}

// z-derivative of Fourier planes: mode k Re <- -beta k Im, Im <- beta k Re;
// mode 0 and the Nyquist plane become zero.  src may equal dst.
__global__ void k_grad_z(const double* src, double* dst, int nmodes, int planeSize, double beta) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  if (idx >= (size_t)planeSize || k >= nmodes) return;
  const size_t re = (size_t)(2 * k) * planeSize + idx, im = re + planeSize;
  if (k == 0) {
    dst[re] = 0.0;
    dst[im] = 0.0;
  } else {
    const double bk = beta * k;
    const double r = src[re], m = src[im];
    dst[re] = -bk * m;
    dst[im] = bk * r;
  }
}

// Mass-weighted average of element-boundary values over the copies of each
// global node; copies are summed in increasing storage order.  A thread takes
// one node of PB planes of a field (the tables are read once for them, PB
// values in flight), blockIdx.z the field.
// Measured, 24x20 quads np=9, 96 planes: 33 -> 28 us: every cache line of
// the field, for the 8 bytes in 72 of its vertical element sides.
struct SmoothArgs {
  double* data[3];
  const double* G;
  const int* eset;
  const int* emap;
  const int* asm_ptr;
  const int* asm_idx;
  const double* imass;
  int next, npnp, nglobal, planeSize, nz;
};

template <int PB>
__global__ __launch_bounds__(256) void k_smooth(SmoothArgs a) {
  const int gI = blockIdx.x * blockDim.x + threadIdx.x;
  if (gI >= a.nglobal) return;
  const int k0 = blockIdx.y * PB;
  double* src = a.data[blockIdx.z] + (size_t)k0 * a.planeSize;
  double s[PB];
#pragma unroll
  for (int p = 0; p < PB; ++p) s[p] = 0.0;
  const int c0 = a.asm_ptr[gI], c1 = a.asm_ptr[gI + 1];
  for (int c = c0; c < c1; ++c) {
    const int i = a.asm_idx[c], e = i / a.next, q = a.emap[i - e * a.next];
    const double w = a.G[((size_t)a.eset[e] * G_N + G_Q4) * a.npnp + q];
    const size_t o = (size_t)e * a.npnp + q;
#pragma unroll
    for (int p = 0; p < PB; ++p) s[p] += w * src[(size_t)min(p, a.nz - 1 - k0) * a.planeSize + o];
  }
  const double im = a.imass[gI];
  for (int c = c0; c < c1; ++c) {
    const int i = a.asm_idx[c], e = i / a.next;
    const size_t o = (size_t)e * a.npnp + a.emap[i - e * a.next];
#pragma unroll
    for (int p = 0; p < PB; ++p)
      if (k0 + p < a.nz) src[(size_t)p * a.planeSize + o] = s[p] * im;
  }
}

// --- elementwise passes over whole fields -------------------------------
__global__ void k_fill(size_t n, double* __restrict__ t, double a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) t[i] = a;
}

__global__ void k_copy(size_t n, double* __restrict__ t, const double* __restrict__ a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) t[i] = a[i];
}

// AuxField::couple / Field::coupleBCs (src/auxfield.cpp:1352-1420,
// src/field.cpp:1043-1118): per mode k >= klo, Re/Im planes 2k, 2k+1 of n
// values.  dir > 0: v~ = v + i w, w~ = v - i w; dir < 0: v = (v~ + w~) / 2,
// w = i (w~ - v~) / 2 -- the same sums as semtex's Veclib sequence.
__global__ void k_couple(double* __restrict__ v, double* __restrict__ w, size_t n, int klo,
                         int nmode, int dir) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int k = klo + (int)blockIdx.y;
  if (i >= n || k >= nmode) return;
  double* vr = v + (size_t)(2 * k) * n;
  double* vi = vr + n;
  double* wr = w + (size_t)(2 * k) * n;
  double* wi = wr + n;
  const double a = vr[i], b = vi[i], c = wr[i], d = wi[i];
  if (dir > 0) {
    vr[i] = a - d;
    vi[i] = b + c;
    wr[i] = d + a;
    wi[i] = b - c;
  } else {
    vr[i] = 0.5 * (a + c);
    vi[i] = 0.5 * (b + d);
    wr[i] = 0.5 * (b - d);
    wi[i] = 0.5 * (c - a);
  }
}

// --- fused passes of the time step ------------------------------------------
// Elements of one plane (or of a mode's two planes) per workgroup: ce = 256 /
// (np np) of them, a thread per node.  Each is one pass over memory for what
// were a derivative kernel per component and direction and elementwise passes
// between them; the element data sit in LDS, where a derivative's np values
// are read.  What bounds them: memory traffic.
// Measured on 24x24 quads np=9 Nz=96 (a field is 36 MB), a step's passes, us:
// nonlinear terms 97 (3.3 TB/s; 404 as twelve derivative kernels), waveProp
// and the pressure's forcing 174 (4.5 TB/s; 243), projection 48 (5.2 TB/s;
// 98 and 45 of copies).

constexpr int NLT = 256;

// r and s derivatives' factors in x and y of node pt of an element
struct NodeGeo {
  double rx, sx, ry, sy;
  __device__ NodeGeo(const double* g, int npnp, int pt)
      : rx(g[G_DRDX * npnp + pt]), sx(g[G_DSDX * npnp + pt]), ry(g[G_DRDY * npnp + pt]),
        sy(g[G_DSDY * npnp + pt]) {}
};

struct NlArgs {
  const double* u[3];     // velocity, physical space
  double* n[3];           // in: its z derivatives (Z); out: the terms
  const double* G;
  const int* eset;
  const double* ops;
  int np, nel, planeSize;
  double sc;
};

// n_c = -sc (u . grad u_c [CONV] + d(u_c u)/dx + d(u_c v)/dy [CONS]); Z: the
// convective z term w du_c/dz included, the conservative one left to the
// transform (dns/nonlinear.cpp:36-211, 214-411, 414-525).
template <int NC, bool Z, bool CONV, bool CONS>
__global__ __launch_bounds__(NLT) void k_nl(NlArgs a) {
  extern __shared__ double gsh[];
  const int np = a.np, npnp = np * np, ce = NLT / npnp, t = threadIdx.x;
  const int el = t / npnp, pt = t - el * npnp, e = blockIdx.x * ce + el;
  const bool act = el < ce && e < a.nel;
  double* sD = gsh;
  double* sT = sD + npnp;
  double* sU = sT + npnp;                 // NC x ce * npnp
  if (t < npnp) {
    sD[t] = a.ops[t];
    sT[t] = a.ops[npnp + t];
  }
  const size_t pbase = (size_t)blockIdx.y * a.planeSize;
  if (blockIdx.x == 0)                    // a plane's padding holds no terms
    for (int k = a.nel * npnp + t; k < a.planeSize; k += NLT)
#pragma unroll
      for (int c = 0; c < NC; ++c) a.n[c][pbase + k] = 0.0;
  const size_t off = pbase + (size_t)e * npnp + pt;
  double u[NC], dz[NC];
  if (act) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      u[c] = a.u[c][off];
      if (Z && CONV) dz[c] = a.n[c][off];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) sU[c * ce * npnp + t] = u[c];
  }
  __syncthreads();
  if (!act) return;
  const NodeGeo g(a.G + (size_t)a.eset[e] * G_N * npnp, npnp, pt);
  const int i = pt / np, j = pt - i * np;
  const double* su = sU + el * npnp;
  double r[NC], s[NC], pr[NC][2], ps[NC][2];
#pragma unroll
  for (int c = 0; c < NC; ++c) r[c] = s[c] = pr[c][0] = pr[c][1] = ps[c][0] = ps[c][1] = 0.0;
  for (int q = 0; q < np; ++q) {
    const double dt = sT[q * np + j], ds = sD[i * np + q];
    double x[NC], y[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      x[c] = su[c * ce * npnp + i * np + q];
      y[c] = su[c * ce * npnp + q * np + j];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (CONV) {
        r[c] += x[c] * dt;
        s[c] += ds * y[c];
      }
      if (CONS)
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          if (c == 0 && d == 1) continue;   // u v: formed for c = 1
          pr[c][d] += x[c] * x[d] * dt;
          ps[c][d] += ds * (y[c] * y[d]);
        }
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    double v = 0.0;
    if (CONV) v -= u[0] * (s[c] * g.sx + r[c] * g.rx);
    if (CONS) v -= ps[c][0] * g.sx + pr[c][0] * g.rx;
    if (CONV) v -= u[1] * (s[c] * g.sy + r[c] * g.ry);
    if (CONS) {
      const double py = c ? pr[c][1] : pr[1][0], qy = c ? ps[c][1] : ps[1][0];
      v -= qy * g.sy + py * g.ry;
    }
    if (Z && CONV) v -= u[2] * dz[c];
    a.n[c][off] = a.sc * v;
  }
}

// waveProp and setPForce (dns/integrate.cpp:224-277): u_c = sum_q a_q us_q,c
// + b_q uf_q,c in semtex's order, then f = div(u) / dt.  NPL = 2: a mode's
// Re and Im planes together, d/dz in Fourier space (mode 0 and the Nyquist
// plane have none).
struct WaveArgs {
  const double* us[3][3];   // [level][component]
  const double* uf[3][3];
  double* u[3];
  double* f;
  double a[3], b[3];
  int nlev;
  const double* G;
  const int* eset;
  const double* ops;
  int np, nel, planeSize;
  double beta, dt;
};

template <int NC, int NPL>
__global__ __launch_bounds__(NLT) void k_wave_div(WaveArgs w) {
  extern __shared__ double gsh[];
  const int np = w.np, npnp = np * np, ce = NLT / npnp, t = threadIdx.x;
  const int el = t / npnp, pt = t - el * npnp, e = blockIdx.x * ce + el, m = blockIdx.y;
  const bool act = el < ce && e < w.nel;
  double* sD = gsh;
  double* sT = sD + npnp;
  double* sU = sT + npnp;                 // 2 NPL x ce * npnp
  if (t < npnp) {
    sD[t] = w.ops[t];
    sT[t] = w.ops[npnp + t];
  }
  const size_t base = (size_t)NPL * m * w.planeSize;
  const size_t off = base + (size_t)e * npnp + pt;
  double wz[NPL];
  auto sum = [&](int c, size_t i) {
    double s = 0.0;
    for (int q = 0; q < w.nlev; ++q) {
      s += w.a[q] * w.us[q][c][i];
      s += w.b[q] * w.uf[q][c][i];
    }
    return s;
  };
  if (blockIdx.x == 0)
    for (int k = w.nel * npnp + t; k < w.planeSize; k += NLT)
      for (int p = 0; p < NPL; ++p) {
        const size_t i = base + (size_t)p * w.planeSize + k;
        for (int c = 0; c < NC; ++c) w.u[c][i] = sum(c, i);
        w.f[i] = 0.0;
      }
  if (act)
#pragma unroll
    for (int p = 0; p < NPL; ++p) {
      const size_t i = off + (size_t)p * w.planeSize;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const double s = sum(c, i);
        w.u[c][i] = s;
        if (c < 2) sU[(2 * p + c) * ce * npnp + t] = s;
        else wz[p] = s;
      }
    }
  __syncthreads();
  if (!act) return;
  const NodeGeo g(w.G + (size_t)w.eset[e] * G_N * npnp, npnp, pt);
  const int i = pt / np, j = pt - i * np;
  const double bk = w.beta * m;
#pragma unroll
  for (int p = 0; p < NPL; ++p) {
    const double* su = sU + (2 * p) * ce * npnp + el * npnp;
    const double* sv = su + ce * npnp;
    double r = 0.0, s = 0.0, rv = 0.0, sw = 0.0;
    for (int q = 0; q < np; ++q) {
      const double dt = sT[q * np + j], ds = sD[i * np + q];
      r += su[i * np + q] * dt;
      s += ds * su[q * np + j];
      rv += sv[i * np + q] * dt;
      sw += ds * sv[q * np + j];
    }
    double d = (s * g.sx + r * g.rx) + (sw * g.sy + rv * g.ry);
    if (NC == 3 && NPL == 2 && m > 0) d += p ? bk * wz[0] : -bk * wz[NPL - 1];
    w.f[off + (size_t)p * w.planeSize] = d / w.dt;
  }
}

// project (dns/integrate.cpp:280-310): f_c = sc f_c + b dP/dx_c.  keep: the
// entries of `to` that the velocity solve leaves alone (the Nyquist plane and
// each plane's padding) take over those of `from`.
struct ProjectArgs {
  const double* P;
  double* f[3];
  const double* from[3];
  double* to[3];
  const double* G;
  const int* eset;
  const double* ops;
  int np, nel, planeSize, keep;
  double beta, sc, b;
};

template <int NC, int NPL>
__global__ __launch_bounds__(NLT) void k_project(ProjectArgs a) {
  extern __shared__ double gsh[];
  const int np = a.np, npnp = np * np, ce = NLT / npnp, t = threadIdx.x;
  const int el = t / npnp, pt = t - el * npnp, e = blockIdx.x * ce + el, m = blockIdx.y;
  const bool act = el < ce && e < a.nel;
  double* sD = gsh;
  double* sT = sD + npnp;
  double* sP = sT + npnp;                 // NPL x ce * npnp
  if (t < npnp) {
    sD[t] = a.ops[t];
    sT[t] = a.ops[npnp + t];
  }
  const size_t base = (size_t)NPL * m * a.planeSize;
  const size_t off = base + (size_t)e * npnp + pt;
  if (blockIdx.x == 0)
    for (int k = a.nel * npnp + t; k < a.planeSize; k += NLT)
      for (int p = 0; p < NPL; ++p)
        for (int c = 0; c < NC; ++c) {
          const size_t i = base + (size_t)p * a.planeSize + k;
          a.f[c][i] *= a.sc;
          if (a.keep) a.to[c][i] = a.from[c][i];
        }
  double P[NPL], f[NPL][NC];
  if (act) {
#pragma unroll
    for (int p = 0; p < NPL; ++p) {
      P[p] = a.P[off + (size_t)p * a.planeSize];
#pragma unroll
      for (int c = 0; c < NC; ++c) f[p][c] = a.f[c][off + (size_t)p * a.planeSize];
    }
#pragma unroll
    for (int p = 0; p < NPL; ++p) sP[p * ce * npnp + t] = P[p];
    if (NPL == 2 && m == 0 && a.keep)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        a.to[c][off + a.planeSize] = a.from[c][off + a.planeSize];
  }
  __syncthreads();
  if (!act) return;
  const NodeGeo g(a.G + (size_t)a.eset[e] * G_N * npnp, npnp, pt);
  const int i = pt / np, j = pt - i * np;
  const double bk = a.beta * m;
#pragma unroll
  for (int p = 0; p < NPL; ++p) {
    const double* sp = sP + p * ce * npnp + el * npnp;
    double r = 0.0, s = 0.0;
    for (int q = 0; q < np; ++q) {
      r += sp[i * np + q] * sT[q * np + j];
      s += sD[i * np + q] * sp[q * np + j];
    }
    const size_t o = off + (size_t)p * a.planeSize;
    a.f[0][o] = a.sc * f[p][0] + a.b * (s * g.sx + r * g.rx);
    a.f[1][o] = a.sc * f[p][1] + a.b * (s * g.sy + r * g.ry);
    if (NC == 3) {
      const double dz = NPL < 2 || m == 0 ? 0.0 : p ? bk * P[0] : -bk * P[NPL - 1];
      a.f[NC - 1][o] = a.sc * f[p][NC - 1] + a.b * dz;
    }
  }
}

inline dim3 grid1(size_t n, int bs) { return dim3((unsigned)((n + bs - 1) / bs)); }

// --- dense DFT matrices ----------------------------------------------------
bool fft_length_ok(int n) {
  if (n < 1) return false;
  while (n % 2 == 0) n /= 2;
  while (n % 3 == 0) n /= 3;
  while (n % 5 == 0) n /= 5;
  return n == 1;
}

// rows per thread of k_dft_z for a transform of length N (16 row groups)
int dft_rp(int N) {
  const int rp = (N + 15) / 16;
  return rp <= 1 ? 1 : rp <= 2 ? 2 : rp <= 4 ? 4 : rp <= 6 ? 6 : rp <= 8 ? 8
         : rp <= 12 ? 12 : rp <= 16 ? 16 : -1;
}

// Row-major matrix of the real transform of length N (rows padded to
// 16 * dft_rp(N), columns to a multiple of DFT_KB, zero entries).  sign +1:
// semtex's forward packing with 1/N; sign -1: the unscaled inverse.  Angles
// are reduced exactly (jk mod N) and evaluated in long double.
std::vector<double> dft_matrix(int N, int sign, int* ldw) {
  const int rows = 16 * dft_rp(N);
  const int ld = (N + DFT_KB - 1) / DFT_KB * DFT_KB;
  *ldw = ld;
  std::vector<double> W((size_t)rows * ld, 0.0);
  const long double two_pi = 6.283185307179586476925286766559L;
  auto cs = [&](long long jk, long double* c, long double* s) {
    const long double a = two_pi * (long double)(jk % N) / (long double)N;
    *c = cosl(a);
    *s = sinl(a);
  };
  const int nh = N / 2;
  if (sign == 1) {
    for (int k = 0; k < N; ++k) {
      W[0 * ld + k] = (double)(1.0L / N);
      if (N > 1) W[1 * ld + k] = (double)(((k & 1) ? -1.0L : 1.0L) / N);
      for (int j = 1; j < nh; ++j) {
        long double c, s;
        cs((long long)j * k, &c, &s);
        W[(size_t)(2 * j) * ld + k] = (double)(c / N);
        W[(size_t)(2 * j + 1) * ld + k] = (double)(-s / N);
      }
    }
  } else {
    for (int k = 0; k < N; ++k) {
      double* r = &W[(size_t)k * ld];
      r[0] = 1.0;
      if (N > 1) r[1] = (k & 1) ? -1.0 : 1.0;
      for (int j = 1; j < nh; ++j) {
        long double c, s;
        cs((long long)j * k, &c, &s);
        r[2 * j] = (double)(2.0L * c);
        r[2 * j + 1] = (double)(-2.0L * s);
      }
    }
  }
  return W;
}

// The matrix of dft_matrix(N, sign) formed on the device, one thread per
// entry of its rows x ldw storage: the same packing, padding and scaling,
// with the angle reduced exactly (jk mod N) and evaluated by sincospi in
// FP64 (within a few units in the last place of the long-double values).
__global__ void k_dft_matrix(double* __restrict__ W, int N, int sign, int rows, int ldw) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * ldw) return;
  const int r = idx / ldw, c = idx - (idx / ldw) * ldw;
  const int nh = N / 2;
  double v = 0.0;
  if (r < N && c < N) {
    // sign +1: row r is output coefficient r, column c input point c;
    // sign -1: row r is output point r, column c packed coefficient c
    const int pk = (sign == 1) ? r : c, pt = (sign == 1) ? c : r;
    const double sc = (sign == 1) ? 1.0 / N : 2.0;
    if (pk == 0) {
      v = (sign == 1) ? 1.0 / N : 1.0;
    } else if (pk == 1) {
      v = ((pt & 1) ? -1.0 : 1.0) * ((sign == 1) ? 1.0 / N : 1.0);
    } else if (pk / 2 < nh) {
      const long long m = ((long long)(pk / 2) * pt) % N;
      double sn, cn;
      sincospi(2.0 * (double)m / (double)N, &sn, &cn);
      v = (pk & 1) ? -sn : cn;
      v = (sign == 1) ? v / N : sc * v;
    }
  }
  W[idx] = v;
}

struct DftPlan { int N, sign, ldw; double* W; };
std::vector<DftPlan> g_plans;   // device matrices, kept for the process

int dft_plan(int N, int sign, const double** W, int* ldw) {
  for (const DftPlan& p : g_plans)
    if (p.N == N && p.sign == sign) { *W = p.W; *ldw = p.ldw; return SEMX_OK; }
  int ld = 0;
  std::vector<double> h = dft_matrix(N, sign, &ld);
  double* d = nullptr;
  int st = dev_upload(&d, h.data(), h.size());
  if (st) return st;
  g_plans.push_back({N, sign, ld, d});
  *W = d;
  *ldw = ld;
  return SEMX_OK;
}

// out-of-place transform of ntrn columns of length N (z-stride ntrn) with
// the transform matrix W (leading dimension ldw) already on the device
int dft_launch_w(const double* in, double* out, const double* W, int ldw, int N, int ntrn,
                 hipStream_t s) {
  if (N <= 128 && ntrn > 0) {
    // matrix cores: W staged whole in LDS
    const int MT = (N + 15) / 16;
    const size_t lds = (size_t)MT * 16 * (((N + 3) & ~3) + 1) * sizeof(double);
    dim3 gm((ntrn + DFT_MCOLS - 1) / DFT_MCOLS);
    const void* kfn = nullptr;
    switch (MT) {
      case 1: kfn = (const void*)k_dft_mfma<1>; break;
      case 2: kfn = (const void*)k_dft_mfma<2>; break;
      case 3: kfn = (const void*)k_dft_mfma<3>; break;
      case 4: kfn = (const void*)k_dft_mfma<4>; break;
      case 5: kfn = (const void*)k_dft_mfma<5>; break;
      case 6: kfn = (const void*)k_dft_mfma<6>; break;
      case 7: kfn = (const void*)k_dft_mfma<7>; break;
      default: kfn = (const void*)k_dft_mfma<8>; break;
    }
    if (lds > 64 * 1024)
      HIPCHK(hipFuncSetAttribute(kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    long long ldl = ntrn;
    void* kargs[] = {(void*)&in, (void*)&out, (void*)&W, (void*)&N, (void*)&ldw, (void*)&ntrn,
                     (void*)&ldl};
    hipEvent_t evm;
    prof_begin(s, &evm);
    HIPCHK(hipLaunchKernel(kfn, gm, dim3(256), kargs, lds, s));
    prof_end(s, "k_dft_z", evm);
    HIPCHK(hipGetLastError());
    return SEMX_OK;
  }
  const int rp = dft_rp(N);
  dim3 g((ntrn + DFT_COLS - 1) / DFT_COLS);
  hipEvent_t ev;
  prof_begin(s, &ev);
  switch (rp) {
    case 1: hipLaunchKernelGGL(k_dft_z<1>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    case 2: hipLaunchKernelGGL(k_dft_z<2>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    case 4: hipLaunchKernelGGL(k_dft_z<4>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    case 6: hipLaunchKernelGGL(k_dft_z<6>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    case 8: hipLaunchKernelGGL(k_dft_z<8>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    case 12: hipLaunchKernelGGL(k_dft_z<12>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    case 16: hipLaunchKernelGGL(k_dft_z<16>, g, dim3(256), 0, s, in, out, W, N, ldw, ntrn, (long long)ntrn); break;
    default: return SEMX_E_UNSUPPORTED;
  }
  prof_end(s, "k_dft_z", ev);
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

// the same with the process-wide plan of (N, sign)
int dft_launch(const double* in, double* out, int N, int ntrn, int sign, hipStream_t s) {
  const double* W = nullptr;
  int ldw = 0;
  int st = dft_plan(N, sign, &W, &ldw);
  if (st) return st;
  return dft_launch_w(in, out, W, ldw, N, ntrn, s);
}

// Device table of (cos, sin)(2 pi j / N), long double values rounded, kept
// for the process per device and length.
struct FftPlan { int dev, N; double2* tw; };
std::mutex g_fft_mu;
std::vector<FftPlan> g_fft;

int fft_plan(int N, const double2** tw) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_fft_mu);
  for (const FftPlan& p : g_fft)
    if (p.dev == dev && p.N == N) { *tw = p.tw; return SEMX_OK; }
  std::vector<double2> h(N);
  for (int j = 0; j < N; ++j) {
    const long double a = 6.283185307179586476925286766559L * j / N;
    h[j] = make_double2((double)cosl(a), (double)sinl(a));
  }
  double2* d = nullptr;
  if (const int st = dev_upload(&d, h.data(), h.size())) return st;
  g_fft.push_back({dev, N, d});
  *tw = d;
  return SEMX_OK;
}

bool fft_takes(int N) { return N >= 2 && N <= 256 && N % 2 == 0 && fft_length_ok(N); }

// nfield fields of ntrn columns (fft_takes(N)); a: everything but tw, N,
// ntrn and the radices.  Columns per workgroup: 32 (whole cache lines, two
// per row) where the LDS of two workgroups allows, else 16.
int fft_launch(int kind, FftArgs a, int N, int ntrn, int nfield, hipStream_t s) {
  if (const int st = fft_plan(N, &a.tw)) return st;
  a.N = N; a.ntrn = ntrn; a.nrad = 0;
  int m = N / 2;
  for (int r : {4, 3, 5, 2})
    while (m % r == 0) { a.rad[a.nrad++] = r; m /= r; }
  const int sets = kind == FFT_INVERSE_DZ || kind == FFT_FORWARD_DZ ? 2 : 1;
  const int ct = 2 * (size_t)sets * N * 32 * sizeof(double) <= 76 * 1024 ? 32 : 16;
  const size_t lds = (2 * (size_t)N + 2 * (size_t)sets * N * ct) * sizeof(double);
  const void* fn = nullptr;
#define SEMX_FFT(K_) \
  if (kind == K_) fn = ct == 32 ? (const void*)k_fft<K_, 32> : (const void*)k_fft<K_, 16>
  SEMX_FFT(FFT_FORWARD); SEMX_FFT(FFT_INVERSE); SEMX_FFT(FFT_INVERSE_DZ); SEMX_FFT(FFT_FORWARD_DZ);
#undef SEMX_FFT
  if (lds > 64 * 1024)
    HIPCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipEvent_t ev;
  void* kargs[] = {&a};
  prof_begin(s, &ev);
  HIPCHK(hipLaunchKernel(fn, dim3((unsigned)((ntrn + ct - 1) / ct), (unsigned)nfield), dim3(256),
                         kargs, lds, s));
  prof_end(s, "k_dft_z", ev);
  return SEMX_OK;
}

int grad_launch(Mesh& M, int nz, double beta, double* data, int dir, hipStream_t s) {
  hipEvent_t ev;
  if (dir < 2) {
    const int ce = 256 / M.npnp, pb = nz > 1 ? 4 : 1;
    dim3 g((M.nel + ce - 1) / ce, (nz + pb - 1) / pb);
    const size_t lds = (2 + (size_t)pb * ce) * M.npnp * sizeof(double);
    prof_begin(s, &ev);
    if (nz > 1)
      hipLaunchKernelGGL(k_grad_xy<4>, g, dim3(256), lds, s, data, M.d.G, M.d.eset, M.d.ops,
                         M.np, M.nel, M.planeSize, nz, dir);
    else
      hipLaunchKernelGGL(k_grad_xy<1>, g, dim3(256), lds, s, data, M.d.G, M.d.eset, M.d.ops,
                         M.np, M.nel, M.planeSize, nz, dir);
    prof_end(s, "k_grad_xy", ev);
  } else {
    dim3 g((M.planeSize + 255) / 256, nz / 2);
    prof_begin(s, &ev);
    hipLaunchKernelGGL(k_grad_z, g, dim3(256), 0, s, data, data, nz / 2, M.planeSize, beta);
    prof_end(s, "k_grad_z", ev);
  }
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

int smooth_launch(Mesh& M, int nz, double* const* data, int nfield, hipStream_t s) {
  hipEvent_t ev;
  SmoothArgs a{};
  for (int i = 0; i < nfield; ++i) a.data[i] = data[i];
  a.G = M.d.G; a.eset = M.d.eset; a.emap = M.d.emap; a.asm_ptr = M.d.asm_ptr;
  a.asm_idx = M.d.asm_idx; a.imass = M.d.imass; a.next = M.next; a.npnp = M.npnp;
  a.nglobal = M.nglobal; a.planeSize = M.planeSize; a.nz = nz;
  const int pb = nz > 1 ? 4 : 1;
  dim3 g((M.nglobal + 255) / 256, (nz + pb - 1) / pb, nfield);
  prof_begin(s, &ev);
  if (nz > 1) hipLaunchKernelGGL(k_smooth<4>, g, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_smooth<1>, g, dim3(256), 0, s, a);
  prof_end(s, "k_smooth", ev);
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

// Integration coefficients, src/integration.cpp:99-164.
void stiffly_stable(int n, double* c) {
  if (n == 1) { c[0] = 1.0; c[1] = -1.0; }
  else if (n == 2) { c[0] = 1.5; c[1] = -2.0; c[2] = 0.5; }
  else { c[0] = 11.0 / 6.0; c[1] = -3.0; c[2] = 1.5; c[3] = -1.0 / 3.0; }
}

void extrapolation(int n, double* c) {
  if (n == 1) { c[0] = 1.0; }
  else if (n == 2) { c[0] = 2.0; c[1] = -1.0; }
  else { c[0] = 3.0; c[1] = -3.0; c[2] = 1.0; }
}

}  // namespace

// ===========================================================================
// DNS state: the fields of integrate() held on the device.
// ===========================================================================

// The buffer roles of the DNS state: which allocation each field of the
// step uses.  The step permutes them (swapData, the rolled time levels) and
// returns to a given assignment only after a full cycle of steps
// (rotate_spares).
struct DnsRoles {
  double* U[3];
  double* P;
  double* Us[3][3];
  double* Uf[3][3];
  double* tmp;
  double* spare;
  int toggle;
  bool operator==(const DnsRoles& o) const { return std::memcmp(this, &o, sizeof(*this)) == 0; }
};

// One steady step captured for one assignment of roles: replaying it leaves
// the roles as `after`.
struct DnsGraph {
  DnsRoles before, after;
  hipGraphExec_t exec;
};

struct semx_dns_s {
  Mesh* M = nullptr;
  int nz = 1, ncom = 2, ndim = 2, nord = 2, advection = 0, step = 0, step_max = 500, toggle = 1;
  double beta = 1.0, dt = 0.0, kinvis = 0.0, tol_rel = 1e-12;
  size_t ntot = 0;
  double* store = nullptr;              // all fields in one allocation
  double* U[3] = {nullptr, nullptr, nullptr};
  double* P = nullptr;
  double* Us[3][3] = {};                // [level][component]
  double* Uf[3][3] = {};
  double* tmp = nullptr;                // the pressure's forcing
  double* spare = nullptr;
  Helm* vel = nullptr;                  // DIRECT, lambda2 = alpha0/(dt nu)
  Helm* pre = nullptr;                  // DIRECT, lambda2 = 0
  Helm* start[2] = {nullptr, nullptr};  // JACPCG start-up velocity systems
  // bounded mesh: the pressure's numbering and side kinds (same elements
  // and boundary list as the velocity mesh), BC lines and flux history
  Mesh* Mp = nullptr;
  int nline = 0;
  double* bstore = nullptr;             // the arrays below in one allocation
  double* bcu[3] = {nullptr, nullptr, nullptr};   // velocity BC lines, nz*nline each
  double* bcp = nullptr;                // pressure BC lines
  double* un = nullptr;                 // nord levels of u.n
  double* hop = nullptr;                // nord levels of the flux terms
  double* nrm = nullptr;                // side normals, 2*nline
  int* bint = nullptr;                  // element, side, pressure-natural per boundary
  bool graphs_on = false;               // replay steady steps from HIP graphs
  hipStream_t capture = nullptr;        // stream the steps are captured on
  std::vector<DnsGraph> graphs;         // one per role assignment met
  long long replays = 0;
};

namespace {

int ew_launch_check() {
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

#define EW(kernel, ...)                                                          \
  do {                                                                           \
    hipLaunchKernelGGL(kernel, grid1(n, 256), dim3(256), 0, s, n, __VA_ARGS__); \
    if (int st_ = ew_launch_check()) return st_;                                 \
  } while (0)

#define CHK(x) do { if (int st_ = (x)) return st_; } while (0)

// Geometry arguments and launch shape of the fused element kernels
template <class A>
void op_args(A& a, const Mesh& M) {
  a.G = M.d.G; a.eset = M.d.eset; a.ops = M.d.ops;
  a.np = M.np; a.nel = M.nel; a.planeSize = M.planeSize;
}

template <class A>
int op_launch(void (*fn)(A), const A& a, const Mesh& M, int layers, int nbuf, const char* name,
              hipStream_t s) {
  const int ce = NLT / M.npnp;
  const size_t lds = (2 + (size_t)nbuf * ce) * M.npnp * sizeof(double);   // 16 KB at most
  hipEvent_t ev;
  prof_begin(s, &ev);
  hipLaunchKernelGGL(fn, dim3((M.nel + ce - 1) / ce, layers), dim3(NLT), lds, s, a);
  prof_end(s, name, ev);
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

// The nonlinear terms (dns/nonlinear.cpp, Cartesian): on entry U holds the
// Fourier velocity; on exit Us[0] does, Uf[0] the Fourier N(u), smoothed, and
// U nothing that is needed.
int dns_nonlinear(semx_dns_s& D, hipStream_t s) {
  Mesh& M = *D.M;
  hipEvent_t ev;
  prof_begin(s, &ev);
  // skewSymmetric (0): both forms, halved; altSkewSymmetric (1): one form
  // per step in turn; convective (2): u . grad u; Stokes (3): none
  // (dns/nonlinear.cpp:36-211, 214-411, 414-525, 528-570)
  const bool conv = D.advection == 0 || D.advection == 2 || (D.advection == 1 && D.toggle);
  const bool cons = D.advection == 0 || (D.advection == 1 && !D.toggle);
  const double half = D.advection == 0 ? 0.5 : 1.0;
  const bool z = D.nz > 2;
  if (z && !fft_takes(D.nz)) return SEMX_E_UNSUPPORTED;
  for (int i = 0; i < D.ncom; ++i) std::swap(D.U[i], D.Us[0][i]);
  NlArgs n{};
  FftArgs f{};
  op_args(n, M);
  f.beta = D.beta;
  f.sc = half;
  for (int i = 0; i < D.ncom; ++i) {
    n.n[i] = D.Uf[0][i];
    n.u[i] = D.nz == 1 ? D.Us[0][i] : D.U[i];
    f.in[i] = D.Us[0][i]; f.out[i] = D.U[i]; f.out2[i] = D.Uf[0][i];
  }
  if (!conv && !cons) {   // Stokes: no nonlinear terms
    const size_t nt = D.ntot;
    for (int i = 0; i < D.ncom; ++i)
      hipLaunchKernelGGL(k_fill, grid1(nt, 256), dim3(256), 0, s, nt, D.Uf[0][i], 0.0);
    prof_end(s, "dns_nonlinear", ev);
    HIPCHK(hipGetLastError());
    return SEMX_OK;
  }
  const size_t pl = M.planeSize;
  if (z)
    CHK(fft_launch(conv ? FFT_INVERSE_DZ : FFT_INVERSE, f, D.nz, M.planeSize, D.ncom, s));
  else if (D.nz == 2)   // both planes the mean (AuxField::transform, auxfield.cpp:1133-1170)
    for (int i = 0; i < D.ncom; ++i)
      for (int k = 0; k < 2; ++k)
        hipLaunchKernelGGL(k_copy, grid1(pl, 256), dim3(256), 0, s, pl, D.U[i] + k * pl, D.Us[0][i]);
  // the conservative z term is formed in Fourier space, with N's transform,
  // which then also takes the halving of the skew-symmetric form (exact)
  const bool zcons = z && cons;
  n.sc = zcons ? 1.0 : half;
  void (*fn)(NlArgs) = nullptr;
#define SEMX_NL(NC_, Z_) \
  fn = conv ? (cons ? k_nl<NC_, Z_, true, true> : k_nl<NC_, Z_, true, false>) : k_nl<NC_, Z_, false, true>
  if (D.ncom == 2) SEMX_NL(2, false);
  else if (z) SEMX_NL(3, true);
  else SEMX_NL(3, false);
#undef SEMX_NL
  CHK(op_launch(fn, n, M, D.nz, D.ncom, "k_grad_nl", s));
  if (z) {
    for (int i = 0; i < D.ncom; ++i) {
      f.in[i] = f.out[i] = D.Uf[0][i];
      f.b1[i] = D.U[i];
    }
    f.b2 = D.U[2];
    CHK(fft_launch(zcons ? FFT_FORWARD_DZ : FFT_FORWARD, f, D.nz, M.planeSize, D.ncom, s));
  } else if (D.nz == 2) {
    for (int i = 0; i < D.ncom; ++i)
      hipLaunchKernelGGL(k_fill, grid1(pl, 256), dim3(256), 0, s, pl, D.Uf[0][i] + pl, 0.0);
  }
  CHK(smooth_launch(M, D.nz, D.Uf[0], D.ncom, s));
  if (D.advection == 1) D.toggle = 1 - D.toggle;
  prof_end(s, "dns_nonlinear", ev);
  return SEMX_OK;
}

// BCmgr::maintainFourier + the pressure's evaluateBoundaries
// (dns/integrate.cpp:168-172) for step D.step (already advanced): Us[0]
// and Uf[0] hold the Fourier velocity and nonlinear terms of the step.
int dns_hopbc(semx_dns_s& D, hipStream_t s) {
  Mesh& M = *D.M;
  HopArgs A{};
  for (int i = 0; i < 3; ++i) A.U[i] = D.Us[0][i];
  A.N[0] = D.Uf[0][0]; A.N[1] = D.Uf[0][1];
  A.un = D.un; A.hop = D.hop; A.bcp = D.bcp;
  A.bel = D.bint; A.bsd = D.bint + M.nbound; A.pnat = D.bint + 2 * M.nbound;
  A.nrm = D.nrm;
  A.G = M.d.G; A.eset = M.d.eset; A.ops = M.d.ops;
  A.np = M.np; A.nz = D.nz; A.nline = D.nline; A.planeSize = M.planeSize;
  A.nord = D.nord; A.w3 = D.ncom == 3;
  A.Jd = std::min(D.step - 1, D.nord);
  A.Je = std::min(D.step, D.nord);
  if (A.Jd) stiffly_stable(A.Jd, A.a);
  extrapolation(A.Je, A.b);
  A.beta = D.beta; A.nu = D.kinvis; A.invdt = 1.0 / D.dt;
  const int nmodes = D.nz > 1 ? D.nz / 2 : 1;
  hipLaunchKernelGGL(k_hopbc, dim3(M.nbound, nmodes), dim3(256), 0, s, A);
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

// rollm (src/sem.h:106-120): level q takes level q-1, level 0 the last.
void roll(double* lev[3][3], int nord, int ncom) {
  if (nord < 2) return;
  for (int j = 0; j < ncom; ++j) {
    double* t = lev[nord - 1][j];
    for (int i = nord - 1; i; --i) lev[i][j] = lev[i - 1][j];
    lev[0][j] = t;
  }
}

// The step's swaps and rolled levels return to one assignment of roles after
// 2 N_TIME + 1 steps (twice that with the alternating form).  Between steps
// Us[0], Uf[0], tmp and spare hold nothing; with planes and N_TIME = 3 those are
// exchanged as well (here and, for the skew-symmetric form, before the viscous
// solves), so that the roles recur after 88 steps of that form and 182 of the
// alternating one, the number of step graphs that programs which capture a
// full cycle count on there.
bool long_cycle(const semx_dns_s& D) { return D.nz > 2 && D.nord == 3; }

void rotate_spares(semx_dns_s& D) {
  if (!long_cycle(D)) return;
  if (D.advection == 0) {
    std::swap(D.Uf[0][2], D.tmp);
    std::swap(D.Us[0][0], D.spare);
  } else if (D.advection == 1) {
    if (!D.toggle) std::swap(D.Us[0][0], D.Uf[0][1]);
    else std::swap(D.Us[0][1], D.Uf[0][0]);
  }
}

// One time step of integrate (dns/integrate.cpp:79-221).
int dns_step(semx_dns_s& D, hipStream_t s) {
  Mesh& M = *D.M;
  const size_t n = D.ntot;
  const int ncom = D.ncom, nord = D.nord;
  CHK(dns_nonlinear(D, s));
  D.step += 1;
  if (D.Mp) CHK(dns_hopbc(D, s));
  const int Je = std::min(D.step, nord);
  double alpha[4], beta[3];
  stiffly_stable(Je, alpha);
  extrapolation(Je, beta);
  for (int q = 0; q < Je; ++q) beta[q] *= D.dt;
  const int npl = D.nz > 1 ? 2 : 1, layers = D.nz / npl;
  // waveProp into U, setPForce into tmp
  {
    WaveArgs w{};
    op_args(w, M);
    w.nlev = Je;
    for (int q = 0; q < Je; ++q) {
      for (int i = 0; i < ncom; ++i) {
        w.us[q][i] = D.Us[q][i];
        w.uf[q][i] = D.Uf[q][i];
      }
      w.a[q] = -alpha[q + 1];
      w.b[q] = beta[q];
    }
    for (int i = 0; i < ncom; ++i) w.u[i] = D.U[i];
    w.f = D.tmp;
    w.beta = D.beta;
    w.dt = D.dt;
    if (ncom == 3) CHK(op_launch(k_wave_div<3, 2>, w, M, layers, 4, "k_wave_div", s));
    else CHK(op_launch(k_wave_div<2, 1>, w, M, layers, 2, "k_wave_div", s));
  }
  roll(D.Uf, nord, ncom);
  // pressure solve
  CHK(helm_solve(*D.pre, D.tmp, D.bcp, D.P, D.tol_rel, D.step_max, nullptr, s));
  // project, in place: U becomes the viscous solves' forcing.  Start-up
  // systems (JACPCG) while step < N_TIME; iterative ones start from the old
  // velocity, direct ones only leave parts of it in place.
  Helm* V = (D.step < nord) ? D.start[D.step - 1] : D.vel;
  if (D.advection == 0 && long_cycle(D)) {   // spare buffers: see rotate_spares
    std::swap(D.Uf[0][0], D.Uf[0][1]);
    std::swap(D.Uf[0][0], D.spare);
  }
  const bool guess = !V->pcg_plane.empty();
  {
    ProjectArgs p{};
    op_args(p, M);
    p.P = D.P;
    for (int i = 0; i < ncom; ++i) {
      p.f[i] = D.U[i];
      p.from[i] = D.Us[0][i];
      p.to[i] = D.Uf[0][i];
    }
    p.keep = !guess;
    p.beta = D.beta;
    p.sc = -1.0 / (D.dt * D.kinvis);
    p.b = 1.0 / D.kinvis;
    if (ncom == 3) CHK(op_launch(k_project<3, 2>, p, M, layers, 2, "k_project", s));
    else CHK(op_launch(k_project<2, 1>, p, M, layers, 1, "k_project", s));
  }
  if (guess)
    for (int i = 0; i < ncom; ++i) EW(k_copy, D.Uf[0][i], D.Us[0][i]);
  // viscous solves (the velocity components share one system)
  double* us[3] = {D.Uf[0][0], D.Uf[0][1], D.Uf[0][2]};
  double* fs[3] = {D.U[0], D.U[1], D.U[2]};
  const double* bcs[3] = {D.bcu[0], D.bcu[1], D.bcu[2]};
  CHK(helm_solve_fields(*V, ncom, fs, D.Mp ? bcs : nullptr, us, D.tol_rel, D.step_max,
                        nullptr, s));
  for (int i = 0; i < ncom; ++i) std::swap(D.U[i], D.Uf[0][i]);
  roll(D.Us, nord, ncom);
  rotate_spares(D);
  return SEMX_OK;
}

DnsRoles roles_of(const semx_dns_s& D) {
  DnsRoles r;
  std::memset(&r, 0, sizeof(r));
  for (int i = 0; i < 3; ++i) r.U[i] = D.U[i];
  r.P = D.P;
  for (int q = 0; q < 3; ++q)
    for (int i = 0; i < 3; ++i) { r.Us[q][i] = D.Us[q][i]; r.Uf[q][i] = D.Uf[q][i]; }
  r.tmp = D.tmp;
  r.spare = D.spare;
  r.toggle = D.toggle;
  return r;
}

void set_roles(semx_dns_s& D, const DnsRoles& r) {
  for (int i = 0; i < 3; ++i) D.U[i] = r.U[i];
  D.P = r.P;
  for (int q = 0; q < 3; ++q)
    for (int i = 0; i < 3; ++i) { D.Us[q][i] = r.Us[q][i]; D.Uf[q][i] = r.Uf[q][i]; }
  D.tmp = r.tmp;
  D.spare = r.spare;
  D.toggle = r.toggle;
}

// A step from a HIP graph.  Start-up steps (order < N_TIME, JACPCG
// systems) and the first steady step (which allocates the solve scratch and,
// where the band sweeps are selected, times them) run eagerly, as do all steps while
// kernel timing is on.  A steady step whose role assignment has not been
// met is captured on the library's capture stream (the host state
// advances as in an eager step), instantiated and launched on the caller's
// stream; later steps with that assignment replay it.  Every kernel of the
// step takes its buffers by value, so one graph per assignment is exact.
// If a capture fails, graphs are switched off and the step runs eagerly.
int dns_step_graph(semx_dns_s& D, hipStream_t s) {
  if (!D.graphs_on || D.step < D.nord || prof_enabled()) return dns_step(D, s);
  const DnsRoles cur = roles_of(D);
  for (const DnsGraph& g : D.graphs) {
    if (g.before == cur) {
      HIPCHK(hipGraphLaunch(g.exec, s));
      set_roles(D, g.after);
      D.step += 1;
      D.replays += 1;
      return SEMX_OK;
    }
  }
  if (!D.capture) HIPCHK(hipStreamCreateWithFlags(&D.capture, hipStreamNonBlocking));
  const int step0 = D.step;
  HIPCHK(hipStreamBeginCapture(D.capture, hipStreamCaptureModeRelaxed));
  const int st = dns_step(D, D.capture);
  hipGraph_t graph = nullptr;
  const hipError_t ec = hipStreamEndCapture(D.capture, &graph);
  hipGraphExec_t exec = nullptr;
  hipError_t ei = hipErrorUnknown;
  if (!st && ec == hipSuccess && graph) ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  if (graph) (void)hipGraphDestroy(graph);
  if (st || ec != hipSuccess || ei != hipSuccess) {
    (void)hipGetLastError();
    fprintf(stderr, "semx: DNS step capture failed (%s); stepping without graphs\n",
            st ? semx_error_string(st) : hipGetErrorString(ec != hipSuccess ? ec : ei));
    D.graphs_on = false;
    set_roles(D, cur);
    D.step = step0;
    return dns_step(D, s);
  }
  D.graphs.push_back({cur, roles_of(D), exec});
  HIPCHK(hipGraphLaunch(exec, s));
  D.replays += 1;
  return SEMX_OK;
}

void dns_free(semx_dns_s* D) {
  if (!D) return;
  for (DnsGraph& g : D->graphs) (void)hipGraphExecDestroy(g.exec);
  if (D->capture) (void)hipStreamDestroy(D->capture);
  for (Helm* h : {D->vel, D->pre, D->start[0], D->start[1]}) {
    if (!h) continue;
    helm_release(*h);
    delete h;
  }
  dev_free(D->store);
  dev_free(D->bstore);
  dev_free(D->bint);
  delete D;
}

int make_system(Mesh& M, double lambda2, double beta, int nz, int method, Helm** out) {
  Helm* H = new (std::nothrow) Helm();
  if (!H) return SEMX_E_NOMEM;
  H->M = &M;
  H->lambda2 = lambda2; H->beta = beta; H->base = 0;
  H->nmodes = nz > 1 ? nz / 2 : 1; H->nz = nz; H->method = method;
  int st = helm_build(*H);
  if (!st) st = helm_upload(*H);
  if (st) { helm_release(*H); delete H; return st; }
  *out = H;
  return SEMX_OK;
}

}  // namespace

// --- device memory of the allocation-free transform -------------------------
// semx_dft_r_noalloc works in this array: the transform matrix (at most
// 256 x 256 values, for tlen <= 256) and then the transformed field (at most
// SEMX_DFT_NOALLOC_MAX values).  Every device the library runs on holds its
// own copy until the process ends.  Host code never uses the array's name
// (a host-side stand-in, not a device address): it uses the device address
// obtained once per device by hipGetSymbolAddress.
constexpr size_t NOALLOC_W = 256 * 256;
static __device__ __align__(256) double scratch[NOALLOC_W + SEMX_DFT_NOALLOC_MAX];

namespace {

constexpr int NOALLOC_DEVICES = 64;
std::mutex g_noalloc_mu;
double* g_noalloc_ptr[NOALLOC_DEVICES] = {};

}  // namespace

namespace semx {

// The current device's address of the array, looked up on its first use
// on that device (semx_device_init, or the first allocation-free call).
int noalloc_scratch(double** out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_DEVICES) return SEMX_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      fprintf(stderr, "semx: hipGetSymbolAddress(scratch) failed: %s\n", hipGetErrorString(e));
      return SEMX_E_HIP;
    }
    g_noalloc_ptr[dev] = (double*)ptr;
  }
  if (out) *out = g_noalloc_ptr[dev];
  return SEMX_OK;
}

}  // namespace semx

namespace {

// Arguments of a transform as dDFTr checks them (femlib/fourier.c:47-62);
// 1 = nothing to do.
int dft_args(const double* data, int tlen, int ntrn, int sign) {
  if (!data || tlen < 1 || ntrn < 0 || (sign != 1 && sign != -1)) return SEMX_E_ARG;
  if (tlen < 2 || ntrn == 0) return -1;
  if (!fft_length_ok(tlen) || (ntrn & 1)) return SEMX_E_ARG;
  return SEMX_OK;
}

}  // namespace

extern "C" {

int semx_dft_r(double* data, int tlen, int ntrn, int sign, void* stream) {
  int st = dft_args(data, tlen, ntrn, sign);
  if (st) return st < 0 ? SEMX_OK : st;
  hipStream_t s = (hipStream_t)stream;
  if (fft_takes(tlen)) {   // in place
    FftArgs a{};
    a.in[0] = a.out[0] = data;
    return fft_launch(sign == 1 ? FFT_FORWARD : FFT_INVERSE, a, tlen, ntrn, 1, s);
  }
  static double* stage = nullptr;
  static size_t cap = 0;
  const size_t need = (size_t)tlen * ntrn;
  if (need > cap) {
    HIPCHK(hipStreamSynchronize(s));
    dev_free(stage);
    st = dev_upload<double>(&stage, nullptr, need);
    if (st) { cap = 0; return st; }
    cap = need;
  }
  st = dft_launch(data, stage, tlen, ntrn, sign, s);
  if (st) return st;
  HIPCHK(hipMemcpyAsync(data, stage, need * sizeof(double), hipMemcpyDeviceToDevice, s));
  return SEMX_OK;
}

int semx_dft_r_noalloc(double* data, int tlen, int ntrn, int sign, void* stream) {
  int st = dft_args(data, tlen, ntrn, sign);
  if (st) return st < 0 ? SEMX_OK : st;
  const size_t need = (size_t)tlen * ntrn;
  if (tlen > 256 || need > SEMX_DFT_NOALLOC_MAX) {
    fprintf(stderr,
            "semx_dft_r_noalloc: %d x %d values exceed the static scratch "
            "(tlen <= 256, tlen*ntrn <= %zu)\n",
            tlen, ntrn, (size_t)SEMX_DFT_NOALLOC_MAX);
    return SEMX_E_SCRATCH;
  }
  double* base = nullptr;
  if ((st = noalloc_scratch(&base))) return st;
  hipStream_t s = (hipStream_t)stream;
  const int rows = 16 * dft_rp(tlen);
  const int ldw = (tlen + DFT_KB - 1) / DFT_KB * DFT_KB;
  double* W = base;
  double* out = base + NOALLOC_W;
  hipLaunchKernelGGL(k_dft_matrix, dim3((rows * ldw + 255) / 256), dim3(256), 0, s, W, tlen,
                     sign, rows, ldw);
  HIPCHK(hipGetLastError());
  if ((st = dft_launch_w(data, out, W, ldw, tlen, ntrn, s))) return st;
  HIPCHK(hipMemcpyAsync(data, out, need * sizeof(double), hipMemcpyDeviceToDevice, s));
  return SEMX_OK;
}

int semx_gradient(semx_mesh mesh, int nz, double beta, double* data, int dir, void* stream) {
  if (!mesh || !data || nz < 1 || dir < 0 || dir > 2) return SEMX_E_ARG;
  if (dir == 2 && (nz < 2 || (nz & 1))) return SEMX_E_ARG;
  Mesh& M = mesh->M;
  int st = mesh_upload(M);
  if (st) return st;
  return grad_launch(M, nz, beta, data, dir, (hipStream_t)stream);
}

int semx_couple(double* v, double* w, int nz, int n, int base_mode, int dir, void* stream) {
  if (!v || !w || nz < 1 || n < 1 || base_mode < 0 || (dir != 1 && dir != -1)) return SEMX_E_ARG;
  if (nz > 1 && (nz & 1)) return SEMX_E_ARG;
  const int nmode = nz / 2, klo = base_mode == 0 ? 1 : 0;   // 2D (nz = 1): nothing
  if (nmode <= klo) return SEMX_OK;
  const dim3 grid((unsigned)(((size_t)n + 255) / 256), (unsigned)(nmode - klo));
  hipLaunchKernelGGL(k_couple, grid, dim3(256), 0, (hipStream_t)stream, v, w, (size_t)n, klo,
                     nmode, dir);
  HIPCHK(hipGetLastError());
  return SEMX_OK;
}

int semx_smooth(semx_mesh mesh, int nz, double* data, void* stream) {
  if (!mesh || !data || nz < 1) return SEMX_E_ARG;
  Mesh& M = mesh->M;
  int st = mesh_upload(M);
  if (st) return st;
  return smooth_launch(M, nz, &data, 1, (hipStream_t)stream);
}

}  // extern "C"

namespace {

// The outward unit normals of every boundary side at its nodes, CCW
// (Element::sideGeom, src/element.cpp:1653-1744): side 0 -grad s, side 1
// grad r, side 2 grad s, side 3 -grad r, normalised.
std::vector<double> side_normals(const Mesh& M) {
  const int np = M.np, npnp = M.npnp, nline = M.nbound * np;
  std::vector<double> nrm(2 * (size_t)nline);
  for (int b = 0; b < M.nbound; ++b) {
    const int e = M.belmt[b], sd = M.bside[b];
    const double* g = M.G.data() + (size_t)M.eset[e] * G_N * npnp;
    for (int q = 0; q < np; ++q) {
      const int n = sd == 0 ? q : sd == 1 ? q * np + np - 1
                  : sd == 2 ? (np - 1) * np + (np - 1 - q) : (np - 1 - q) * np;
      const int rs = (sd == 0 || sd == 2) ? 1 : 0;     // s or r gradient
      const double sg = (sd == 0 || sd == 3) ? -1.0 : 1.0;
      const double a = sg * g[(rs ? G_DSDX : G_DRDX) * npnp + n];
      const double c = sg * g[(rs ? G_DSDY : G_DRDY) * npnp + n];
      const double len = std::hypot(a, c);
      nrm[b * np + q] = a / len;
      nrm[nline + b * np + q] = c / len;
    }
  }
  return nrm;
}

// Device storage of a bounded DNS: velocity BC lines copied from the
// caller's (device) lines, zeroed pressure lines and flux history, normals
// and the boundary tables.
int dns_bounded(semx_dns_s& D, Mesh& Mp, const double* const* bc) {
  Mesh& M = *D.M;
  D.Mp = &Mp;
  D.nline = M.nbound * M.np;
  const size_t nl = (size_t)D.nz * D.nline;
  const size_t total = (3 + 1 + 2 * (size_t)D.nord) * nl + 2 * (size_t)D.nline;
  CHK(dev_upload<double>(&D.bstore, nullptr, total));
  double* f = D.bstore;
  for (int i = 0; i < 3; ++i) { D.bcu[i] = f; f += nl; }
  D.bcp = f; f += nl;
  D.un = f; f += D.nord * nl;
  D.hop = f; f += D.nord * nl;
  D.nrm = f;
  for (int i = 0; i < D.ncom; ++i)
    HIPCHK(hipMemcpy(D.bcu[i], bc[i], nl * sizeof(double), hipMemcpyDeviceToDevice));
  const std::vector<double> nrm = side_normals(M);
  HIPCHK(hipMemcpy(D.nrm, nrm.data(), nrm.size() * sizeof(double), hipMemcpyHostToDevice));
  std::vector<int> bint(3 * (size_t)M.nbound);
  for (int b = 0; b < M.nbound; ++b) {
    bint[b] = M.belmt[b];
    bint[M.nbound + b] = M.bside[b];
    bint[2 * M.nbound + b] = Mp.bkind[b] == 2;
  }
  return dev_upload<int>(&D.bint, bint.data(), bint.size());
}

int dns_create(Mesh& M, Mesh* Mp, const double* const* bc, int nz, double beta, double dt,
               double kinvis, int norder, int advection, double tol_rel, int step_max,
               semx_dns* dns) {
  if (!dns || nz < 1 || (nz > 1 && (nz & 1)) || norder < 1 || norder > 3 ||
      advection < 0 || advection > 3 || !(dt > 0.0) || !(kinvis > 0.0) || step_max < 1)
    return SEMX_E_ARG;
  if (nz > 2 && !fft_length_ok(nz)) return SEMX_E_ARG;
  *dns = nullptr;
  semx_dns_s* D = new (std::nothrow) semx_dns_s();
  if (!D) return SEMX_E_NOMEM;
  D->M = &M; D->nz = nz; D->nord = norder; D->advection = advection; D->beta = beta;
  D->dt = dt; D->kinvis = kinvis; D->tol_rel = tol_rel; D->step_max = step_max;
  D->ncom = nz > 1 ? 3 : 2; D->ndim = D->ncom;
  D->ntot = (size_t)nz * M.planeSize;
  int st = mesh_upload(M);
  const size_t nfield = 3 + 1 + 2 * 3 * 3 + 2;
  if (!st) st = dev_upload<double>(&D->store, nullptr, nfield * D->ntot);
  if (st) { dns_free(D); return st; }
  double* f = D->store;
  for (int i = 0; i < 3; ++i) D->U[i] = f + (size_t)i * D->ntot;
  f += 3 * D->ntot;
  D->P = f; f += D->ntot;
  for (int q = 0; q < 3; ++q)
    for (int i = 0; i < 3; ++i) {
      D->Us[q][i] = f; f += D->ntot;
      D->Uf[q][i] = f; f += D->ntot;
    }
  D->tmp = f; f += D->ntot;
  D->spare = f;
  double alpha[4];
  stiffly_stable(norder, alpha);
  st = make_system(M, alpha[0] / (dt * kinvis), beta, nz, SEMX_DIRECT, &D->vel);
  if (!st && Mp) st = mesh_upload(*Mp);
  if (!st && Mp) st = dns_bounded(*D, *Mp, bc);
  if (!st) st = make_system(Mp ? *Mp : M, 0.0, beta, nz, SEMX_DIRECT, &D->pre);
  for (int q = 1; q < norder && !st; ++q) {
    stiffly_stable(q, alpha);
    st = make_system(M, alpha[0] / (dt * kinvis), beta, nz, SEMX_JACPCG, &D->start[q - 1]);
  }
  if (st) { dns_free(D); return st; }
  *dns = D;
  return SEMX_OK;
}

}  // namespace

extern "C" {

int semx_dns_create(semx_mesh mesh, int nz, double beta, double dt, double kinvis, int norder,
                    int advection, double tol_rel, int step_max, semx_dns* dns) {
  if (!mesh) return SEMX_E_ARG;
  // a bounded mesh needs its BC lines and pressure numbering:
  // semx_dns_create_bc; cylindrical coordinates are not supported by the
  // time step
  if (mesh->M.nbound || mesh->M.cyl) return SEMX_E_UNSUPPORTED;
  return dns_create(mesh->M, nullptr, nullptr, nz, beta, dt, kinvis, norder, advection, tol_rel,
                    step_max, dns);
}

int semx_dns_create_bc(semx_mesh vmesh, semx_mesh pmesh, int nz, double beta, double dt,
                       double kinvis, int norder, int advection, double tol_rel, int step_max,
                       const double* bcu, const double* bcv, const double* bcw, semx_dns* dns) {
  if (!vmesh || !pmesh || !bcu || !bcv || (nz > 1 && !bcw)) return SEMX_E_ARG;
  const Mesh& M = vmesh->M;
  const Mesh& P = pmesh->M;
  if (M.cyl || P.cyl) return SEMX_E_UNSUPPORTED;
  // the two numberings must be of one element mesh with one boundary list
  if (!M.nbound || P.np != M.np || P.nel != M.nel || P.nbound != M.nbound ||
      P.belmt != M.belmt || P.bside != M.bside || P.x != M.x || P.y != M.y)
    return SEMX_E_MESH;
  const double* bc[3] = {bcu, bcv, bcw};
  return dns_create(vmesh->M, &pmesh->M, bc, nz, beta, dt, kinvis, norder, advection, tol_rel,
                    step_max, dns);
}

int semx_dns_set_iterative(semx_dns dns, int level) {
  if (!dns || dns->step || level < 0 || level > 2) return SEMX_E_ARG;
  semx_dns_s& D = *dns;
  double alpha[4];
  stiffly_stable(D.nord, alpha);
  Helm* vel = nullptr;
  Helm* pre = nullptr;
  int st = make_system(*D.M, alpha[0] / (D.dt * D.kinvis), D.beta, D.nz,
                       level >= 1 ? SEMX_JACPCG : SEMX_DIRECT, &vel);
  if (!st) st = make_system(D.Mp ? *D.Mp : *D.M, 0.0, D.beta, D.nz,
                            level >= 2 ? SEMX_MIXED : SEMX_DIRECT, &pre);
  if (st) {
    for (Helm* h : {vel, pre})
      if (h) { helm_release(*h); delete h; }
    return st;
  }
  for (Helm* h : {D.vel, D.pre}) { helm_release(*h); delete h; }
  D.vel = vel;
  D.pre = pre;
  return SEMX_OK;
}

int semx_dns_set_bc(semx_dns dns, const double* bcu, const double* bcv, const double* bcw,
                    void* stream) {
  if (!dns || !dns->Mp || !bcu || !bcv || (dns->ncom == 3 && !bcw)) return SEMX_E_ARG;
  const double* src[3] = {bcu, bcv, bcw};
  const size_t nl = (size_t)dns->nz * dns->nline;
  for (int i = 0; i < dns->ncom; ++i)
    HIPCHK(hipMemcpyAsync(dns->bcu[i], src[i], nl * sizeof(double), hipMemcpyDeviceToDevice,
                          (hipStream_t)stream));
  return SEMX_OK;
}

int semx_dns_destroy(semx_dns dns) {
  if (!dns) return SEMX_E_ARG;
  dns_free(dns);
  return SEMX_OK;
}

int semx_dns_run(semx_dns dns, int nstep, double* u, double* v, double* w, double* p,
                 void* stream) {
  if (!dns || nstep < 0 || !u || !v || !p || (dns->ncom == 3 && !w)) return SEMX_E_ARG;
  semx_dns_s& D = *dns;
  hipStream_t s = (hipStream_t)stream;
  double* ext[3] = {u, v, w};
  const size_t bytes = D.ntot * sizeof(double);
  for (int i = 0; i < D.ncom; ++i)
    HIPCHK(hipMemcpyAsync(D.U[i], ext[i], bytes, hipMemcpyDeviceToDevice, s));
  HIPCHK(hipMemcpyAsync(D.P, p, bytes, hipMemcpyDeviceToDevice, s));
  const bool startup = D.step + 1 < D.nord;
  for (int k = 0; k < nstep; ++k) CHK(dns_step_graph(D, s));
  for (int i = 0; i < D.ncom; ++i)
    HIPCHK(hipMemcpyAsync(ext[i], D.U[i], bytes, hipMemcpyDeviceToDevice, s));
  HIPCHK(hipMemcpyAsync(p, D.P, bytes, hipMemcpyDeviceToDevice, s));
  // the solves of the steps ran without host synchronisation: any expired
  // wait between workgroups among them is reported here (every system is
  // checked, so that none keeps its mark for a later run)
  int st = SEMX_OK;
  for (Helm* h : {D.vel, D.pre, startup ? D.start[0] : nullptr, startup ? D.start[1] : nullptr})
    if (const int e = h ? helm_check(*h, s) : SEMX_OK) st = e;
  return st;
}

int semx_dns_info(semx_dns dns, int* info) {
  if (!dns || !info) return SEMX_E_ARG;
  info[0] = dns->step; info[1] = dns->nz; info[2] = dns->ncom; info[3] = dns->nord;
  return SEMX_OK;
}

int semx_dns_set_graph(semx_dns dns, int on) {
  if (!dns) return SEMX_E_ARG;
  dns->graphs_on = on != 0;
  return SEMX_OK;
}

int semx_dns_graph_info(semx_dns dns, int* ngraphs, long long* replays) {
  if (!dns || !ngraphs || !replays) return SEMX_E_ARG;
  *ngraphs = (int)dns->graphs.size();
  *replays = dns->replays;
  return SEMX_OK;
}

}  // extern "C"
