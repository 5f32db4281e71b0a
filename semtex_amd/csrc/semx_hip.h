// semx_hip.h -- HIP-side helpers shared by the kernel sources of libsemx:
// status-checked HIP calls, device uploads, and the launch timing registry
// behind semx_profile_*.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>

#include "semx_internal.h"

#define HIPCHK(x)                                                        \
  do {                                                                   \
    hipError_t e_ = (x);                                                 \
    if (e_ != hipSuccess) {                                              \
      fprintf(stderr, "semx: %s failed: %s\n", #x, hipGetErrorString(e_)); \
      return SEMX_E_HIP;                                                 \
    }                                                                    \
  } while (0)

namespace semx {

// HIP events around a launch on its stream, accumulated per kernel name
// while profiling is enabled (no-ops otherwise).
void prof_begin(hipStream_t s, hipEvent_t* a);
void prof_end(hipStream_t s, const char* name, hipEvent_t a);
void prof_flush();
bool prof_enabled();

template <class T>
inline int dev_upload(T** dptr, const T* src, size_t count) {
  *dptr = nullptr;
  const size_t alloc = count ? count : 1;
  HIPCHK(hipMalloc((void**)dptr, alloc * sizeof(T)));
  if (src && count) HIPCHK(hipMemcpy(*dptr, src, count * sizeof(T), hipMemcpyHostToDevice));
  else HIPCHK(hipMemset(*dptr, 0, alloc * sizeof(T)));
  return SEMX_OK;
}

template <class T>
inline void dev_free(T*& p) {
  if (p) (void)hipFree((void*)p);
  p = nullptr;
}

// Gives back scratch that a larger one replaces, or keeps it until the system
// is released where a solve has been captured: the graph goes on using it.
template <class T>
inline void retire(Helm& H, T*& p) {
  if (p && H.pcg_frozen) H.d.retired.push_back((void*)p);
  else if (p) (void)hipFree((void*)p);
  p = nullptr;
}

// Field::solve over all planes of one system (the body of semx_helm_solve).
int helm_solve(Helm& H, double* f, const double* bc, double* u, double tol_rel, int step_max,
               int* iters, hipStream_t s);
// The same for nf <= SEMX_MAX_FIELDS fields sharing the system, in the launches
// of one (the band sweeps, where they are selected, may take one per field).
int helm_solve_fields(Helm& H, int nf, double* const* fs, const double* const* bcs,
                      double* const* us, double tol_rel, int step_max, int* iters,
                      hipStream_t s);
// Element right-hand sides (condensed for the direct modes) into d.Fb and,
// for PCG planes, d.Fi; and the direct modes' element solutions from d.sol.
// pFb, pFi, psol: strides between fields.
int elem_condense(Helm& H, int nf, double* const* fs, const double* const* bcs, double* const* us,
                  size_t pFb, size_t pFi, size_t psol, hipStream_t s);
int elem_backsub(Helm& H, int nf, double* const* fs, const double* const* bcs, double* const* us,
                 size_t pFb, size_t pFi, size_t psol, hipStream_t s);
// The boundary systems of the direct modes through the elimination tree:
// condensed right-hand sides d.Fb (pFb doubles per field) to d.sol (psol).
int tree_solve(Helm& H, int nf, size_t pFb, size_t psol, hipStream_t s);
// Device address (current device) of the static scratch array of the
// allocation-free entry points; looked up once per device.
int noalloc_scratch(double** out);
// Waits for the stream, then reports (SEMX_E_TIMEOUT) and clears a
// cooperative band sweep's expired hand-off wait since the last check.
int helm_check(Helm& H, hipStream_t s);

}  // namespace semx


