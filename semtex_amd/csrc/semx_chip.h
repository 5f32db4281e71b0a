// semx_chip.h -- the on-chip Jacobi PCG (semx_pcg.hip): its tables and the
// interface the solve code (semx_solve.hip) uses.
#pragma once
#include <vector>

#include "semx_hip.h"

namespace semx {

// One workgroup's share of a mesh: elements [elo, elo + ne), the boundary
// results of other workgroups it adds (nrem of them) and its own that others
// add (npub).
struct ChipPart { int elo, ne, rem0, nrem, pub0, npub; };

// A mesh split over W workgroups, on the device.  LDS indices of boundary
// results: el * next + b of the workgroup's own elements, then the received
// ones.
struct ChipMesh {
  int np, npnp, next, nint, nel, nglobal, nsolve, nset, W, nif;
  const ChipPart* part;
  const ushort4* tab;      // per element-boundary slot: LDS indices of the results
                           // its node sums, in increasing slot order (0xFFFF: none)
  const int4* gsrc;        // the same as slots of the whole mesh (-1: none)
  const int* rem;          // exchange positions of the received results
  const int2* pub;         // own LDS index and exchange position of the sent ones
  const double* G;
  const int* eset;
  const int* btog;
  const double* aff;       // per set: Q1..Q4 over the product of GLL weights, where
                           // every element is a parallelogram; else null
  const double* wq;        // GLL weights
  const float* wqf;
  const double* ops;       // D D^T, SVV D D^T
  const float* opsf;
  const int* ess_src;      // batch: BC-line index of essential nodes
  const int* nat_ptr;      // batch: natural boundary sides per element
  const int* nat_b;
  const int* bside;
  const double* barea;
};

// One problem: a PCG plane of a system, or a problem of a batch.
struct ChipInst {
  const ChipMesh* mesh;
  const double* pc;
  const float* pc32;
  const double* mq;        // cylindrical mass factors of the mode, or null
  double* work;            // element-ordered scratch: nel * npnp doubles
  double hcon;
  int n, svv;
  int plane, pidx;         // field plane, plane-list index (planes)
  long long exch, red;     // this problem's exchange and partial-sum slots
};

struct ChipArgs {
  const ChipInst* inst;
  const int2* order;       // (problem, part) in the order workgroups take them
  unsigned* ticket;
  double* exch;            // 4 x nif slots per problem and field
  double* red;             // 4 x 3 x W slots per problem and field
  long long exchF, redF, workF;   // strides between fields
  int* iters;
  int* err;
  int count;               // problems per field
  int planeSize, nzero;
  double tol, inner_tol;
  int step_max, max_outer;
  bool no_wait;            // set by chip_launch
  // planes: condensed right-hand sides, essential values, solutions
  const double* Fb;
  const double* Fi;
  const double* g;
  long long FbF, FiF, gF;
  double* u[SEMX_MAX_FIELDS];
  // batch: pointer arrays (null for planes)
  const double* const* bf;
  const double* const* bbc;
  double* const* bu;
};

// Device tables of one mesh split over W workgroups.
struct ChipPlan {
  bool ok = false;
  int W = 0, nif = 0;
  size_t lds64 = 0;
  void* store = nullptr;   // every array below in one allocation
  ChipMesh m;
};

// The planes of a system.
struct ChipDev {
  ChipPlan plan;
  ChipInst* inst = nullptr;
  double* exch = nullptr;
  double* red = nullptr;
  unsigned* ticket = nullptr;
  int nf_cap = 0;                      // fields the slots hold
  const double* work = nullptr;        // the scratch inst points into
  std::vector<int> rank;               // planes in the order they are taken:
                                       // as listed, or by iteration counts
  int2* order[SEMX_MAX_FIELDS + 1] = {nullptr};
};

// Workgroups of a mesh's problem, 0 if the on-chip iteration does not take it.
int chip_workgroups(const Mesh& M);
// Builds the tables (M on the device); mesh descriptor included in `store`.
int chip_plan(Mesh& M, ChipPlan& P, const ChipMesh** dev);
void chip_release(ChipPlan& P);
// np: that of every problem, or 0 where they differ (a batch)
int chip_launch(const ChipArgs& a, int np, bool refine, int groups, size_t lds, long long nexch,
                long long nred, hipStream_t s);

}  // namespace semx
