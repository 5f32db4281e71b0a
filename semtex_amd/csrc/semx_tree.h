// semx_tree.h -- elimination tree of the condensed boundary systems: the
// elements are merged level by level into larger and larger regions, and
// the boundary unknowns a merge makes interior are eliminated there, with
// dense matrices per region (static condensation continued above the
// element).  The direct solve is then a forward pass (each region reduces
// its right-hand side to its boundary), and a backward pass (each region
// recovers its eliminated unknowns from its boundary values).
#pragma once

#include <memory>
#include <vector>

namespace semx {

struct Helm;

// Doubles that a resize leaves as they are: large matrices are written whole,
// by the threads that compute them, and would only be touched twice.
template <class T>
struct NoInit : std::allocator<T> {
  template <class U> struct rebind { typedef NoInit<U> other; };
  template <class U> void construct(U*) noexcept {}
  template <class U, class V> void construct(U* p, const V& v) { *p = v; }
};
typedef std::vector<double, NoInit<double>> RawDoubles;

// A region type: regions built the same way from the same child types
// share their matrices (translated copies on uniform meshes).
struct TreeType {
  int stage = 0;
  int ni = 0, nb = 0;            // eliminated unknowns, boundary unknowns
  int pin = -1;                  // eliminated unknown that a singular mode pins
  std::vector<int> child;        // child types; -1-l: leaf (element) type l
  std::vector<char> merge;       // how the bisection merges them: 0 the next child,
                                 // 1 the last two parts
  std::vector<int> cptr, cmap;   // child's boundary entry -> unknown (0..ni+nb)
  long long off_f = 0, off_b = 0;  // packed matrices within a mode's block
};

struct TreeLeaf {                // an element's condensed matrix on its solved nodes
  int set = 0;
  std::vector<int> loc;          // element-boundary positions (emap order)
};

// Regions in stage order, those of one type next to each other.
struct TreeNode {
  int type = 0;
  int uptr = 0;                  // first of its ni + nb unknowns in gid / rowptr
  int cslot = 0, yslot = 0;      // its boundary contributions, its kept unknowns
};

struct Tree {
  bool on = false;
  int nstage = 0, nslot_c = 0, nslot_y = 0;
  std::vector<TreeType> type;
  std::vector<TreeLeaf> leaf;
  std::vector<TreeNode> node;
  std::vector<int> stage_ptr;    // nodes of each stage
  std::vector<int> gid;          // global node of each region unknown
  std::vector<int> rowptr, src;  // contributions to each: element-boundary slots
                                 // [0, nel*next), then child slots from there on
  long long mstride = 0;         // doubles per direct mode
  RawDoubles mat;                // direct modes' packed matrices, released on upload
};

// A matrix (rows x cols) in the order the matrix cores take it: 16-row
// tiles by 8-column steps, each 64 lanes x 2 doubles, lane l holding rows
// l%16 and columns l/16 and 4 + l/16 of the step.
inline int tree_mt(int rows) { return (rows + 15) / 16; }
inline int tree_kp(int cols) { return (cols + 7) / 8; }
inline long long tree_packed(int rows, int cols) {
  return (long long)tree_mt(rows) * tree_kp(cols) * 128;
}

// Column capacity of a workgroup's right-hand-side tile in LDS, and the
// regions of one type that one workgroup takes together.
constexpr int TREE_LDS = 128 * 1024;
constexpr int TREE_GROUP = 8;

// Chooses the merges and lays the tree out (structure only); leaves T.on
// false where the band sweeps are to be used.
void tree_plan(Helm& H);
// Factorises every direct mode along the tree; SEMX_E_NOT_SPD as the
// banded Cholesky reports it.
int tree_factor(Helm& H);

}  // namespace semx
