// The multigrid bottom solve as one workgroup on the device: relax from zero (optional),
// then BiCGStabSolver::solve (BiCGStabSolver.H:199-519) in FP64 on the deepest level, with
// the reference's operations and reduction orders (kernel and layout notes in bottom.hip).
#pragma once
#include <functional>
#include <vector>

#include "device.hpp"

namespace amrmg {

// per problem and depth: the operator's coefficients and face rules
struct BatchCoef {
  double dxinv, lambda, alpha, beta, dx;
  int lap;          // 1: GSRBLAPLACIAN / OPERATORLAP forms (alpha == 0 and beta == 1)
  int kind[3][2];   // face rule: 0 Neumann, 1 Dirichlet, 3 periodic (bottom solves only)
  double val[3][2]; // face values (outer residual only; every other use is homogeneous)
};

// BiCGStabSolver's parameters and what the launch does before the Krylov solve
struct BottomParams {
  int imax;
  double reps, hang, small;
  int numRestarts;
  int nbottom;                 // relax iterations before the Krylov solve
  int relaxFirst;              // 1: zero the correction and relax nbottom times first (the
                               // whole bottom of MultiGrid::cycle); 0: start from the correction
};

// One box's terms in the reduction stages: nx values per row, `rows` rows (component, z,
// y), rp rows per stage, at `off` in each stage; col0: its first norm chain
struct BottomBox {
  int off, nx, rows, rp, col0;
};
// Device plan of one level.  A slot is an x-adjacent pair of cells (i = 2a, 2a + 1) of one
// row, one cell of each colour; slots are numbered a fastest, then j, k, component.  Tables
// and vectors list them in another order: nint slots whose neighbours are all inside the
// level (a multiple of 64, the last filled up with empty entries), then the others.
struct BottomPlan {
  int nslot = 0;                       // slots of all components (0: no plan)
  int nint = 0, nlist = 0;             // entries of the first kind / of both
  int ncell = 0;                       // cells of one component
  int nxh = 0, plane = 0;              // slots per row / per plane
  int wrap[3] = {0, 0, 0};             // slot distance between the two ends of a direction
  int two = 0;                         // 1: both colours have an LDS buffer of their own
  int nbox = 0, ncol = 0, nst = 1, stage = 0;  // boxes, box columns, stages and doubles per stage
  int mainDoubles = 0, sumDoubles = 0; // LDS: stencil / stage region, sums region
  const unsigned* word = nullptr;      // per entry: see kGeo* in bottom.hip
  const int2* cell = nullptr;          // per entry: field offsets of its (red, black) cell, -1 absent
  const int2* term = nullptr;          // per entry: reduction positions of its (red, black) cell
  const BottomBox* box = nullptr;
  const int2* col = nullptr;           // per norm chain: (box, column)
  long long base = 0;                  // added to the field offsets
  long long vec = 0;                   // first of its vectors (vectors() of them), in (red, black) pairs
};

// Host tables of a plan and their device copy
constexpr int kBottomMaxSlots = 16384;
constexpr int kBottomVectors = 9;
struct BottomTables {
  BottomPlan plan;                     // device pointers filled by upload
  std::vector<unsigned> word;
  std::vector<int2> cell, term, col;
  std::vector<BottomBox> box;
  // (red, black) pairs of vectors the plan needs
  long long pairs() const { return (long long)plan.nlist * (kBottomVectors + (plan.two ? 0 : 1)); }
  // false when the level does not qualify: more than kBottomMaxSlots slots, a periodic
  // direction of odd extent, or tables that do not fit LDS (the caller then solves another
  // way).  boxes: the level's boxes in layout order, tiling `rect`; offset(b, i, j, k): a
  // cell's offset in a field (below 2^31), components cs apart.
  bool build(const std::vector<Box>& boxes, const Box& rect, const int kind[3][2], int nc, long long cs,
             const std::function<long long(int, int, int, int)>& offset);
  size_t ldsBytes() const { return 8 * (size_t)(plan.mainDoubles + plan.sumDoubles); }
  // the tables of several plans in one device allocation (the caller's to free; its size is
  // added to *bytes); plans without slots are left as they are
  static void* upload(Context* ctx, const std::vector<BottomTables*>& all, long long* bytes);
};


template <class T>
struct BottomLaunch {
  const BottomPlan* plans = nullptr;   // per problem (one entry for a single level)
  const BatchCoef* coef = nullptr;     // per problem; null: cf
  BatchCoef cf{};
  T* const* corr = nullptr;            // per problem; null: corr1 / res1
  const T* const* res = nullptr;
  T* corr1 = nullptr;
  const T* res1 = nullptr;
  double* vecs = nullptr;              // Krylov vectors
  const double* metric = nullptr;      // per problem {convergence metric, eps}; null: metric1 / eps1
  double metric1 = 0, eps1 = 0;
  const int* active = nullptr;         // per problem; null: all
  int* stats = nullptr;                // per problem: BiCGStab iterations, added to
  BottomParams par{};
};
// one workgroup per problem; maxSlots, ldsBytes: the largest plan's slots and LDS; tree: the
// fixed pairwise reduction order in place of the reference's
template <class T>
void launch_bottom(Context* ctx, const BottomLaunch<T>& a, int nprob, int maxSlots, size_t ldsBytes, bool tree);

}  // namespace amrmg
