// Resident CG (fem_resident.hip): one launch runs a whole solve, or the recurrence between two
// hand-overs, with the operator's rows, the vectors and the scalars on chip.
#pragma once
#include "fem_internal.h"

namespace fem {

// Where the rows of the scaled operator Â come from.  src 0: the columns of K's CSC arrays
// (= rows, K is symmetric) scaled by sc; 1: lattice value planes; 2: the cell form (one
// coefficient per cell, masked scaling t, class values f).  1 and 2 number the rows by the
// padded lattice (dofp: the dof of a padded row, −1 on padding).
struct ResSource {
  int src = 0;
  int64_t n = 0;                 // rows: dofs (0) or padded lattice rows (1, 2)
  int widest = 0;                // most entries of a column of K
  int dim = 0;                   // lattice dimension; 0 with `node`: of the coordinates
  const int32_t* node = nullptr;           // 0: a node of each row and the nodes' coordinates, or null:
  const double* x[3] = {};                 //    those of the context's mesh
  int nsys = 0;                            // independent systems, their row ranges sys[2 i], sys[2 i + 1];
  const int32_t* sys = nullptr;            //    0: all rows are one
  int32_t px = 0, pxy = 0;
  int64_t npad = 0;
  const int32_t *dofp = nullptr, *map = nullptr;   // map: the padded row of a dof
  const void* val = nullptr;     // 1: planes [s][npad]
  const double* kc = nullptr;    // 2: k_c at the padded row of each cell's first corner
  const void* t = nullptr;       // 2: masked scaling (X precision; 0 on prescribed rows and padding)
  double f[8] = {};              // 2: K¹ per corner-offset class
};

struct ResOp;

// Device memory of a one-launch solve.  It is optional: without it the separate kernels solve, so
// what prepares one answers "does not fit" (no_memory) instead of failing.
template <class T>
int copy_alloc(fem_ctx* c, T** p, size_t n) {
  if (c->copy_limit >= 0 && n * sizeof(T) > (size_t)c->copy_limit)
    return set_error(c, FEM_ERR_OOM, "over the limit of fem_set_copy_limit");
  return dev_alloc(c, p, n);
}
inline bool no_memory(fem_ctx* c, int rc) {
  if (rc != FEM_ERR_OOM) return false;
  (void)hipGetLastError();       // (of the hipMalloc)
  c->err.clear();
  return true;
}

// What the launch did for one system.
struct ResState {
  double rr;                     // square of the true residual of u
  int iters, handovers;
  int status;                    // 1: rr <= tol2
  int lost;                      // 1: a block gave up waiting for another one
  int prods;                     // products with Â run
  uint32_t epoch;                // exchange numbers used up to here
  long long ticks, begin, end;   // 100 MHz clock: in the largest part's products (time), the system's first and last
};

// Fewest blocks that hold a system of several in a launch (0: its rows have too many entries), and
// the blocks of a launch.
int resident_blocks(int64_t rows, int widest, bool fp32);
int resident_most_blocks(const fem_ctx* c);

// Ready to run on `s` in FP32 or FP64 (structure once per pattern, values when K or the scaling
// changed); *ok = false when the rows do not fit, or memory for them is not to be had (the caller keeps
// the separate kernels).
int resident_prepare(fem_ctx* c, ResOp** op, const ResSource& s, const double* sc, int jacobi, bool fp32, bool* ok);

// The whole solve K u = f from u = 0: the recurrence and its hand-overs (u, the FP64 residual, the
// reseed) until the true residual meets the tolerance, stalls, or `lim` steps are done.  in:
// per system the squares of |f| and of the tolerance in device memory, or null (one system):
// bnorm2, tol2.  Returns when it is done; *out: what it did per system, until the next run.
// *launched = false: the device did not take the launch.
template <typename X>
int resident_run(fem_ctx* c, ResOp* op, const ResSource& s, const double* sc, const double* f, double* u,
                 const double* in, double bnorm2, double tol2, double hold_factor2, int lim, const ResState** out,
                 bool* launched);

void resident_free(ResOp** op);

// The same on the 3D cell form in FP32, for lattices too large for the rows' entries
// (fem_resident_cells.hip).
struct BrickSource {
  int32_t px = 0, pxy = 0;
  const float *t = nullptr, *kc = nullptr;   // masked scaling and coefficients on the padded rows
  const int32_t* dofp = nullptr;
  double f[8] = {};
};
struct BrickOp;
int brick_prepare(fem_ctx* c, BrickOp** op, int nx, int ny, int nz, bool* ok);
int brick_run(fem_ctx* c, BrickOp* op, const BrickSource& s, const double* res, const double* sc, float* p, float* sv,
              double* u, Scal* scal, double hold_factor2, double tol2, int restart, int lim, bool* launched);
void brick_free(BrickOp** op);

// The same on the stored Q2 hex³ element matrices (fem_resident_elems.hip), in FP32 or FP64; the
// matrices of the current K are read by elems_prepare.
struct ElemsOp;
int elems_prepare(fem_ctx* c, ElemsOp** op, const double* sc, bool fp32, bool* ok);
template <typename X>
int elems_run(fem_ctx* c, ElemsOp* op, const double* res, const double* sc, X* p, X* sv, double* u, Scal* scal,
              double hold_factor2, double tol2, int restart, int lim, bool* launched);
void elems_free(ElemsOp** op);

}  // namespace fem
