// Preconditioned FP32 MINRES of one system as one cooperative launch (nfx_minres_grid.hip).
#pragma once

#include "nfx_grid.h"
#include "nfx_minres.h"

namespace nfx {

// work space of a solver: the slots and the result
struct MinresGrid {
  int max_blocks = 0;  // 0: not available on this device
  grid_word* slots = nullptr;
  GridResult* res = nullptr;
  GridResult* h_res = nullptr;  // pinned
  int* h_other = nullptr;       // pinned, kGridDiagBlocks
  GridControl control;
};

int minres_grid_capacity();

// Blocks for a system of n rows and nnz entries, 0 if it does not fit the blocks' LDS.
int minres_grid_blocks(const MinresGrid* g, int n, int64_t nnz);

// Whether the rows of a CSR preconditioner are one diagonal entry each, in three steps: minres_grid_ask queues
// the look, the caller waits for the stream, minres_grid_diagonal reads the answer.
constexpr int kGridDiagBlocks = 256;
int minres_grid_ask(MinresGrid* g, int n, const int32_t* prp, const int32_t* pci, hipStream_t st);
bool minres_grid_diagonal(const MinresGrid* g);

// One inner solve with a diagonal preconditioner (CSR arrays as nfx_solve_minres_ir has them);
// z: 2 n floats. *status as GridResult::status; *iters and x are set when it is 0.
int minres_grid_solve(MinresGrid* g, int nblk, int lanes, int n, const int32_t* rp, const int32_t* ci, const float* va,
                      const float* sign, const int32_t* prp, const int32_t* pci, const float* pva, const float* rhs,
                      float* x, float* z, double tol, int maxit, int* iters, int* status, hipStream_t st);

}  // namespace nfx
