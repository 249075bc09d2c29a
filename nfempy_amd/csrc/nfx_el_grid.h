// MINRES of one dual-mixed elasticity system with its two-grid preconditioner as one cooperative launch
// (nfx_el_grid.hip).
#pragma once

#include "nfx_minres_grid.h"

namespace nfx {

// Blocks for a system (n_blocks 3 x 3 blocks of the operator), 0 if it does not fit.
int el_grid_blocks(int max_blocks, const nfx_elasticity_tg* pc, int n_blocks);
// 0 where the device does not allow it
int el_grid_capacity();

// One inner solve; vec: 8 vectors of n floats. *status as GridResult::status.
int el_grid_solve(MinresGrid* g, int nblk, int n, int n_blocks, const int32_t* brp, const int32_t* bci,
                  const float* bva, const nfx_elasticity_tg* pc, const float* rhs, float* x, float* vec, double tol,
                  int maxit, int* iters, int* status, hipStream_t st);

}  // namespace nfx
