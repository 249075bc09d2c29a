// Batched MINRES with the instances resident in the CUs (nfx_bm_grid.hip).
#pragma once

#include <vector>

#include "nfx_grid.h"
#include "nfx_minres.h"

namespace nfx {

// a block of a launch: its instance, its place among the instance's blocks, the first of them
struct BmGridBlock {
  int inst, rank, nblk, first;
};

// Launch plan and work space of a batch. An instance's block count follows from its own size, so its
// sums, and its result, are the same in every batch that is resident; a stepwise batch has other roundings.
struct BmGrid {
  char *dev = nullptr, *host = nullptr;  // one allocation each
  int cap = 0;                 // blocks of a launch
  std::vector<int> wave_of;    // launch of each instance, -1: not resident
  std::vector<int> wave_at;    // first block of each launch in blocks[], and the end
  std::vector<char> tail;      // per launch: its last block is one of several of an instance
  BmGridBlock* blocks = nullptr;
  int32_t* ranges = nullptr;   // kBmRanges per instance
  grid_word* slots = nullptr;
  GridResult* res = nullptr;   // per instance
  double* tol = nullptr;       // per instance
  GridResult* h_res = nullptr; // pinned, per instance
  double* h_tol = nullptr;
  GridControl control;
};

// per preconditioner group: first, end and run count of cells and of flux blocks; then the aggregates
constexpr int kBmRanges = 13;

// Plans the launches and allocates (nothing resident when the device or the sizes do not allow it).
int bm_grid_create(BmGrid* g, int n_inst, const nfx_minres_batch_item* items, const nfx_minres_batch_item* d_items,
                   hipStream_t st);
void bm_grid_destroy(BmGrid* g);

// The route of a whole solve, from all instances of the batch, whichever still iterate: resident or not.
int bm_grid_route(BmGrid* g, int n_inst, int64_t n_total, const std::vector<nfx_batch_tg>& pc, bool* resident,
                  hipStream_t st);

// Inner solves of the instances with h_mode 0 on the resident route. done[i]: set where instance i was solved,
// with iters[i] and its rows of x. vec: 8 vectors of n_total floats, own: 3 more.
int bm_grid_solve(BmGrid* g, int n_inst, int64_t n_total, const nfx_minres_batch_item* d_items, const int32_t* d_mode,
                  const int32_t* h_mode, const std::vector<nfx_batch_tg>& pc, const float* rhs, float* x, float* vec,
                  float* own, const double* tol, int maxit, int* iters, std::vector<char>* done, hipStream_t st);

}  // namespace nfx
