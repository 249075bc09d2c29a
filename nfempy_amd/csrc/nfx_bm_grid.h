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
  bool planned = false;        // by the first solve, from the instances' row pointers
  char *dev = nullptr, *host = nullptr;  // one allocation each, only where the batch is resident
  std::vector<int> wave_of;    // launch of each instance; empty: the batch is not resident
  std::vector<int> wave_at;    // first block of each launch in blocks[], and the end
  std::vector<char> tail;      // per launch: its last block is one of several of an instance
  BmGridBlock* blocks = nullptr;
  int32_t* ranges = nullptr;   // kBmRanges per instance
  grid_word* slots = nullptr;
  GridResult* res = nullptr;   // per instance
  double* tol = nullptr;       // per instance
  float* own = nullptr;        // 3 vectors of all rows
  GridResult* h_res = nullptr; // pinned, per instance
  double* h_tol = nullptr;
  GridControl control;
};

// per preconditioner group: first, end and run count of cells and of flux blocks; then the aggregates
constexpr int kBmRanges = 13;

void bm_grid_destroy(BmGrid* g);

// The route of a whole solve, from all instances of the batch, whichever still iterate: resident or not.
// rows: of each instance; scratch: n_inst words on the device.
int bm_grid_route(BmGrid* g, const std::vector<int>& rows, int64_t n_total, const nfx_minres_batch_item* d_items,
                  const std::vector<nfx_batch_tg>& pc, int32_t* scratch, bool* resident, hipStream_t st);

// Inner solves of the instances with h_mode 0 on the resident route. done[i]: set where instance i was solved,
// with iters[i] and its rows of x. vec: 8 vectors of n_total floats.
int bm_grid_solve(BmGrid* g, int n_inst, int64_t n_total, const nfx_minres_batch_item* d_items, const int32_t* d_mode,
                  const int32_t* h_mode, const std::vector<nfx_batch_tg>& pc, const float* rhs, float* x, float* vec,
                  const double* tol, int maxit, int* iters, std::vector<char>* done, hipStream_t st);

}  // namespace nfx
