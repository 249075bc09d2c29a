// Device-wide sums and vector exchange between the blocks of one cooperative launch.
//
// A Krylov iteration on a system of 1e3..1e5 rows is a handful of sums and short products; as launches
// each costs 4-10 us whatever its work. A cooperative kernel keeps the blocks resident for the whole
// solve, the operator and the vectors in LDS, and pays only for the exchange between blocks:
//  * a sum: every block writes its partial into its slot (eight copies, so that readers spread over
//    memory channels) and polls all slots of one copy. A slot is two 64-bit words, each half a double
//    and the step's tag, so a reader needs no counter, no ordering between the words and no fence, and
//    every block adds the same numbers in the same order;
//  * a vector: stored and loaded with relaxed device-scope accesses (they pass the caches that are not
//    coherent between XCDs); a block waits for its stores before it posts the next sum.
// Device-scope fences instead of these accesses cost 5-30 us per step (measured, 8-256 blocks).
//
// That is no release / acquire pair of the language: the accesses are relaxed, and a thread's vector stores come
// before its block's post only by what this GPU does with them. Relied on, in what hipcc makes of them for gfx950
// (global_store / global_load with sc1, no cache write-back or invalidate): a device-scope store is written
// through the XCD's L2, and counts in vmcnt until it is where every XCD's device-scope load finds it; such a load
// does not return an older line of its own L2; and a load is not issued before the barrier that ends the wait
// for the post. A wait for vmcnt(0) in every wave and a barrier stand between the stores and the post. Vectors
// that other blocks read go through grid_store and grid_load only; plain accesses are to a block's own rows.
// Two slot sets alternate: a block posts step k + 2 only after every block has read step k.
//
// Every wait is bounded (kGridWaitTicks): a block that gives up leaves, the others then give up in
// their turn, the launch ends and the caller takes its general path.
#pragma once

#include "nfx_common.h"

namespace nfx {

// 1,024 against 512 threads, us an iteration of MINRES: 4.5 / 4.5 at 5,184 rows (30 k entries), 7.7 / 9.9 at
// 41,088 rows (1.06 M entries) and 8.7 / 11.3 at 252,288 rows (1.9 M): more rows in flight beside the waits
constexpr int kGridThreads = 1024;

// A device gives the resources of cooperative launches to one process at a time; a launch in another is
// refused, after ~35 ms. The callers then take the stepwise kernels, and for kGridRetrySeconds they do not
// ask that device again (nfx_backoff.h); nor after a launch whose blocks gave up waiting for each other.
constexpr int kGridRetrySeconds = 10;

// what a launch (or one system of it) reports
struct GridResult {
  int iters;
  int status;  // 0 solved or out of iterations, 1 not applicable (nothing was done), 2 a wait was given up
};

// What a solver object allows, and has seen, of resident launches.
struct GridControl {
  int64_t launches = -1;               // still allowed (-1: any number)
  int absent = 0;                      // != 0: the last block is not launched, the others give up their wait for it
  int64_t solved = 0, declined = 0;    // inner solves that ran so; that were tried so and ran stepwise
};
bool grid_allowed(const GridControl& c);  // a launch on the current device, now
// Launches kernel on nblk blocks of kGridThreads with all their LDS. *ran = false: not launched (refused, no
// resources, or no more allowed) and nothing ran, the stepwise kernels take it. Any other failure is an error.
int grid_launch(GridControl* c, const void* kernel, int nblk, void** args, hipStream_t st, bool* ran);
// Counts an inner solve (of an instance) by the status that its launch left, and pauses the device after 2.
void grid_count(GridControl* c, int status);
constexpr int kGridCheck = 16;  // iterations between tests of the estimate, as in the stepwise solvers
constexpr int kGridMaxBlocks = 256;
constexpr int kGridCopies = 8;
constexpr int kGridBlockWords = 2 * kGridCopies * 2;  // 64-bit words of slots per block
constexpr int64_t kGridSlotWords = (int64_t)kGridBlockWords * kGridMaxBlocks;
constexpr long long kGridWaitTicks = 50000000;  // 0.5 s of the 100 MHz clock
constexpr int kGridLdsBytes = 158 * 1024;       // dynamic LDS of a block: all of a CU but the static arrays

using grid_word = unsigned long long;

template <typename T>
__device__ __forceinline__ void grid_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T grid_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sums by cross-lane moves in the vector unit (a shuffle through the LDS unit takes ~50 ns a step, and
// these steps are on the path of every iteration).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
  return __hiloint2double(hi, lo);
}

// sum over the 64 lanes (all active), the same in every lane
__device__ __forceinline__ double wave_total(double v) {
  v += dpp_move<0x111, 0xf>(v);  // lane - 1, - 2, - 4, - 8 of the row of 16: its last lane has its sum
  v += dpp_move<0x112, 0xf>(v);
  v += dpp_move<0x114, 0xf>(v);
  v += dpp_move<0x118, 0xf>(v);
  v += dpp_move<0x142, 0xa>(v);  // last lane of rows 0, 2 into rows 1, 3
  v += dpp_move<0x143, 0xc>(v);  // last lane of row 1 into rows 2, 3
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// sum over groups of LANES (4, 8, 16) consecutive lanes, in every lane of the group
template <int LANES>
__device__ __forceinline__ float lanes_total(float v) {
  v += dpp_move<0xb1>(v);  // neighbour, then neighbour pair
  v += dpp_move<0x4e>(v);
  if (LANES >= 8) v += dpp_move<0x141>(v);   // mirrored in 8: the other four
  if (LANES >= 16) v += dpp_move<0x140>(v);  // mirrored in 16: the other eight
  return v;
}

// Clears the slots of a launch of nblk blocks, and n_res results.
int grid_clear(grid_word* slots, int nblk, GridResult* res, int n_res, hipStream_t st);

struct GridSync {
  grid_word* slots;   // kGridBlockWords a block, zero before the launch
  int nblk, rank;     // blocks that take part (at most kGridMaxBlocks and the threads of a block)
  unsigned tag;       // steps posted so far
  double (*post)[kGridThreads / 64];  // LDS, [2]
  double (*part)[kGridThreads / 64];  // LDS, [2]
  int (*good)[kGridThreads / 64];     // LDS, [2]
};

__device__ __forceinline__ grid_word* grid_slot(const GridSync& g, int copy, int b) {
  return g.slots + (((int64_t)(g.tag & 1) * kGridCopies + copy) * g.nblk + b) * 2;
}

// Adds the block's v (in wave order) and posts it. Contains a barrier; every exchange store that a
// thread made before is complete when the post can be seen.
__device__ __forceinline__ void grid_post(GridSync& g, double v) {
  v = wave_total(v);
  ++g.tag;
  double* sh = g.post[g.tag & 1];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x < kGridCopies) {
    double r = 0;
#pragma unroll
    for (int w = 0; w < kGridThreads / 64; ++w) r += sh[w];
    const grid_word bits = (grid_word)__double_as_longlong(r);
    grid_word* p = grid_slot(g, threadIdx.x, g.rank);
    grid_store(p, (bits & 0xffffffff00000000ull) | g.tag);
    grid_store(p + 1, (bits << 32) | g.tag);
  }
}

// The sum of the last post over all blocks, the same in every thread. False: some wait was given up.
// Contains a barrier.
__device__ __forceinline__ bool grid_wait(GridSync& g, double& sum) {
  const int waves = (g.nblk + 63) >> 6, wave = threadIdx.x >> 6;
  if (wave < waves) {
    double v = 0;
    bool ok = true;
    if ((int)threadIdx.x < g.nblk) {
      const grid_word* p = grid_slot(g, g.rank % kGridCopies, threadIdx.x);
      long long t0 = 0;
      grid_word hi, lo;
      for (int spin = 1;; ++spin) {
        hi = grid_load(p);
        lo = grid_load(p + 1);
        if ((unsigned)hi == g.tag && (unsigned)lo == g.tag) break;
        if ((spin & 63) == 0) {
          const long long now = wall_clock64();
          if (t0 == 0) t0 = now;
          if (now - t0 > kGridWaitTicks) {
            ok = false;
            break;
          }
        }
      }
      v = __longlong_as_double((long long)((hi & 0xffffffff00000000ull) | (lo >> 32)));
    }
    v = wave_total(v);
    ok = __all(ok);
    if ((threadIdx.x & 63) == 0) {
      g.part[g.tag & 1][wave] = v;
      g.good[g.tag & 1][wave] = ok;
    }
  }
  __syncthreads();
  bool ok = true;
  sum = 0;
  for (int w = 0; w < waves; ++w) {
    sum += g.part[g.tag & 1][w];
    ok = ok && g.good[g.tag & 1][w];
  }
  return ok;
}

// a value that all threads share, in a scalar register
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The columns that a block's rows meet, as a list, and the rows' columns as 16-bit places in it.
// Row i has entries start(i) .. start(i) + rowp[i + 1] - rowp[i] of ci; n columns in all.
// bits, before: (n + 31) / 32 words each. grid_columns counts them (barriers inside; the count is the
// same in every thread), grid_renumber writes list and idx.
template <int LANES, typename Start>
__device__ __forceinline__ int grid_columns(const int32_t* __restrict__ ci, int n, int R, const int* rowp, Start start,
                                            unsigned* bits, int* before, int* scan) {
  constexpr int T = kGridThreads;
  const int t = threadIdx.x, nw = (n + 31) >> 5;
  for (int w = t; w < nw; w += T) bits[w] = 0;
  __syncthreads();
  for (int i = t / LANES; i < R; i += T / LANES) {
    const int32_t* c = ci + start(i);
    for (int j = t % LANES, len = rowp[i + 1] - rowp[i]; j < len; j += LANES)
      atomicOr(&bits[c[j] >> 5], 1u << (c[j] & 31));
  }
  __syncthreads();
  // exclusive prefix of the bit counts: a run of words per thread, then waves, then the block
  const int run = (nw + T - 1) / T, w0 = min(nw, t * run), w1 = min(nw, w0 + run);
  int cnt = 0;
  for (int w = w0; w < w1; ++w) cnt += __popc(bits[w]);
  int inc = cnt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(inc, off, 64);
    if ((t & 63) >= off) inc += o;
  }
  if ((t & 63) == 63) scan[t >> 6] = inc;
  __syncthreads();
  int pre = inc - cnt, total = 0;
  for (int w = 0; w < T / 64; ++w) {
    if (w < (t >> 6)) pre += scan[w];
    total += scan[w];
  }
  for (int w = w0; w < w1; ++w) {
    before[w] = pre;
    pre += __popc(bits[w]);
  }
  __syncthreads();
  return total;
}

template <int LANES, typename Start>
__device__ __forceinline__ void grid_renumber(const int32_t* __restrict__ ci, int n, int R, const int* rowp,
                                              Start start, const unsigned* bits, const int* before, int* list,
                                              unsigned short* idx) {
  constexpr int T = kGridThreads;
  const int t = threadIdx.x, nw = (n + 31) >> 5;
  for (int w = t; w < nw; w += T) {
    int p = before[w];
    for (unsigned b = bits[w]; b; b &= b - 1) list[p++] = 32 * w + __ffs(b) - 1;
  }
  for (int i = t / LANES; i < R; i += T / LANES) {
    const int32_t* c = ci + start(i);
    for (int j = t % LANES, len = rowp[i + 1] - rowp[i]; j < len; j += LANES)
      idx[rowp[i] + j] = (unsigned short)(before[c[j] >> 5] + __popc(bits[c[j] >> 5] & ((1u << (c[j] & 31)) - 1)));
  }
  __syncthreads();
}

}  // namespace nfx
