// FP32 MINRES with a diagonal preconditioner, one cooperative launch per inner solve.
//
// Block b owns a contiguous range of rows (cut so that 6 bytes an entry and 40 a row are even). It
// keeps its rows of D A in LDS (values, and columns renumbered to 16 bits into the list of columns
// that the block meets), and its pieces of the seven vectors. Iteration k:
//   load z at the block's columns | scalars of k | y = s D A z - ratio r1, post alpha
//   | w/x update of k - 1 | wait alpha | y' = y - (alpha/beta) r2, z = P^-1 y', store z, post y'.z | wait
// so it is bound by two exchanges between blocks (~2.2 us each at 64 blocks) and the LDS gathers.
// An iteration took 10.1 us as two launches and 4.5 us here at 5,184 rows (triangles, degree 1), 14.0
// and 7.7 at 41,088 rows (tetrahedra, degree 2), 18.7 and 8.7 at 252,288 rows (tetrahedra, degree 1).
#include <algorithm>
#include <chrono>
#include <cstdint>

#include "nfx_backoff.h"
#include "nfx_minres_grid.h"

namespace nfx {

struct MinresGridArgs {
  int n, nblk, maxit, lds;
  const int32_t *rp, *ci;
  const float *va, *sign;
  const int32_t *prp, *pci;
  const float *pva, *rhs;
  float *x, *z;
  double tol;
  grid_word* slots;
  GridResult* res;
};

__global__ __launch_bounds__(256) void k_grid_clear(int64_t words, grid_word* slots, int n_res, GridResult* res) {
  const int64_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < words) slots[i] = 0;
  if (i < n_res) res[i] = GridResult{0, 0};
}

// first row whose weight (6 bytes an entry, 40 a row) reaches b / nblk of the whole
__device__ __forceinline__ int grid_bound(int n, const int32_t* __restrict__ rp, int b, int nblk) {
  if (b >= nblk) return n;
  const int64_t want = (6 * (int64_t)rp[n] + 40 * (int64_t)n) * b / nblk;
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (6 * (int64_t)rp[mid] + 40 * (int64_t)mid < want)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

template <int LANES>
__global__ __launch_bounds__(kGridThreads) void k_minres_grid(MinresGridArgs a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ double sh_post[2][kGridThreads / 64], sh_part[2][kGridThreads / 64];
  __shared__ int sh_good[2][kGridThreads / 64];
  __shared__ int sh_scan[kGridThreads / 64], sh_row[2];
  constexpr int T = kGridThreads;
  const int t = threadIdx.x, n = a.n;
  GridSync g{a.slots, a.nblk, (int)blockIdx.x, 0, sh_post, sh_part, sh_good};

  if (t < 2) sh_row[t] = grid_bound(n, a.rp, blockIdx.x + t, a.nblk);
  __syncthreads();
  const int r0 = sh_row[0], R = sh_row[1] - r0;
  const int e0 = a.rp[r0], nz = a.rp[r0 + R] - e0;

  // LDS: values | row starts | columns (16 bits) | vectors | z at the columns | ... | column list.
  // While the columns are renumbered the space from the vectors on holds a bit per column of the
  // system and the count of set bits before each word.
  float* val = reinterpret_cast<float*>(lds);
  int* rowp = reinterpret_cast<int*>(val + nz);
  unsigned short* idx = reinterpret_cast<unsigned short*>(rowp + R + 1);
  const int64_t base = 4 * (int64_t)nz + 4 * (int64_t)(R + 1) + 4 * (int64_t)((nz + 1) / 2);
  const int nw = (n + 31) >> 5;
  bool fits = base + 8 * (int64_t)nw <= a.lds;
  bool diag = true;  // known to the host (k_grid_diagonal); pva is indexed by it
  for (int i = t; i < R; i += T) {
    const int j = a.prp[r0 + i];
    diag = diag && a.prp[r0 + i + 1] == j + 1 && a.pci[j] == r0 + i;
  }
  fits = __syncthreads_and(fits && diag);
  int H = 0;
  int* list = nullptr;
  float* vec = reinterpret_cast<float*>(lds + base);
  if (fits) {
    unsigned* bits = reinterpret_cast<unsigned*>(lds + base);
    int* before = reinterpret_cast<int*>(bits + nw);
    for (int i = t; i <= R; i += T) rowp[i] = a.rp[r0 + i] - e0;
    __syncthreads();
    const auto start = [&](int i) { return e0 + rowp[i]; };
    H = grid_columns<LANES>(a.ci, n, R, rowp, start, bits, before, sh_scan);
    // room for the list above the bits, and for vectors + z below it
    fits = H <= 65535 && base + 8 * (int64_t)nw + 4 * (int64_t)H <= a.lds &&
           base + 4 * (9 * (int64_t)R + 2 * (int64_t)H) <= a.lds;
    if (fits) {
      list = reinterpret_cast<int*>(lds + a.lds) - H;
      grid_renumber<LANES>(a.ci, n, R, rowp, start, bits, before, list, idx);
      const int lane = t % LANES;
      for (int i = t / LANES; i < R; i += T / LANES) {
        const float sg = a.sign ? a.sign[r0 + i] : 1.f;
        for (int j = rowp[i] + lane, j1 = rowp[i + 1]; j < j1; j += LANES) val[j] = sg * a.va[e0 + j];
      }
    }
  }
  double sum;
  grid_post(g, t == 0 && !fits ? 1.0 : 0.0);
  bool ok = grid_wait(g, sum);
  if (!ok || sum != 0) {
    if (t == 0) atomicMax(&a.res->status, ok ? 1 : 2);
    return;
  }

  float *r1 = vec, *r2 = r1 + R, *zc = r2 + R, *zp = zc + R, *wa = zp + R, *wb = wa + R, *xv = wb + R, *pin = xv + R,
        *ys = pin + R, *zh = ys + R;
  MinresState st{};
  double acc = 0;
  for (int i = t; i < R; i += T) {
    const float b = a.rhs[r0 + i], p = a.pva[a.prp[r0 + i]], z = p * b;
    r1[i] = r2[i] = b;
    pin[i] = p;
    zc[i] = z;
    zp[i] = wa[i] = wb[i] = xv[i] = 0.f;
    grid_store(a.z + n + r0 + i, z);
    acc += (double)b * (double)z;
  }
  grid_post(g, acc);
  ok = grid_wait(g, sum);

  int k = 1;
  bool last = false;  // only the update of iteration k - 1 is left
  for (; ok; ++k) {
    const float* zg = a.z + (int64_t)(k & 1) * n;
    float* zn = a.z + (int64_t)((k + 1) & 1) * n;
    // z of iteration k at the block's columns, the scalars beside the loads
    constexpr int kPre = 4;
    float zl[kPre];
    if (!last) {
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * T < H) zl[u] = grid_load(zg + list[t + u * T]);
    }
    // of the scalars the product needs only these two; the rotation follows the post
    const double beta = sqrt(sum > 0 ? sum : 0);
    last = last || !(beta > 0);
    const float s = (float)(1.0 / beta), ratio = k == 1 ? 0.f : (float)(beta / st.beta);
    if (!last) {
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * T < H) zh[t + u * T] = zl[u];
      for (int h = t + kPre * T; h < H; h += T) zh[h] = grid_load(zg + list[h]);
      __syncthreads();
      const int lane = t % LANES;
      for (int i = t / LANES; i < R; i += T / LANES) {
        float v = 0.f;
#pragma unroll 4
        for (int j = rowp[i] + lane, j1 = rowp[i + 1]; j < j1; j += LANES) v += val[j] * zh[idx[j]];
        v = lanes_total<LANES>(v);
        if (lane == 0) ys[i] = v;
      }
      __syncthreads();
      acc = 0;
      for (int i = t; i < R; i += T) {
        const float y = s * ys[i] - ratio * r1[i];
        r1[i] = y;
        acc += (double)(s * zc[i]) * (double)y;
      }
      grid_post(g, acc);
    }
    const MinresState in = st;
    minres_scalars(in, st, beta, k == 1);
    if (k > 1) {
      const MinresStep step(st);
      for (int i = t; i < R; i += T) {
        const float w = step.w(zp[i], wa[i], wb[i]);
        wa[i] = wb[i];
        wb[i] = w;
        xv[i] += step.phi * w;
      }
    }
    if (last) break;
    ok = grid_wait(g, sum);
    if (!ok) break;
    st.alfa = sum;
    const float c = (float)(sum / st.beta);
    acc = 0;
    for (int i = t; i < R; i += T) {
      const float y = r1[i] - c * r2[i], z = pin[i] * y;
      grid_store(zn + r0 + i, z);
      r1[i] = r2[i];
      r2[i] = y;
      zp[i] = zc[i];
      zc[i] = z;
      acc += (double)y * (double)z;
    }
    grid_post(g, acc);
    last = k >= a.maxit || (k % kGridCheck == 0 && st.phibar <= a.tol * st.beta1);
    ok = grid_wait(g, sum);
  }
  if (!ok) {
    if (t == 0) atomicMax(&a.res->status, 2);
    return;
  }
  for (int i = t; i < R; i += T) a.x[r0 + i] = xv[i];
  if (blockIdx.x == 0 && t == 0) a.res->iters = k > 1 ? k - 1 : 1;
}

namespace {
GridBackoff g_backoff;
int64_t grid_clock() {  // ns
  return std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now().time_since_epoch())
      .count();
}
int grid_device() {
  int dev = -1;
  return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}
}  // namespace

static void grid_pause() { g_backoff.note(grid_device(), grid_clock(), (int64_t)kGridRetrySeconds * 1000000000); }
bool grid_allowed(const GridControl& c) { return c.launches != 0 && !g_backoff.waits(grid_device(), grid_clock()); }

void grid_count(GridControl* c, int status) {
  ++(status ? c->declined : c->solved);
  if (status == 2 && !c->absent) grid_pause();
}

int grid_clear(grid_word* slots, int nblk, GridResult* res, int n_res, hipStream_t st) {
  const int64_t words = (int64_t)nblk * kGridBlockWords;
  hipLaunchKernelGGL(k_grid_clear, dim3(grid_for(std::max<int64_t>(words, n_res), 256)), dim3(256), 0, st, words, slots,
                     n_res, res);
  NFX_LAUNCH_CHECK();
  return NFX_OK;
}

int grid_launch(GridControl* c, const void* kernel, int nblk, void** args, hipStream_t st, bool* ran) {
  *ran = false;
  if (!grid_allowed(*c)) return NFX_OK;
  if (c->launches > 0) --c->launches;
  const hipError_t e = hipLaunchCooperativeKernel(kernel, dim3(nblk), dim3(kGridThreads), args, kGridLdsBytes, st);
  const GridLaunch what = grid_outcome(e);
  if (what != GridLaunch::ran) (void)hipGetLastError();
  if (what == GridLaunch::error) {
    set_error(std::string("cooperative launch: ") + hipGetErrorString(e));
    return NFX_E_HIP;
  }
  if (what == GridLaunch::busy) grid_pause();
  *ran = what == GridLaunch::ran;
  return NFX_OK;
}

// Resident blocks that the device allows (0: no cooperative launch, or too little LDS).
int minres_grid_capacity() {
  int dev = 0, coop = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !coop ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  for (const void* f : {(const void*)k_minres_grid<4>, (const void*)k_minres_grid<8>, (const void*)k_minres_grid<16>}) {
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kGridLdsBytes) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, kGridThreads, kGridLdsBytes) != hipSuccess ||
        per_cu < 1) {
      (void)hipGetLastError();
      return 0;
    }
  }
  return std::min(cus, kGridMaxBlocks);
}

// A sum over the grid takes 1.2 us with 8 blocks, 1.9 with 32, 2.2 with 64, 2.8 with 128, 3.3 with 256;
// the product and the loads of z shrink with the block's share. Best counts measured (us an iteration):
// 16 at 53 KB of entries and rows (4.5; 64 blocks 5.0), 32-64 at 0.39 MB (4.5; 128 blocks 5.4), 64 at
// 2 MB (5.3; 32 blocks 6.0, 128 blocks 5.7), 128 at 6.4-8 MB (6.5 and 7.7; 64 blocks 7.4 and 9.3, 256
// blocks 7.1 and 8.2), 256 at 22 MB (8.7).
int minres_grid_blocks(const MinresGrid* g, int n, int64_t nnz) {
  const int64_t bytes = 6 * nnz + 40 * (int64_t)n;
  const int64_t limits[] = {128 << 10, 512 << 10, 3 << 20, 10 << 20, INT64_MAX};
  int nblk = 16;
  for (const int64_t* l = limits; bytes > *l; ++l) nblk *= 2;
  for (; nblk <= g->max_blocks; nblk *= 2) {
    // room for the block's longest row beyond its share, for the columns it meets and, at set-up,
    // for the bit per column (the kernel looks again at what it finds)
    const int64_t spare = kGridLdsBytes - (24 << 10);
    if (bytes / nblk <= spare && (6 * nnz + 4 * (int64_t)n) / nblk + n / 4 <= spare) return nblk;
  }
  return 0;
}

// one flag a block, written to the host: the answer comes with whatever the stream is waited for next
__global__ __launch_bounds__(256) void k_grid_diagonal(int n, const int32_t* __restrict__ prp,
                                                       const int32_t* __restrict__ pci, int* __restrict__ other) {
  bool diag = true;
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += kGridDiagBlocks * 256) {
    const int j = prp[i];
    diag = diag && prp[i + 1] == j + 1 && pci[j] == i;
  }
  const int all = __syncthreads_and(diag);
  if (threadIdx.x == 0) other[blockIdx.x] = !all;
}

int minres_grid_ask(MinresGrid* g, int n, const int32_t* prp, const int32_t* pci, hipStream_t st) {
  hipLaunchKernelGGL(k_grid_diagonal, dim3(kGridDiagBlocks), dim3(256), 0, st, n, prp, pci, g->h_other);
  NFX_LAUNCH_CHECK();
  return NFX_OK;
}

bool minres_grid_diagonal(const MinresGrid* g) {
  return std::none_of(g->h_other, g->h_other + kGridDiagBlocks, [](int o) { return o != 0; });
}

int minres_grid_solve(MinresGrid* g, int nblk, int lanes, int n, const int32_t* rp, const int32_t* ci, const float* va,
                      const float* sign, const int32_t* prp, const int32_t* pci, const float* pva, const float* rhs,
                      float* x, float* z, double tol, int maxit, int* iters, int* status, hipStream_t st) {
  NFX_REQUIRE(nblk > 0 && nblk <= g->max_blocks, "minres_grid_solve: blocks");
  *status = 1;
  NFX_CHECK(grid_clear(g->slots, nblk, g->res, 1, st));
  MinresGridArgs a{n, nblk, maxit, kGridLdsBytes, rp, ci, va, sign, prp, pci, pva, rhs, x, z, tol, g->slots, g->res};
  void* args[] = {&a};
  const void* f = lanes == 16  ? (const void*)k_minres_grid<16>
                  : lanes == 8 ? (const void*)k_minres_grid<8>
                               : (const void*)k_minres_grid<4>;
  bool ran = false;
  NFX_CHECK(grid_launch(&g->control, f, nblk - (g->control.absent ? 1 : 0), args, st, &ran));
  if (!ran) return NFX_OK;
  NFX_CHECK_HIP(hipMemcpyAsync(g->h_res, g->res, sizeof(GridResult), hipMemcpyDeviceToHost, st));
  NFX_CHECK_HIP(hipStreamSynchronize(st));
  *iters = g->h_res->iters;
  *status = g->h_res->status;
  return NFX_OK;
}

}  // namespace nfx
