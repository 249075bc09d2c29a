// Batched MINRES: every instance resident in a few CUs for a whole inner solve, all instances of a
// launch side by side, each with its own recurrence, exchange and stopping test.
//
// A block owns a share of an instance's flux rows and of its aggregates of cells with their pressure
// rows; the matrix columns (renumbered to 16 bits), the values where they fit, and the vectors stay in
// LDS; a thread works for each pressure row.
// With the two-grid cycle an iteration has three exchanges within the instance:
//   z | product, alpha | y', x1 = W y' (a cell's and, again, its neighbours'), t1 = y' - S x1 and its
//   sums cv over the aggregates | y = Ac^-1 cv in every block, t2 = t1 - S P y, z = x1 + P y + W t2, y'.z
// where the stepwise kernels need eight launches over the whole batch. Without a cycle (diagonal
// preconditioner) the middle one falls away; the learned smoother's couplings add two, for x1 and t2.
// Bound by the exchanges (1.2-2.6 us each, and ~1 us for what is then loaded) and the product. Twelve
// instances of 384-4,374 cells, both degrees: 70 us an iteration stepwise, 17.5 us here; the largest (58,320
// rows, 1.5 M entries, 87 blocks) alone takes 18 us with the cycle and 10 us without.
#include <algorithm>
#include <climits>

#include "nfx_bm_grid.h"

namespace nfx {
namespace {

constexpr int kT = kGridThreads;
constexpr int kBmGridAgg = 128;    // coarse unknowns of an instance: 16 inverse entries a thread
// Bytes of an instance (6 an entry, 40 a row) per block: what leaves room for the values in LDS. Half of
// it is no faster (the sums over twice the blocks take longer) and fills two launches instead of one.
constexpr int64_t kBmGridShare = 128 << 10;
// Launches of a resident batch: they run one after the other, 10-18 us an iteration each, where the stepwise
// kernels take all instances in the same launches (25 us an iteration with the diagonal, 56 with the cycle, and
// 7-15 for what a full launch here holds). Up to three pay, up to six where they are three quarters full. Set-up
// and solve in ms, resident / stepwise, diagonal | two-grid: instances of 9 cubed of degree 2 (87 blocks, two a
// launch) in 1 launch 12.6/35.1 | 5.1/15.1, in 2 24.1/39.2 | 9.7/16.5, in 3 35.9/42.4 | 14.6/18.4, in 4 46.4/45.6
// | 19.2/19.6, in 6 68.5/64.9 | 28.4/25.9, in 12 137/98 | 56/43; of 5 cubed (15 blocks, 17 a launch) in 3
// 19.7/26.6 | 12.9/17.1, in 6 38.8/43.7 | 25.3/26.7; of degree 1, 6 cubed (3 blocks) in 3 8.0/11.9 | 9.8/13.5.
constexpr int kBmGridLaunches = 6;
inline bool bm_grid_pays(int launches, int blocks, int cap) {
  return launches <= 3 || (launches <= kBmGridLaunches && 4 * (int64_t)blocks >= 3 * (int64_t)launches * cap);
}

struct BmGridArgs {
  const nfx_minres_batch_item* items;
  const BmGridBlock* blocks;
  const int32_t* mode;
  const int32_t* ranges;
  nfx_batch_tg pc[2];
  int n_groups, maxit, lds;
  int64_t n_total;
  const float* rhs;
  float *x, *vec, *own;
  const double* tol;
  grid_word* slots;
  GridResult* res;
};

__global__ __launch_bounds__(256) void k_bm_grid_zero(int n, int32_t* p) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

// runs of equal instance in a group's cells (what 0) or flux blocks (1): first, end, number of runs
// (and, of cells, the instance's aggregates)
__global__ __launch_bounds__(256) void k_bm_ranges(int n, const int32_t* __restrict__ inst, int n_inst, int group,
                                                   int what, const int32_t* __restrict__ agg_of,
                                                   const int32_t* __restrict__ alen, int32_t* __restrict__ ranges) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  const int i = inst[c];
  if (i < 0 || i >= n_inst) return;
  int32_t* r = ranges + (int64_t)i * kBmRanges + group * 6 + what * 3;
  if (c == 0 || inst[c - 1] != i) {
    r[0] = c;
    atomicAdd(r + 2, 1);
    if (what == 0) atomicMax(ranges + (int64_t)i * kBmRanges + 12, alen[agg_of[c]]);
  }
  if (c == n - 1 || inst[c + 1] != i) r[1] = c + 1;
}

__global__ __launch_bounds__(256) void k_bm_nnz(int n_inst, const nfx_minres_batch_item* __restrict__ items,
                                                int32_t* __restrict__ nnz) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n_inst) nnz[i] = items[i].rowptr[items[i].n_rows];
}

// Blocks of an instance: from its own size alone.
inline int bm_grid_blocks(int n, int64_t nnz) {
  return (int)((6 * nnz + 40 * (int64_t)n + kBmGridShare - 1) / kBmGridShare);
}

// value of lane `J` of the thread's group of four
template <int J>
__device__ __forceinline__ float quad(float v) {
  return dpp_move<J * 0x55>(v);
}

// row of a cell block (w) times the cell's values, one per lane of its NB lanes
template <int NB>
__device__ __forceinline__ float cell_dot(const float (&w)[NB], float v) {
  if (NB == 1) return w[0] * v;
  return w[0] * quad<0>(v) + w[NB > 1 ? 1 : 0] * quad<1>(v) + w[NB > 2 ? 2 : 0] * quad<2>(v) +
         w[NB > 3 ? 3 : 0] * quad<3>(v);
}

// One instance on the calling blocks. NB: pressure unknowns of a cell under the two-grid cycle, 0 without.
template <int NB>
__device__ __forceinline__ void bm_grid_run(const BmGridArgs& a, const BmGridBlock& bl, GridSync& g, char* lds, int* scan,
                                            MinresState* sts,
                            const nfx_batch_tg& pc, int c0, int c1, int f0, int f1) {
  constexpr int LANES = 8;
  constexpr int NBS = NB ? NB : 1;
  const int t = threadIdx.x, B = bl.nblk, rank = bl.rank;
  const nfx_minres_batch_item it = a.items[bl.inst];
  const int n = uniform(it.n_rows);
  const int32_t off = uniform((int32_t)it.row_off);
  const bool wo = NB == 1 && pc.wo != nullptr;

  // the block's share: flux blocks or rows [u0, u1), aggregates [A0 + a0, A0 + a1) with their cells
  const int n_u = n - (NB ? (c1 - c0) * NB : 0);
  const bool fb = f1 > f0;
  const int units = n_u < 0 ? 0 : fb ? f1 - f0 : n_u;
  int A0 = 0, A = 0, a0 = 0, a1 = 0, m0 = 0, nC = 0;
  bool good = n_u >= 0 && (!fb || 3 * units == n_u);
  if (NB) {
    const int first = uniform(pc.agg_of[c0]);
    A0 = uniform(pc.a0[first]);
    A = uniform(pc.alen[first]);
    good = good && (int64_t)c1 * 4 * NBS * NBS <= INT_MAX && A > 0 && A <= kBmGridAgg && A0 >= 0 && A0 + A <= pc.n_agg &&
           pc.agg_ptr[A0 + A] - pc.agg_ptr[A0] == c1 - c0;
    if (good) {
      a0 = (int)((int64_t)A * rank / B);
      a1 = (int)((int64_t)A * (rank + 1) / B);
      m0 = uniform(pc.agg_ptr[A0 + a0]);
      nC = uniform(pc.agg_ptr[A0 + a1]) - m0;
      good = nC >= 0 && nC * NB <= kT;
    }
  }
  if (!good) nC = a0 = a1 = A = 0;
  // aggregates are few and uneven, so the flux rows make up for them: bounds where 3 a flux row and 2 a
  // pressure row are even (an even split of the flux rows cost 22 us against 16 us an iteration where
  // a block has one or two aggregates), or evenly split where some block's cells alone exceed the share
  const int per = fb ? 3 : 1;
  const auto bound = [&](int r) {
    const int64_t cells = A > 0 ? pc.agg_ptr[A0 + (int)((int64_t)A * r / B)] - pc.agg_ptr[A0] : 0;
    const int64_t all = 3 * (int64_t)units * per + 2 * (int64_t)NB * (c1 - c0);
    const int64_t u = r >= B ? units : (all * r / B - 2 * NB * cells) / (3 * per);
    return (int)(u < 0 ? 0 : u > units ? units : u);
  };
  bool even = true;
  if (NB && good) {
    bool up = true;
    for (int r = t; r < B; r += kT) up = up && bound(r + 1) >= bound(r);
    even = !__syncthreads_and(up);
  }
  const int u0 = uniform(even ? (int)((int64_t)units * rank / B) : bound(rank)),
            u1 = uniform(even ? (int)((int64_t)units * (rank + 1) / B) : bound(rank + 1));
  const int Rf = (u1 - u0) * per;
  const int Rp = nC * NB, R = Rf + Rp;

  // one thread per pressure row: its cell's rows of S and W, neighbours' rows, aggregates
  const bool mine = t < Rp;
  const int comp = t % NBS;
  // (a byte each); S, W and the coarse inverse are loaded in the waits (held, they would spill)
  int row = 0, d_at = 0, nrow[4] = {-1, -1, -1, -1}, wq_at[4] = {-1, -1, -1, -1};
  unsigned ag = 0, agc = 0;
  if (NB && mine) {
    const int c = pc.agg_mem[m0 + t / NBS];
    good = c >= c0 && c < c1;
    if (good) {
      row = pc.prow[(int64_t)c * NBS + comp];
      good = row >= off + n_u && row < off + n;
      d_at = c;
      const int x = pc.agg_of[c] - A0;
      agc = x & 255;
      good = good && x >= a0 && x < a1;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int q = pc.nbr[4 * c + k];
        if (q < 0) continue;
        if (q < c0 || q >= c1) {
          good = false;
          continue;
        }
        nrow[k] = pc.prow[(int64_t)q * NBS + comp];
        wq_at[k] = (q * NBS + comp) * NBS;
        const int y = pc.agg_of[q] - A0;
        ag |= (unsigned)(y & 255) << (8 * k);
        good = good && nrow[k] >= off + n_u && nrow[k] < off + n && y >= 0 && y < A;
      }
    }
  }
  const bool coarse = NB && t / 8 < A;  // takes row t / 8 of the coarse inverse, entries t % 8 + 8 u
  const float* arow = coarse && good ? pc.ainv + pc.arow[A0 + t / 8] + t % 8 : nullptr;

  // LDS: row starts | row numbers | vectors | flux blocks | cells' t1, cv, y | columns (16 bits)
  // | z at the columns | values, if they fit | ... | column list, if it is not in registers
  int* rowp = reinterpret_cast<int*>(lds);
  int* rid = rowp + R + 1;
  float *r1 = reinterpret_cast<float*>(rid + R), *r2 = r1 + R, *zc = r2 + R, *sgv = zc + R, *ys = sgv + R;
  float *fbl = ys + R, *tc = fbl + (fb ? 3 : 1) * Rf, *cv = tc + Rp, *yl = cv + (NB ? kBmGridAgg : 0);
  int* at = reinterpret_cast<int*>(yl + (NB ? kBmGridAgg : 0));  // where the aggregates' rows start in tc
  unsigned short* idx = reinterpret_cast<unsigned short*>(at + (a1 - a0 + 1));
  const int64_t fixed = reinterpret_cast<char*>(idx) - lds;
  good = __syncthreads_and(good && fixed + 4 <= a.lds);
  constexpr int kPre = 4;  // places of the list that a thread holds
  int nz = 0, H = 0, col[kPre] = {};
  int* list = nullptr;
  float *zh = nullptr, *val = nullptr;
  if (good) {
    // rows and the starts of their entries (a scan of their lengths)
    const int run = (R + kT - 1) / kT, i0 = min(R, t * run), i1 = min(R, i0 + run);
    int cnt = 0;
    for (int i = i0; i < i1; ++i) {
      int r;
      if (i >= Rf)
        r = pc.prow[(int64_t)pc.agg_mem[m0 + (i - Rf) / NBS] * NBS + (i - Rf) % NBS] - off;
      else if (fb)
        r = pc.fb_rows[(int64_t)(f0 + u0) * 3 + i] - off;
      else
        r = u0 + i;
      if (r < 0 || r >= n || (i < Rf && r >= n_u)) {
        good = false;
        r = 0;
      }
      rid[i] = r;
      cnt += it.rowptr[r + 1] - it.rowptr[r];
    }
    int inc = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if ((t & 63) >= o) inc += v;
    }
    if ((t & 63) == 63) scan[t >> 6] = inc;
    __syncthreads();
    int pre = inc - cnt;
    for (int w = 0; w < kT / 64; ++w) {
      if (w < (t >> 6)) pre += scan[w];
      nz += scan[w];
    }
    nz = uniform(nz);
    for (int i = i0; i < i1; ++i) {
      rowp[i] = pre;
      pre += it.rowptr[rid[i] + 1] - it.rowptr[rid[i]];
    }
    if (t == 0) rowp[R] = nz;
    const int64_t base = fixed + 4 * (((int64_t)nz + 1) / 2), nw = (n + 31) >> 5;
    good = __syncthreads_and(good && base + 8 * nw <= a.lds);
    if (good) {
      unsigned* bits = reinterpret_cast<unsigned*>(lds + base);
      int* before = reinterpret_cast<int*>(bits + nw);
      const auto start = [&](int i) { return it.rowptr[rid[i]]; };
      H = uniform(grid_columns<LANES>(it.col, n, R, rowp, start, bits, before, scan));
      good = H <= 65535 && base + 8 * nw + 4 * (int64_t)H <= a.lds && base + 8 * (int64_t)H <= a.lds;
      if (good) {
        list = reinterpret_cast<int*>(lds + a.lds) - H;
        grid_renumber<LANES>(it.col, n, R, rowp, start, bits, before, list, idx);
        zh = reinterpret_cast<float*>(lds + base);
#pragma unroll
        for (int u = 0; u < kPre; ++u) col[u] = t + u * kT < H ? list[t + u * kT] : 0;
        __syncthreads();
        if (base + (H > kPre * kT ? 8 : 4) * (int64_t)H + 4 * (int64_t)nz <= a.lds) {
          val = zh + H;
          for (int i = t / LANES; i < R; i += kT / LANES) {
            const float* v = it.val32 + start(i);
            for (int j = t % LANES, len = rowp[i + 1] - rowp[i]; j < len; j += LANES) val[rowp[i] + j] = v[j];
          }
        }
        for (int i = t; i < R; i += kT) {
          sgv[i] = it.sign ? it.sign[rid[i]] : 1.f;
        }
        if (NB && t <= a1 - a0) at[t] = (pc.agg_ptr[A0 + a0 + t] - m0) * NBS;
        for (int i = t; i < (fb ? 3 : 1) * Rf; i += kT)
          fbl[i] = fb ? pc.fb_inv[(int64_t)(f0 + u0) * 9 + i] : it.pinv ? it.pinv[rid[i]] : 1.f;
      }
    }
  }
  double sum;
  grid_post(g, t == 0 && !good ? 1.0 : 0.0);
  bool ok = grid_wait(g, sum);
  if (!ok || sum != 0) {
    if (t == 0) atomicMax(&a.res[bl.inst].status, ok ? 1 : 2);
    return;
  }

  // exchanged vectors, by row of the stacked system
  const int64_t N = a.n_total;
  float *Z = a.vec, *Y = a.vec + 2 * N, *RR = a.vec + 3 * N, *X1 = a.vec + 5 * N, *T2 = a.vec + 6 * N,
        *CV = a.vec + 7 * N + off;
  // of the block's own rows, off the path of the exchanges: w of the last two steps, z before zc
  float *wa = a.own + off, *wb = wa + N, *zp = wb + N, *xv = a.x + off;
  int lr = Rf + t;
  double acc = 0;
  int k = 0;
  for (; ok; ++k) {
    float c = 0.f;
    // opaque to the compiler: addresses made from these would be kept over the loop, in scratch memory
    asm volatile("" : "+v"(d_at), "+v"(row), "+v"(nrow[0]), "+v"(nrow[1]), "+v"(nrow[2]), "+v"(nrow[3]));
    asm volatile("" : "+v"(wq_at[0]), "+v"(wq_at[1]), "+v"(wq_at[2]), "+v"(wq_at[3]), "+v"(lr));
#pragma unroll
    for (int u = 0; u < kPre; ++u) asm volatile("" : "+v"(col[u]));
    // the neighbours' rows of W come during a wait (held for the whole solve they would spill)
    float wq[4][NBS], wd[NBS];
    const auto load_wq = [&]() {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < NBS; ++j)
          wq[q][j] = !NB || wq_at[q] < 0 ? 0.f : wo ? pc.wo[4 * d_at + q] : pc.wd[wq_at[q] + j];
#pragma unroll
      for (int j = 0; j < NBS; ++j) wd[j] = mine ? pc.wd[(d_at * NBS + comp) * NBS + j] : 0.f;
    };
    if (k == 0) {
      load_wq();
      for (int i = t; i < R; i += kT) {
        const float b = a.rhs[off + rid[i]];
        r1[i] = r2[i] = b;
        const int r = rid[i];
        zc[i] = zp[r] = wa[r] = wb[r] = xv[r] = 0.f;
        if (NB && i >= Rf) grid_store(RR + N + off + rid[i], b);
      }
    } else {
      const float* zg = Z + (int64_t)(k & 1) * N + off;
      float zl[kPre];
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * kT < H) zl[u] = grid_load(zg + col[u]);
      const double beta = sqrt(sum > 0 ? sum : 0);
      const float s = (float)(1.0 / beta), ratio = k == 1 ? 0.f : (float)(beta / sts[(k + 1) & 1].beta);
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * kT < H) zh[t + u * kT] = zl[u];
      for (int h = t + kPre * kT; h < H; h += kT) zh[h] = grid_load(zg + list[h]);
      __syncthreads();
      for (int i = t / LANES; i < R; i += kT / LANES) {
        float v = 0.f;
        const int j0 = rowp[i], len = rowp[i + 1] - j0;
        if (val) {
#pragma unroll 4
          for (int j = t % LANES; j < len; j += LANES) v += val[j0 + j] * zh[idx[j0 + j]];
        } else {
          const float* va = it.val32 + it.rowptr[rid[i]];
#pragma unroll 4
          for (int j = t % LANES; j < len; j += LANES) v += va[j] * zh[idx[j0 + j]];
        }
        v = lanes_total<LANES>(v);
        if (t % LANES == 0) ys[i] = v;
      }
      __syncthreads();
      acc = 0;
      for (int i = t; i < R; i += kT) {
        const float y = s * sgv[i] * ys[i] - ratio * r1[i];
        r1[i] = y;
        if (NB && i >= Rf) grid_store(Y + off + rid[i], y);
        acc += (double)(s * zc[i]) * (double)y;
      }
      grid_post(g, acc);
      // the rotation, and every kGridCheck iterations the test of the estimate after k - 1 of them
      MinresState st;
      minres_scalars(sts[(k + 1) & 1], st, beta, k == 1);
      if (t == 0) sts[k & 1] = st;  // read after the next barrier only
      const bool last = !(beta > 0) || k - 1 >= a.maxit ||
                        (k > 1 && (k - 1) % kGridCheck == 0 && st.phibar <= a.tol[bl.inst] * st.beta1);
      if (k > 1) {
        const MinresStep step(st);
        for (int i = t; i < R; i += kT) {
          const int r = rid[i];
          const float w1 = wb[r], w = step.w(zp[r], wa[r], w1);
          wa[r] = w1;
          wb[r] = w;
          xv[r] += step.phi * w;
          zp[r] = zc[i];
        }
      } else {
        for (int i = t; i < R; i += kT) zp[rid[i]] = zc[i];
      }
      if (last) break;
      load_wq();
      ok = grid_wait(g, sum);
      if (!ok) break;
      if (t == 0) sts[k & 1].alfa = sum;
      c = (float)(sum / sts[k & 1].beta);
      for (int i = t; i < R; i += kT) {
        const float y = r1[i] - c * r2[i];
        r1[i] = r2[i];
        r2[i] = y;
        if (NB && i >= Rf) grid_store(RR + (int64_t)((k + 1) & 1) * N + off + rid[i], y);
      }
    }
    __syncthreads();

    // z of iteration k + 1 from y' (r2); RR[(k + 1) & 1] holds y' of this step, RR[k & 1] that before it
    float* zn = Z + (int64_t)((k + 1) & 1) * N;
    float x1 = 0.f, t1 = 0.f;
    if (NB) {
      float xq[4] = {}, so[4][NBS], sd[NBS];
      if (mine) {
        // r of the neighbours from what they published: y and the r2 before it
        float yq[4], rq[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          yq[q] = rq[q] = 0.f;
          if (nrow[q] < 0) continue;
          if (k) {
            yq[q] = grid_load(Y + nrow[q]);
            rq[q] = grid_load(RR + (int64_t)(k & 1) * N + nrow[q]);
          } else {
            yq[q] = a.rhs[nrow[q]];
          }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int j = 0; j < NBS; ++j) so[q][j] = pc.so[((d_at * 4 + q) * NBS + comp) * NBS + j];
#pragma unroll
        for (int j = 0; j < NBS; ++j) sd[j] = pc.sd[(d_at * NBS + comp) * NBS + j];
        x1 = cell_dot<NBS>(wd, r2[lr]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float rn = yq[q] - c * rq[q];
          if (wo)
            x1 += wq[q][0] * rn;
          else
            xq[q] = cell_dot<NBS>(wq[q], rn);
        }
      }
      if (wo) {  // x1 of the neighbours takes their own neighbours: exchanged
        if (mine) grid_store(X1 + row, x1);
        grid_post(g, 0.0);
        ok = grid_wait(g, sum);
        if (!ok) break;
        if (mine) {
#pragma unroll
          for (int q = 0; q < 4; ++q) xq[q] = nrow[q] >= 0 ? grid_load(X1 + nrow[q]) : 0.f;
        }
      }
      if (mine) {
        float s = cell_dot<NBS>(sd, x1);
#pragma unroll
        for (int q = 0; q < 4; ++q) s += cell_dot<NBS>(so[q], xq[q]);
        t1 = r2[lr] - s;
        tc[t] = t1;
      }
      __syncthreads();
      for (int x = a0 + (t >> 6); x < a1; x += kT / 64) {
        double v = 0;
        for (int j = at[x - a0] + (t & 63), j1 = at[x - a0 + 1]; j < j1; j += 64) v += (double)tc[j];
        v = wave_total(v);
        if ((t & 63) == 0) grid_store(CV + x, (float)v);
      }
      grid_post(g, 0.0);
    }
    acc = 0;
    for (int i = t; i < Rf; i += kT) {
      float z;
      if (fb) {
        const int j = i - i % 3;
        z = fbl[3 * i] * r2[j] + fbl[3 * i + 1] * r2[j + 1] + fbl[3 * i + 2] * r2[j + 2];
      } else {
        z = fbl[i] * r2[i];
      }
      grid_store(zn + off + rid[i], z);
      zc[i] = z;
      acc += (double)r2[i] * (double)z;
    }
    if (NB) {
      float ai[kBmGridAgg / 8], rs[5];
#pragma unroll
      for (int q = 0; q < 5; ++q) rs[q] = mine ? pc.rs[(d_at * 5 + q) * NBS + comp] : 0.f;
#pragma unroll
      for (int u = 0; u < kBmGridAgg / 8; ++u) ai[u] = coarse && t % 8 + 8 * u < A ? arow[8 * u] : 0.f;
      ok = grid_wait(g, sum);
      if (!ok) break;
      if (t < A) cv[t] = grid_load(CV + t);
      __syncthreads();
      {
        float v = 0.f;
#pragma unroll
        for (int u = 0; u < kBmGridAgg / 8; ++u)
          if (t % 8 + 8 * u < A) v += ai[u] * cv[t % 8 + 8 * u];
        v = lanes_total<8>(v);
        if (t % 8 == 0 && coarse) yl[t / 8] = v;
      }
      __syncthreads();
      float z = 0.f, t2 = 0.f;
      if (mine) {
        float spy = rs[0] * yl[agc];
#pragma unroll
        for (int q = 0; q < 4; ++q) spy += rs[1 + q] * yl[(ag >> (8 * q)) & 255];
        t2 = t1 - spy;
        z = x1 + yl[agc];
        z += cell_dot<NBS>(wd, t2);
      }
      if (wo) {  // the smoother's couplings: t2 of the neighbours
        if (mine) grid_store(T2 + row, t2);
        grid_post(g, 0.0);
        ok = grid_wait(g, sum);
        if (!ok) break;
        if (mine) {
          float tq[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) tq[q] = nrow[q] >= 0 ? grid_load(T2 + nrow[q]) : 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) z += wq[q][0] * tq[q];
        }
      }
      if (mine) {
        grid_store(zn + row, z);
        zc[lr] = z;
        acc += (double)r2[lr] * (double)z;
      }
    }
    grid_post(g, acc);
    ok = grid_wait(g, sum);
  }
  if (!ok) {
    if (t == 0) atomicMax(&a.res[bl.inst].status, 2);
    return;
  }
  if (rank == 0 && t == 0) a.res[bl.inst].iters = k > 1 ? k - 1 : 1;
}

__global__ __launch_bounds__(kT) void k_bm_grid(BmGridArgs a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ double sh_post[2][kT / 64], sh_part[2][kT / 64];
  __shared__ int sh_good[2][kT / 64], scan[kT / 64];
  __shared__ MinresState sts[2];
  BmGridBlock bl = a.blocks[blockIdx.x];
  bl = BmGridBlock{uniform(bl.inst), uniform(bl.rank), uniform(bl.nblk), uniform(bl.first)};
  if (a.mode[bl.inst] != 0) return;
  GridSync g{a.slots + (int64_t)bl.first * kGridBlockWords, bl.nblk, bl.rank, 0, sh_post, sh_part, sh_good};
  const int32_t* r = a.ranges + (int64_t)bl.inst * kBmRanges;
  // the instance's group: the one that has cells of it, in one run
  int group = -1;
  bool one = true;
  for (int q = 0; q < a.n_groups; ++q)
    if (r[6 * q + 2] + r[6 * q + 5]) {
      one = one && group < 0 && r[6 * q + 2] == 1 && r[6 * q + 5] <= 1;
      group = q;
    }
  if (!one) {
    if (threadIdx.x == 0) atomicMax(&a.res[bl.inst].status, 1);
    return;
  }
  if (group < 0) {
    bm_grid_run<0>(a, bl, g, lds, scan, sts, a.pc[0], 0, 0, 0, 0);
    return;
  }
  group = uniform(group);
  const nfx_batch_tg& pc = a.pc[group];
  const int32_t* q = r + 6 * group;
  const int c0 = uniform(q[0]), c1 = uniform(q[1]), f0 = uniform(q[5] ? q[3] : 0), f1 = uniform(q[5] ? q[4] : 0);
  if (pc.nb == 1)
    bm_grid_run<1>(a, bl, g, lds, scan, sts, pc, c0, c1, f0, f1);
  else
    bm_grid_run<4>(a, bl, g, lds, scan, sts, pc, c0, c1, f0, f1);
}

}  // namespace

// Launches of the batch; where it can be resident, its work space. One that cannot allocates nothing.
static int bm_grid_plan(BmGrid* g, const std::vector<int>& rows, int64_t n_total, const nfx_minres_batch_item* d_items,
                        int32_t* scratch, hipStream_t st) {
  const int n_inst = (int)rows.size();
  int dev = 0, coop = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !coop ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipFuncSetAttribute((const void*)k_bm_grid, hipFuncAttributeMaxDynamicSharedMemorySize, kGridLdsBytes) !=
          hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_bm_grid, kT, kGridLdsBytes) !=
          hipSuccess ||
      per_cu < 1) {
    (void)hipGetLastError();
    return NFX_OK;
  }
  const int cap = std::min(cus, kGridMaxBlocks);

  // entries of each instance, its blocks, and launches of at most `cap` blocks, largest instances first
  std::vector<int32_t> nnz(n_inst);
  hipLaunchKernelGGL(k_bm_nnz, dim3(grid_for(n_inst, 256)), dim3(256), 0, st, n_inst, d_items, scratch);
  NFX_LAUNCH_CHECK();
  NFX_CHECK_HIP(hipMemcpyAsync(nnz.data(), scratch, sizeof(int32_t) * n_inst, hipMemcpyDeviceToHost, st));
  NFX_CHECK_HIP(hipStreamSynchronize(st));
  std::vector<int> nblk(n_inst), order(n_inst);
  int64_t total = 0;
  for (int i = 0; i < n_inst; ++i) {
    nblk[i] = bm_grid_blocks(rows[i], nnz[i]);
    order[i] = i;
    total += nblk[i];
    if (nblk[i] < 1 || nblk[i] > cap || total > (int64_t)kBmGridLaunches * cap) return NFX_OK;
  }
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return nblk[a] > nblk[b]; });
  std::vector<std::vector<BmGridBlock>> waves;
  std::vector<int> wave_of(n_inst);
  for (int i : order) {
    size_t w = 0;
    while (w < waves.size() && (int)waves[w].size() + nblk[i] > cap) ++w;
    if (w == waves.size()) waves.emplace_back();
    wave_of[i] = (int)w;
    const int first = (int)waves[w].size();
    for (int r = 0; r < nblk[i]; ++r) waves[w].push_back(BmGridBlock{i, r, nblk[i], first});
  }
  std::vector<BmGridBlock> all;
  std::vector<int> wave_at(1, 0);
  for (const auto& w : waves) {
    all.insert(all.end(), w.begin(), w.end());
    wave_at.push_back((int)all.size());
  }
  if (!bm_grid_pays((int)waves.size(), (int)all.size(), cap)) return NFX_OK;

  // one device and one pinned allocation; without them the batch runs stepwise
  size_t at = 0;
  const auto piece = [&at](size_t bytes) {
    const size_t here = at;
    at += (bytes + 255) & ~(size_t)255;
    return here;
  };
  const size_t o_rng = piece(sizeof(int32_t) * (size_t)n_inst * kBmRanges),
               o_slots = piece(sizeof(grid_word) * kGridSlotWords), o_res = piece(sizeof(GridResult) * n_inst),
               o_tol = piece(sizeof(double) * n_inst), o_blk = piece(sizeof(BmGridBlock) * all.size()),
               o_own = piece(sizeof(float) * 3 * (size_t)n_total);
  hipError_t e = hipMalloc(&g->dev, at);
  at = 0;
  const size_t h_res = piece(sizeof(GridResult) * n_inst), h_tol = piece(sizeof(double) * n_inst);
  if (e == hipSuccess) e = hipHostMalloc(&g->host, at, hipHostMallocDefault);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    if (g->dev) (void)hipFree(g->dev);
    g->dev = nullptr;
    return NFX_OK;
  }
  g->ranges = reinterpret_cast<int32_t*>(g->dev + o_rng);
  g->slots = reinterpret_cast<grid_word*>(g->dev + o_slots);
  g->res = reinterpret_cast<GridResult*>(g->dev + o_res);
  g->tol = reinterpret_cast<double*>(g->dev + o_tol);
  g->blocks = reinterpret_cast<BmGridBlock*>(g->dev + o_blk);
  g->own = reinterpret_cast<float*>(g->dev + o_own);
  g->h_res = reinterpret_cast<GridResult*>(g->host + h_res);
  g->h_tol = reinterpret_cast<double*>(g->host + h_tol);
  NFX_CHECK_HIP(hipMemcpy(g->blocks, all.data(), sizeof(BmGridBlock) * all.size(), hipMemcpyHostToDevice));
  for (const auto& w : waves) g->tail.push_back(w.back().nblk > 1);
  g->wave_of.swap(wave_of);
  g->wave_at.swap(wave_at);
  return NFX_OK;
}

void bm_grid_destroy(BmGrid* g) {
  if (g->dev) (void)hipFree(g->dev);
  if (g->host) (void)hipHostFree(g->host);
  *g = BmGrid();
}

int bm_grid_route(BmGrid* g, const std::vector<int>& rows, int64_t n_total, const nfx_minres_batch_item* d_items,
                  const std::vector<nfx_batch_tg>& pc, int32_t* scratch, bool* resident, hipStream_t st) {
  const int n_inst = (int)rows.size();
  *resident = false;
  if (n_total > INT32_MAX || !grid_allowed(g->control)) return NFX_OK;
  // all or none: beside instances that have to iterate stepwise the others cost little there and a launch
  // each here (32 instances up to 16 x 16 x 16 cubes: 79.5 ms stepwise, 94.5 ms split)
  if (!g->planned) {
    g->planned = true;
    NFX_CHECK(bm_grid_plan(g, rows, n_total, d_items, scratch, st));
  }
  if (g->wave_of.empty()) return NFX_OK;
  hipLaunchKernelGGL(k_bm_grid_zero, dim3(grid_for(n_inst * kBmRanges, 256)), dim3(256), 0, st, n_inst * kBmRanges,
                     g->ranges);
  for (size_t q = 0; q < pc.size(); ++q) {
    hipLaunchKernelGGL(k_bm_ranges, dim3(grid_for(pc[q].n_cells, 256)), dim3(256), 0, st, pc[q].n_cells,
                       pc[q].cell_inst, n_inst, (int)q, 0, pc[q].agg_of, pc[q].alen, g->ranges);
    if (pc[q].n_fb > 0)
      hipLaunchKernelGGL(k_bm_ranges, dim3(grid_for(pc[q].n_fb, 256)), dim3(256), 0, st, pc[q].n_fb, pc[q].fb_inst,
                         n_inst, (int)q, 1, nullptr, nullptr, g->ranges);
  }
  NFX_LAUNCH_CHECK();
  if (!pc.empty()) {
    std::vector<int32_t> r((size_t)n_inst * kBmRanges);
    NFX_CHECK_HIP(hipMemcpyAsync(r.data(), g->ranges, sizeof(int32_t) * r.size(), hipMemcpyDeviceToHost, st));
    NFX_CHECK_HIP(hipStreamSynchronize(st));
    for (int i = 0; i < n_inst; ++i)
      if (r[(size_t)i * kBmRanges + 12] > kBmGridAgg) return NFX_OK;
  }
  *resident = true;
  return NFX_OK;
}

int bm_grid_solve(BmGrid* g, int n_inst, int64_t n_total, const nfx_minres_batch_item* d_items, const int32_t* d_mode,
                  const int32_t* h_mode, const std::vector<nfx_batch_tg>& pc, const float* rhs, float* x, float* vec,
                  const double* tol, int maxit, int* iters, std::vector<char>* done, hipStream_t st) {
  done->assign(n_inst, 0);
  const int waves = (int)g->wave_at.size() - 1;
  std::vector<char> runs(waves, 0);
  for (int i = 0; i < n_inst; ++i) {
    if (h_mode[i] == 0) runs[g->wave_of[i]] = 1;
    g->h_tol[i] = tol[i];
  }
  NFX_CHECK_HIP(hipMemcpyAsync(g->tol, g->h_tol, sizeof(double) * n_inst, hipMemcpyHostToDevice, st));
  BmGridArgs a{};
  a.items = d_items;
  a.mode = d_mode;
  a.ranges = g->ranges;
  a.n_groups = (int)pc.size();
  a.maxit = maxit;
  a.lds = kGridLdsBytes;
  a.n_total = n_total;
  a.rhs = rhs;
  a.x = x;
  a.vec = vec;
  a.own = g->own;
  a.tol = g->tol;
  a.slots = g->slots;
  a.res = g->res;
  for (int q = 0; q < a.n_groups; ++q) a.pc[q] = pc[q];
  bool first = true;
  int runs_until = waves;
  for (int w = 0; w < waves; ++w) {
    if (!runs[w]) continue;
    const int nblk = g->wave_at[w + 1] - g->wave_at[w];
    NFX_CHECK(grid_clear(g->slots, nblk, g->res, first ? n_inst : 0, st));
    first = false;
    a.blocks = g->blocks + g->wave_at[w];
    void* args[] = {&a};
    bool ran = false;
    NFX_CHECK(grid_launch(&g->control, (const void*)k_bm_grid, nblk - (g->control.absent && g->tail[w] ? 1 : 0), args,
                          st, &ran));
    if (!ran) {  // the stepwise kernels take this and the later launches
      runs_until = w;
      break;
    }
  }
  NFX_CHECK_HIP(hipMemcpyAsync(g->h_res, g->res, sizeof(GridResult) * n_inst, hipMemcpyDeviceToHost, st));
  NFX_CHECK_HIP(hipStreamSynchronize(st));
  for (int i = 0; i < n_inst; ++i) {
    if (h_mode[i] != 0) continue;
    if (g->wave_of[i] < runs_until && g->h_res[i].status == 0) {
      (*done)[i] = 1;
      iters[i] = g->h_res[i].iters;
    }
    grid_count(&g->control, (*done)[i] ? 0 : g->wave_of[i] < runs_until ? g->h_res[i].status : 1);
  }
  return NFX_OK;
}

}  // namespace nfx
