// FP32 MINRES of the dual-mixed elasticity operator (3 x 3 blocks) with its two-grid preconditioner, one
// cooperative launch per inner solve.
//
// A block owns a range of faces (9 stress rows each) and a range of cells in aggregate order (6 rows
// each); its rows of the operator, the face inverses and the vectors stay in LDS. A thread works for one
// of a cell's five blocks of S (its own and its neighbours') in one component and keeps that row of the
// block and of the W it meets in registers. An iteration has three exchanges:
//   z | y = A z, alpha | y', x1 = W y' of the cells and, again, of their neighbours, t1 = y' - S x1 and
//   its sums over the aggregates (a piece per block) | the coarse values that the block needs,
//   z = x1 + P y + W (t1 - S P y), y'.z
// where the stepwise solver has five launches: 31.9 and 15.6-16.7 us an iteration at 3,072 cells (77,184 rows),
// of which the exchanges with the loads after them take ~12.
#include <algorithm>
#include <climits>

#include "nfx_el_grid.h"
#include "nfx_el_twogrid.h"

namespace nfx {
namespace {

constexpr int kT = kGridThreads;
constexpr int kElGridAgg = 128;    // aggregates (the coarse vector and its pieces are in LDS)
constexpr int kElGridCells = kT / 30;  // cells of a block: 5 blocks x 6 components, a thread each

struct ElGridArgs {
  int n, n_blocks, nblk, maxit, lds;
  const int32_t *brp, *bci;
  const float* bva;
  nfx_elasticity_tg pc;
  const float* rhs;
  float *x, *vec;
  double tol;
  grid_word* slots;
  GridResult* res;
};

__global__ __launch_bounds__(kT) void k_el_grid(ElGridArgs a) {
  extern __shared__ __align__(16) char lds[];
  __shared__ double sh_post[2][kT / 64], sh_part[2][kT / 64];
  __shared__ int sh_good[2][kT / 64], scan[kT / 64];
  __shared__ MinresState sts[2];
  constexpr int LANES = 8;
  const int t = threadIdx.x, B = a.nblk, rank = blockIdx.x;
  const nfx_elasticity_tg& pc = a.pc;
  const int E = pc.n_cells, ns = pc.n_s, nu = pc.n_u, NA = pc.n_agg, nc = 6 * NA;
  GridSync g{a.slots, B, rank, 0, sh_post, sh_part, sh_good};

  const int f0 = (int)((int64_t)(ns / 9) * rank / B), nf = (int)((int64_t)(ns / 9) * (rank + 1) / B) - f0;
  const int m0 = (int)((int64_t)E * rank / B), nC = (int)((int64_t)E * (rank + 1) / B) - m0;
  const int RB = 3 * nf + 2 * nC, R = 3 * RB, Rf = 9 * nf;  // block rows, rows, stress rows

  // LDS: block row starts and numbers | vectors | face inverses | a word per thread (r, x1, products, t)
  // | pieces of the aggregates, coarse vector, the values needed | columns (16 bits) | z | values | list
  int* rowp = reinterpret_cast<int*>(lds);
  int* bid = rowp + RB + 1;
  float *r1 = reinterpret_cast<float*>(bid + RB), *r2 = r1 + R, *zc = r2 + R, *zp = zc + R, *ys = zp + R;
  float *dl = ys + R, *ra = dl + 9 * Rf, *xa = ra + kT, *sa = xa + kT;
  float *pv = sa + kT, *cv = pv + 6 * (kElGridAgg + kGridMaxBlocks), *yl = cv + 6 * kElGridAgg;
  int* pp = reinterpret_cast<int*>(yl + 6 * kElGridAgg);  // positions where pieces start
  int* pa = pp + kElGridAgg + kGridMaxBlocks;             // first piece of each aggregate
  int* need = pa + kElGridAgg + 1;                        // aggregates whose coarse values are needed
  int* slot = need + kElGridAgg;                          // their places in yl
  unsigned short* idx = reinterpret_cast<unsigned short*>(slot + kElGridAgg);
  const int64_t fixed = reinterpret_cast<char*>(idx) - lds;
  bool good = __syncthreads_and(NA <= kElGridAgg && 30 * nC <= kT && fixed + 4 <= a.lds);

  // the thread's item: block b (0 own, 1 + k neighbour k), component i, cell p; row is that of component i
  // of the block's cell
  const int items = 30 * nC, p = nC ? t % nC : 0, bi = nC ? t / nC : 0, b = bi / 6, i = bi % 6;
  const bool item = good && t < items, own = item && b == 0;
  int row = -1, ag = 0;
  float W[6] = {}, S[6] = {};
  constexpr int kPre = 4;
  int nz = 0, H = 0, nP = 0, nN = 0, col[kPre] = {};
  int* list = nullptr;
  float *zh = nullptr, *val = nullptr;
  if (good) {
    if (t < kElGridAgg) slot[t] = 0;
    __syncthreads();
    bool fine = true;
    if (item) {
      const int m = m0 + p, q = b ? pc.nbr[(int64_t)m * 4 + b - 1] : m;
      if (q >= 0) {
        fine = q < E;
        const int c = fine ? pc.agg_mem[q] : -1;
        ag = fine ? pc.agg_of[q] : 0;
        fine = fine && c >= 0 && c < E && ag >= 0 && ag < NA;
        if (fine) {
          row = (int)el_row(c, ns, nu, i);
#pragma unroll
          for (int j = 0; j < 6; ++j) {
            W[j] = pc.winv[(int64_t)(i * 6 + j) * E + q];
            S[j] = pc.sblk[(int64_t)(36 * b + i * 6 + j) * E + m];
          }
          slot[ag] = 1;
        }
      }
    }
    if (t < NA) fine = fine && pc.agg_ptr[t] >= 0 && pc.agg_ptr[t] <= pc.agg_ptr[t + 1];
    if (t == 0) fine = fine && pc.agg_ptr[0] == 0 && pc.agg_ptr[NA] == E;
    good = __syncthreads_and(fine);
  }
  if (good) {
    // pieces in order of position: an aggregate starts one, and a block within it; needed aggregates
    int* ptr = reinterpret_cast<int*>(pv);
    if (t <= NA) ptr[t] = pc.agg_ptr[t];
    __syncthreads();
    if (t == 0) {
      int r = 1, n = 0;
      for (int x = 0; x < NA; ++x) {
        const int p0 = ptr[x], p1 = ptr[x + 1];
        pa[x] = n;
        if (p1 > p0) pp[n++] = p0;
        for (; r < B && (int)((int64_t)E * r / B) < p1; ++r) {
          const int s = (int)((int64_t)E * r / B);
          if (s > p0 && s > pp[n - 1]) pp[n++] = s;
        }
      }
      pa[NA] = n;
      int k = 0;
      for (int x = 0; x < NA; ++x)
        if (slot[x]) {
          need[k] = x;
          slot[x] = k++;
        }
      scan[0] = n;
      scan[1] = k;
    }
    __syncthreads();
    nP = uniform(scan[0]);
    nN = uniform(scan[1]);
    ag = 6 * slot[ag];
    __syncthreads();

    // block rows and the starts of their blocks
    const int run = (RB + kT - 1) / kT, i0 = min(RB, t * run), i1 = min(RB, i0 + run);
    int cnt = 0;
    for (int x = i0; x < i1; ++x) {
      int r = 3 * f0 + x;
      if (x >= 3 * nf) {
        const int c = pc.agg_mem[m0 + (x - 3 * nf) / 2];
        r = ((x - 3 * nf) & 1 ? (ns + nu) / 3 : ns / 3) + c;
      }
      bid[x] = r;
      cnt += a.brp[r + 1] - a.brp[r];
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
    for (int x = i0; x < i1; ++x) {
      rowp[x] = pre;
      pre += a.brp[bid[x] + 1] - a.brp[bid[x]];
    }
    if (t == 0) rowp[RB] = nz;
    const int nb = a.n / 3;
    const int64_t base = fixed + 4 * (((int64_t)nz + 1) / 2), nw = (nb + 31) >> 5;
    good = __syncthreads_and(base + 8 * nw <= a.lds);
    if (good) {
      unsigned* bits = reinterpret_cast<unsigned*>(lds + base);
      int* before = reinterpret_cast<int*>(bits + nw);
      const auto start = [&](int x) { return a.brp[bid[x]]; };
      H = uniform(grid_columns<LANES>(a.bci, nb, RB, rowp, start, bits, before, scan));
      good = H <= 65535 && base + 8 * nw + 4 * (int64_t)H <= a.lds && base + 16 * (int64_t)H <= a.lds;
      if (good) {
        list = reinterpret_cast<int*>(lds + a.lds) - H;
        grid_renumber<LANES>(a.bci, nb, RB, rowp, start, bits, before, list, idx);
        zh = reinterpret_cast<float*>(lds + base);
#pragma unroll
        for (int u = 0; u < kPre; ++u) {
          const int e = t + u * kT;
          col[u] = e < 3 * H ? 3 * list[e / 3] + e % 3 : 0;
        }
        __syncthreads();
        if (base + 12 * (int64_t)H + (3 * H > kPre * kT ? 4 * (int64_t)H : 0) + 36 * (int64_t)nz <= a.lds) {
          val = zh + 3 * H;
          for (int x = t / LANES; x < RB; x += kT / LANES) {
            const int s = start(x);
            for (int j = t % LANES, len = rowp[x + 1] - rowp[x]; j < len; j += LANES)
#pragma unroll
              for (int k = 0; k < 9; ++k) val[9 * (rowp[x] + j) + k] = a.bva[(int64_t)k * a.n_blocks + s + j];
          }
        }
        for (int x = t; x < 9 * Rf; x += kT) dl[x] = pc.dinv[(int64_t)f0 * 81 + x];
      }
    }
  }
  double sum;
  grid_post(g, t == 0 && !good ? 1.0 : 0.0);
  bool ok = grid_wait(g, sum);
  if (!ok || sum != 0) {
    if (t == 0) atomicMax(&a.res->status, ok ? 1 : 2);
    return;
  }

  // exchanged vectors; w of the last two steps (own rows only) lies beside them
  const int64_t N = a.n;
  float *Z = a.vec, *Y = a.vec + 2 * N, *RR = a.vec + 3 * N, *CV = a.vec + 5 * N, *wa = a.vec + 6 * N,
        *wb = a.vec + 7 * N;
  int p0 = 0, myP = 0;  // the block's pieces: one starts at m0
  while (p0 < nP && pp[p0] < m0) ++p0;
  while (p0 + myP < nP && pp[p0 + myP] < m0 + nC) ++myP;
  p0 = uniform(p0);
  myP = uniform(myP);
  const auto grow = [&](int x) { return 3 * bid[x / 3] + x % 3; };
  double acc = 0;
  int k = 0;
  for (; ok; ++k) {
    float c = 0.f;
    if (k == 0) {
      for (int x = t; x < R; x += kT) {
        const int r = grow(x);
        const float v = a.rhs[r];
        r1[x] = r2[x] = v;
        zc[x] = zp[x] = wa[r] = wb[r] = a.x[r] = 0.f;
        if (x >= Rf) grid_store(RR + N + r, v);
      }
    } else {
      const float* zg = Z + (int64_t)(k & 1) * N;
      float zl[kPre];
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * kT < 3 * H) zl[u] = grid_load(zg + col[u]);
      const double beta = sqrt(sum > 0 ? sum : 0);
      const float s = (float)(1.0 / beta), ratio = k == 1 ? 0.f : (float)(beta / sts[(k + 1) & 1].beta);
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * kT < 3 * H) zh[t + u * kT] = zl[u];
      for (int e = t + kPre * kT; e < 3 * H; e += kT) zh[e] = grid_load(zg + 3 * list[e / 3] + e % 3);
      __syncthreads();
      for (int x = t / LANES; x < RB; x += kT / LANES) {
        float s0 = 0.f, s1 = 0.f, s2 = 0.f;
        const int j0 = rowp[x], len = rowp[x + 1] - j0;
        const int at = val ? 0 : a.brp[bid[x]];
        for (int j = t % LANES; j < len; j += LANES) {
          const float* z = zh + 3 * (int)idx[j0 + j];
          float v[9];
          if (val) {
#pragma unroll
            for (int e = 0; e < 9; ++e) v[e] = val[9 * (j0 + j) + e];
          } else {
#pragma unroll
            for (int e = 0; e < 9; ++e) v[e] = a.bva[(int64_t)e * a.n_blocks + at + j];
          }
          s0 += v[0] * z[0] + v[1] * z[1] + v[2] * z[2];
          s1 += v[3] * z[0] + v[4] * z[1] + v[5] * z[2];
          s2 += v[6] * z[0] + v[7] * z[1] + v[8] * z[2];
        }
        s0 = lanes_total<LANES>(s0);
        s1 = lanes_total<LANES>(s1);
        s2 = lanes_total<LANES>(s2);
        const int l = t % LANES;
        if (l < 3) ys[3 * x + l] = l == 0 ? s0 : l == 1 ? s1 : s2;
      }
      __syncthreads();
      acc = 0;
      for (int x = t; x < R; x += kT) {
        const float y = s * ys[x] - ratio * r1[x];
        r1[x] = y;
        if (x >= Rf) grid_store(Y + grow(x), y);
        acc += (double)(s * zc[x]) * (double)y;
      }
      grid_post(g, acc);
      // the rotation, and every kGridCheck iterations the test of the estimate after k - 1 of them
      MinresState st;
      minres_scalars(sts[(k + 1) & 1], st, beta, k == 1);
      if (t == 0) sts[k & 1] = st;  // read after the next barrier only
      const bool last = !(beta > 0) || k - 1 >= a.maxit ||
                        (k > 1 && (k - 1) % kGridCheck == 0 && st.phibar <= a.tol * st.beta1);
      const MinresStep step(st);
      for (int x = t; x < R; x += kT) {
        if (k > 1) {
          const int r = grow(x);
          const float w1 = wb[r], w = step.w(zp[x], wa[r], w1);
          wa[r] = w1;
          wb[r] = w;
          a.x[r] += step.phi * w;
        }
        zp[x] = zc[x];
      }
      if (last) break;
      ok = grid_wait(g, sum);
      if (!ok) break;
      if (t == 0) sts[k & 1].alfa = sum;
      c = (float)(sum / sts[k & 1].beta);
      for (int x = t; x < R; x += kT) {
        const float y = r1[x] - c * r2[x];
        r1[x] = r2[x];
        r2[x] = y;
        if (x >= Rf) grid_store(RR + (int64_t)((k + 1) & 1) * N + grow(x), y);
      }
    }
    __syncthreads();

    // z of iteration k + 1 from y' (r2); RR[(k + 1) & 1] holds y' of this step, RR[k & 1] that before it
    float* zn = Z + (int64_t)((k + 1) & 1) * N;
    float r = 0.f, x1 = 0.f, t1 = 0.f;
    if (own) {
      r = r2[Rf + 6 * p + i];
    } else if (row >= 0) {  // what a neighbour published: y and the r2 before it
      r = k ? grid_load(Y + row) - c * grid_load(RR + (int64_t)(k & 1) * N + row) : a.rhs[row];
    }
    if (item) ra[t] = r;
    __syncthreads();
    const int at = 6 * b * nC + p;  // the items of the same block of S
    if (item) {
#pragma unroll
      for (int j = 0; j < 6; ++j) x1 += W[j] * ra[at + j * nC];
      xa[t] = x1;
    }
    __syncthreads();
    if (item) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 6; ++j) s += S[j] * xa[at + j * nC];
      sa[t] = s;
    }
    __syncthreads();
    if (own) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < 5; ++q) s += sa[t + 6 * q * nC];
      t1 = r - s;
      ra[t] = t1;  // component i of cell p at i nC + p
    }
    __syncthreads();
    // the block's pieces: a wave per piece and component
    for (int w = t >> 6; w < 6 * myP; w += kT / 64) {
      const int q = p0 + w / 6, e = w % 6;
      const int s = pp[q] - m0, s1 = min(nC, (q + 1 < nP ? pp[q + 1] : E) - m0);
      double v = 0;
      for (int x = s + (t & 63); x < s1; x += 64) v += (double)ra[e * nC + x];
      v = wave_total(v);
      if ((t & 63) == 0) grid_store(CV + (int64_t)pp[q] * 6 + e, (float)v);
    }
    grid_post(g, 0.0);
    acc = 0;
    for (int x = t; x < Rf; x += kT) {
      const int f = x - x % 9;
      float z = 0.f;
#pragma unroll
      for (int j = 0; j < 9; ++j) z += dl[9 * x + j] * r2[f + j];
      grid_store(zn + grow(x), z);
      zc[x] = z;
      acc += (double)r2[x] * (double)z;
    }
    // the first entries of the first coarse row that the thread helps with, during the wait
    constexpr int kAi = 24;
    float ai[kAi];
    const float* row_a = t / 16 < 6 * nN ? pc.ainv + (int64_t)(6 * need[t / 16 / 6] + t / 16 % 6) * nc : nullptr;
#pragma unroll
    for (int u = 0; u < kAi; ++u) ai[u] = row_a && t % 16 + 16 * u < nc ? row_a[t % 16 + 16 * u] : 0.f;
    ok = grid_wait(g, sum);
    if (!ok) break;
    for (int x = t; x < 6 * nP; x += kT) pv[x] = grid_load(CV + (int64_t)pp[x / 6] * 6 + x % 6);
    __syncthreads();
    for (int x = t; x < nc; x += kT) {
      float v = 0.f;
      for (int q = pa[x / 6]; q < pa[x / 6 + 1]; ++q) v += pv[6 * q + x % 6];
      cv[x] = v;
    }
    __syncthreads();
    for (int x = t / 16; x < 6 * nN; x += kT / 16) {
      float v = 0.f;
      int l = t % 16;
      if (x == t / 16) {
#pragma unroll
        for (int u = 0; u < kAi; ++u, l += 16)
          if (l < nc) v += ai[u] * cv[l];
      } else {
        row_a = pc.ainv + (int64_t)(6 * need[x / 6] + x % 6) * nc;
      }
#pragma unroll 8
      for (; l < nc; l += 16) v += row_a[l] * cv[l];
      v = lanes_total<16>(v);
      if (t % 16 == 0) yl[x] = v;
    }
    __syncthreads();
    if (item) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 6; ++j) s += S[j] * yl[ag + j];
      sa[t] = s;
    }
    __syncthreads();
    if (own) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < 5; ++q) s += sa[t + 6 * q * nC];
      ra[t] = t1 - s;
    }
    __syncthreads();
    if (own) {
      float z = x1 + yl[ag + i];
#pragma unroll
      for (int j = 0; j < 6; ++j) z += W[j] * ra[p + j * nC];
      z *= pc.psign;
      grid_store(zn + row, z);
      zc[Rf + 6 * p + i] = z;
      acc += (double)r * (double)z;
    }
    grid_post(g, acc);
    ok = grid_wait(g, sum);
  }
  if (!ok) {
    if (t == 0) atomicMax(&a.res->status, 2);
    return;
  }
  if (rank == 0 && t == 0) a.res->iters = k > 1 ? k - 1 : 1;
}

}  // namespace

int el_grid_capacity() {
  int per_cu = 0;
  if (hipFuncSetAttribute((const void*)k_el_grid, hipFuncAttributeMaxDynamicSharedMemorySize, kGridLdsBytes) !=
          hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_el_grid, kT, kGridLdsBytes) !=
          hipSuccess ||
      per_cu < 1) {
    (void)hipGetLastError();
    return 0;
  }
  return minres_grid_capacity();
}

// At most 12 cells a block as long as there are CUs (us an iteration at 3,072 cells: 16.7 with 256 blocks,
// 19.0 with 128, 20.5 with 96, 31.9 stepwise; at 750 cells 14.0 with 64, 14.3 with 128, 25.3 stepwise;
// at 162 cells 13.5 with 16, 23.5 stepwise), more where they have to (6,000 cells: 31.2, 39.5 stepwise).
int el_grid_blocks(int max_blocks, const nfx_elasticity_tg* pc, int n_blocks) {
  if (pc->n_agg > kElGridAgg || pc->n_s % 9 || pc->n_u != 3 * pc->n_cells) return 0;
  const int n = pc->n_s + 2 * pc->n_u;
  const auto cells = [&](int nblk) { return (pc->n_cells + nblk - 1) / nblk; };
  // columns, 28 bytes a row and 36 for a face inverse's, beside what is fixed
  const auto bytes = [&](int nblk) { return (2 * (int64_t)n_blocks + 64 * (int64_t)n) / nblk + (48 << 10); };
  int nblk = 16;
  while (2 * nblk <= max_blocks && (cells(nblk) > 12 || bytes(nblk) > kGridLdsBytes)) nblk *= 2;
  return nblk <= max_blocks && cells(nblk) <= kElGridCells && bytes(nblk) <= kGridLdsBytes ? nblk : 0;
}

int el_grid_solve(MinresGrid* g, int nblk, int n, int n_blocks, const int32_t* brp, const int32_t* bci,
                  const float* bva, const nfx_elasticity_tg* pc, const float* rhs, float* x, float* vec, double tol,
                  int maxit, int* iters, int* status, hipStream_t st) {
  *status = 1;
  NFX_CHECK(grid_clear(g->slots, nblk, g->res, 1, st));
  ElGridArgs a{n, n_blocks, nblk, maxit, kGridLdsBytes, brp, bci, bva, *pc, rhs, x, vec, tol, g->slots, g->res};
  void* args[] = {&a};
  bool ran = false;
  NFX_CHECK(grid_launch(&g->control, (const void*)k_el_grid, nblk - (g->control.absent ? 1 : 0), args, st, &ran));
  if (!ran) return NFX_OK;
  NFX_CHECK_HIP(hipMemcpyAsync(g->h_res, g->res, sizeof(GridResult), hipMemcpyDeviceToHost, st));
  NFX_CHECK_HIP(hipStreamSynchronize(st));
  *iters = g->h_res->iters;
  *status = g->h_res->status;
  return NFX_OK;
}

}  // namespace nfx
