// Newton-Schulz, normaliser and update of thin matrices (smaller dim m at most 32), in fp64 on the m x m side.
//
// With A = X X^T every iterate is a polynomial of A times X, so the five iterations need X twice only: once for A, once for
// Q X.  In fp32 that loses the small singular directions -- the chained A inherits the rounding of the first one, which the
// polynomial amplifies by c0^2 an iteration (k_ns_hf.h) -- in fp64 a run of a few does not: products of fp32 values are exact, A is
// off by 1e-16 of its largest eigenvalue, and five iterations leave 1e-10 of a direction.  What of it is not symmetric grows faster,
// 23-fold an iteration (the products take a matrix for its transpose): six iterations are the most that the usual coefficients
// allow.  More are taken in runs (thin_runs, RUNS) that each form the Gram matrix again, from X in fp32.  Every matrix of a run is a
// multiple of the identity and the rest (B = c0 I + P, Q = q0 I + M), the multiple applied by itself: equal rows of X stay equal to
// the bit, as in the formula, and leave no difference for later runs to amplify.  32 x 500 of ones, off by (of the RMS) at 8, 12,
// 20 iterations: one run 2e-6, 6, NaN; runs of six 1e-7 at most; the formula in fp32 1e-5.  And on m x m matrices of at most two
// tiles of v_mfma_f64_16x16x4_f64 a side the fp64 pipe is fast enough.  So a block takes a slab of columns through
//   G += X X^T (fp32 values widened);  [the blocks of a matrix meet once and add their G in slab order]
//   A = G / (sqrt(tr G) + eps)^2;  B = c2 A A + c1 A + c0 I,  Q <- B Q,  A <- B A B  (every block for itself)
//   sum of squares of the result = tr(Q A Q);  X <- Q X / (sqrt(tr G) + eps), normalised, applied to the parameter.
// The chain that k_ns_small has for larger ones, with a class for these, passed over X eight times and met five times.  What
// bounds this: the latency of two passes of loads, and five iterations of three dependent products (0.3 to 0.5 us each with its
// barriers).  Whole ELO-CELO2 steps, then / now: three thousand odd tensors 2.72 / 2.19 ms (one launch of 651 us, now two of 64 and 75), one and
// sixty-four of 32 x 32768 294 / 135 and 2072 / 1441 us, sixteen of 16 x 8192 455 / 131, one of 32 x 1024 93 / 98.  Against the
// formula in fp64 the result is off by the roundings of its last three operations (2e-8 to 7e-7 of its RMS; 2e-7 to 2e-5 in fp32 products).
//
// A matrix of at most eight rows is folded: the sixteen rows of a tile are its rows (rounded up to a power of two) of U columns --
// neighbours where a column's entries lie next to each other in memory, n / U apart where a row's do -- G the sum of the U blocks
// on the tile's diagonal and Q repeated U times there.  (1 x 65536, sixteen of them: 107 us unfolded, 41 folded.)
//
// Layouts of v_mfma_f64_16x16x4_f64 (lane l): A operand row l % 16, reduction l / 16; B operand column l % 16, reduction
// l / 16; D register r row 4 r + l / 16, column l % 16.  All m x m matrices are symmetric, so one LDS copy [row][col] serves
// as either operand.  Which of an operand's reduction slots stands for which row of X is free as long as both sides agree:
// memory order of X decides.
#pragma once

#include "k_ns_small.h"

namespace pylo {

typedef double v4d __attribute__((ext_vector_type(4)));

template <int MT>   // 16 x 16 tiles a side
struct ThinDims {
  static constexpr int MP = 16 * MT, PD = MP + 2, NT = MT * (MT + 1) / 2;
  static constexpr int kMat = MP * PD;                                  // doubles
  static constexpr int kRed = kWaves * NT * 256;                        // the waves' partial G, in the matrices' place
  static constexpr int kLds = 8 * (3 * kMat > kRed ? 3 * kMat : kRed);
  static constexpr int kGroup = 16;                                     // columns a wave takes at a time
};
constexpr int kThinChunk = 64;         // columns of a chunk (NsSmall::chunks): a group of each of the four waves

// A launch takes a run of iterations: all of them, or where they are too many for one Gram matrix (thin_runs) the first, the
// next, ..., the last (RUNS).  Runs but the last leave X <- Q X in place, rounded to fp32, runs but the first start from it as it is.
struct ThinStep {
  double c0, c1, c2, eps;
  int iters, first, last;
};

// A matrix has at most 32 x 65536 elements: 32-bit offsets.
__device__ __forceinline__ float thin_at(const float* p, int i) { return *(const gfloat*)((const gchar*)p + (unsigned)i * 4u); }
__device__ __forceinline__ void thin_put(float* p, int i, float v) { *(gfloat*)((gchar*)p + (unsigned)i * 4u) = v; }

template <int MT, bool RUNS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(MT == 1 ? 5 : 4))) void k_ns_thin(
    const NsSmall* __restrict__ mats, const NsSmallItem* __restrict__ items, const TDesc* __restrict__ descs,
    const PyloTensorArgs* __restrict__ dyn, float* __restrict__ part, int* __restrict__ sync, ThinStep st, int orth_call,
    int* __restrict__ tickets) {
  using D = ThinDims<MT>;
  constexpr int K = 4 * MT;                       // reduction steps of four over the rows
  extern __shared__ __attribute__((aligned(16))) char lds_[];
  typedef PYLO_LDS double ldouble;
  ldouble* const s0 = (ldouble*)(PYLO_LDS char*)lds_;
  ldouble *const s1 = s0 + D::kMat, *const s2 = s1 + D::kMat;
  __shared__ double red[kWaves];
  __shared__ int s_flag;
  int item = (int)blockIdx.x;
  if (tickets != nullptr) {                       // see k_ns_small: blocks take their places in the order they start
    if (threadIdx.x == 0) s_flag = __hip_atomic_fetch_add(tickets, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    item = __builtin_amdgcn_readfirstlane(s_flag);
    if (item == (int)gridDim.x - 1 && threadIdx.x == 0)
      __hip_atomic_store(tickets, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
  }
  const NsSmallItem it = items[item];
  const NsSmall q = mats[it.mat];
  const PyloTensorArgs a = dyn[q.tensor];
  if (a.grad == nullptr) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  float* const x0 = a.step_out + q.elem_off;
  const int m = q.m, n = q.n;
  const bool tall = q.tall;
  const int fold = MT == 1 ? q.fold : 0, nv = (n + (1 << fold) - 1) >> fold;   // columns are folded columns from here on
  const int n0 = it.slab * q.chunks * kThinChunk, n1 = min(nv, n0 + q.chunks * kThinChunk);
  // where row k of the tile sits in column 0, how far it is from a column to the next, and the column its part ends at
  const int step_c = tall ? m << fold : 1;
  auto row_at = [&](int k, int& lim) {
    const int u = MT == 1 ? k >> (4 - fold) : 0, row = MT == 1 ? k & ((16 >> fold) - 1) : k;
    lim = row >= m ? 0 : MT == 2 ? n1 : min(n1, tall ? (n - u + (1 << fold) - 1) >> fold : n - u * nv);
    return tall ? u * m + row : row * n + u * nv;
  };
  const bool orth = orth_call && (a.flags & kArgOrthogonalize);
  const bool first = !RUNS || st.first, last_run = !RUNS || st.last;
  if (!orth && !last_run) return;
  bool good = true;

  // ---- G over the block's columns.  Lane: row 16 t + lo; the four columns of slot hi are neighbours where a row's entries
  // lie next to each other in memory, and one of each four where a column's do.
  v4d g[D::NT];
#pragma unroll
  for (int t = 0; t < D::NT; ++t) g[t] = v4d{0.0, 0.0, 0.0, 0.0};
  int g_at[MT], g_lim[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) g_at[t] = row_at(16 * t + lo, g_lim[t]);
  auto load_rows = [&](int c, float (&x)[MT][4]) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int col = c + (tall ? 4 * i + hi : 4 * hi + i);
        x[t][i] = 0.0f;
        if (col < g_lim[t]) x[t][i] = thin_at(x0, g_at[t] + col * step_c);
      }
  };
  {
    constexpr int kStep = kWaves * D::kGroup;
    float x[MT][4], nx[MT][4];
    int c = n0 + wave * D::kGroup;
    if (c < n1) load_rows(c, x);
    for (; c < n1; c += kStep) {
      if (c + kStep < n1) load_rows(c + kStep, nx);
      double y[MT][4];
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) y[t][i] = (double)x[t][i];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int p = 0;
#pragma unroll
        for (int ti = 0; ti < MT; ++ti)
#pragma unroll
          for (int tj = ti; tj < MT; ++tj, ++p) g[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[ti][i], y[tj][i], g[p], 0, 0, 0);
      }
      if (c + kStep < n1) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) x[t][i] = nx[t][i];
      }
    }
  }
  // thread e holds element (register e / 64, lane e % 64) of every tile, summed over the waves and then over the slabs
  double sum[D::NT];
#pragma unroll
  for (int t = 0; t < D::NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) s0[((wave * D::NT + t) * 4 + r) * 64 + lane] = g[t][r];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < D::NT; ++t) {
    sum[t] = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) sum[t] += s0[(w * D::NT + t) * 256 + threadIdx.x];
  }
  if (q.slabs > 1) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const SmBuf pbuf = sm_buffer(part + q.part, q.slabs * D::NT * 2048);
    // entries outside the matrix are zero: nobody leaves or fetches them
    bool in[D::NT];
    {
      int p = 0;
#pragma unroll
      for (int ti = 0; ti < MT; ++ti)
#pragma unroll
        for (int tj = ti; tj < MT; ++tj, ++p) in[p] = fold > 0 || (16 * ti + 4 * wave + hi < m && 16 * tj + lo < m);
    }
#pragma unroll
    for (int t = 0; t < D::NT; ++t)
      if (in[t])
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, sum[t]), pbuf,
                                              (it.slab * D::NT + t) * 2048 + (int)threadIdx.x * 8, 0, kSmAgent);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // they have been performed
    good = sm_meet(sync + q.sync, q.slabs, &s_flag);
#pragma unroll
    for (int t = 0; t < D::NT; ++t) {
      if (!in[t]) continue;
      sum[t] = 0.0;
      constexpr int kAhead = 16;                       // slabs whose values are asked for together
      for (int b0 = 0; b0 < q.slabs; b0 += kAhead) {
        double v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
          v[u] = b0 + u < q.slabs ? __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(
                                                                   pbuf, ((b0 + u) * D::NT + t) * 2048 + (int)threadIdx.x * 8, 0, kSmAgent))
                                  : 0.0;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) sum[t] += v[u];
      }
    }
  }
  __syncthreads();   // the waves' partial sums have been read: the matrices take their place
  {
    const int r = wave;
    int p = 0;
#pragma unroll
    for (int ti = 0; ti < MT; ++ti)
#pragma unroll
      for (int tj = ti; tj < MT; ++tj, ++p) {
        const int row = 16 * ti + 4 * r + hi, col = 16 * tj + lo;
        s0[row * D::PD + col] = sum[p];
        if (ti != tj) s0[col * D::PD + row] = sum[p];
      }
  }
  __syncthreads();
  if (MT == 1 && fold > 0) {   // the blocks on the diagonal, added up; zero outside the first
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15, w = 4 - fold;
    double t = 0.0;
    if (row < m && col < m)
      for (int u = 0; u < 1 << fold; ++u) t += s0[((u << w) + row) * D::PD + (u << w) + col];
    __syncthreads();
    s0[row * D::PD + col] = t;
    __syncthreads();
  }
  const double tr = wave_sum(lane < D::MP ? s0[lane * D::PD + lane] : 0.0);   // rows past m are zero

  // ---- the m x m matrices.  Wave w < MT^2 owns tile (w / MT, w % MT).
  double ss = tr, xs = 1.0, q0 = 1.0;
  if (orth) {
    const int ti = wave / MT, tj = wave % MT;
    const bool own = wave < MT * MT;
    auto prod = [&](const ldouble* pa, const ldouble* pb) {
      v4d d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < K; ++s)
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[(16 * ti + lo) * D::PD + 4 * s + hi], pb[(16 * tj + lo) * D::PD + 4 * s + hi], d, 0, 0, 0);
      return d;
    };
    auto put = [&](ldouble* p, const v4d& d) {
#pragma unroll
      for (int r = 0; r < 4; ++r) p[(16 * ti + 4 * r + hi) * D::PD + 16 * tj + lo] = d[r];
    };
    if (first) xs = 1.0 / (sqrt(tr) + st.eps);
    v4d A, A0, Q;
    if (own) {
#pragma unroll
      for (int r = 0; r < 4; ++r) A[r] = s0[(16 * ti + 4 * r + hi) * D::PD + 16 * tj + lo] * (xs * xs);
    }
    A0 = A;
    __syncthreads();
    if (own) put(s0, A);
    __syncthreads();
    for (int i = 0; i < st.iters; ++i) {
      const bool last = i == st.iters - 1;
      v4d B, T;                              // RUNS: P, and M in Q's place
      if (own) {
        B = prod(s0, s0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * ti + 4 * r + hi, col = 16 * tj + lo;
          B[r] = st.c2 * B[r] + st.c1 * A[r] + (!RUNS && row == col && row < m ? st.c0 : 0.0);
        }
        put(s1, B);
      }
      __syncthreads();
      if (own) {
        Q = i > 0 ? RUNS ? prod(s2, s1) : prod(s1, s2) : B;        // B Q
        if (!last) T = prod(s0, s1);         // A B
        if constexpr (RUNS) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (i > 0) Q[r] += st.c0 * s2[(16 * ti + 4 * r + hi) * D::PD + 16 * tj + lo] + q0 * B[r];
            if (!last) T[r] += st.c0 * A[r];
          }
        }
      }
      if constexpr (RUNS) q0 *= st.c0;
      __syncthreads();
      if (own) {
        put(s2, Q);
        if (!last) put(s0, T);
      }
      __syncthreads();
      if (!last) {
        if (own) {                           // B A B
          A = RUNS ? prod(s0, s1) : prod(s1, s0);
          if constexpr (RUNS) {
#pragma unroll
            for (int r = 0; r < 4; ++r) A[r] += st.c0 * T[r];
          }
        }
        __syncthreads();
        if (own) put(s0, A);
        __syncthreads();
      }
    }
    // ||Q X0||^2 = tr(Q A0 Q)
    if (own) put(s0, A0);
    __syncthreads();
    double s = 0.0;
    if (own) {
      const v4d t = prod(s2, s0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (RUNS) s += (t[r] + q0 * A0[r]) * (16 * ti + 4 * r + hi == 16 * tj + lo ? Q[r] + q0 : Q[r]);
        else s += t[r] * Q[r];
      }
    }
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    ss = (red[0] + red[1]) + (red[2] + red[3]);
    if (RUNS && !good) xs = __builtin_nan("");
  }
  // ---- step = X * rsqrt(1e-9 + mean X^2) * rmsmult; p <- p - lr (step + wd p)
  const float rm = a.step_mult, wd = a.weight_decay, nlr = -a.lr;
  const float sc = good ? rsq(1e-9f + (float)(ss / ((double)m * (double)n))) : __builtin_nanf("");
  const int store = descs[q.tensor].store;
  float* const pb = a.param + q.elem_off;
  if (!orth) {
    // the raw step as it is
    for (int e = threadIdx.x; e < D::MP * (n1 - n0); e += kThreads) {
      int lim;
      const int k = tall ? e % D::MP : e / (n1 - n0), c = n0 + (tall ? e / D::MP : e % (n1 - n0)), at = row_at(k, lim);
      if (c >= lim) continue;
      const long long i = q.elem_off + at + c * step_c;
      const float w = load_stored(a.param, i, store);
      store_stored(a.param, i, store, fmaf(nlr, (thin_at(x0, at + c * step_c) * sc) * rm + wd * w, w));
    }
  } else {
    // Q in the slots' order: rows 16 t + 4 j + hi of step 4 t + j, or 16 t + 4 hi + j where a lane's rows lie next to each other
    auto slot = [&](int s) { return 16 * (s >> 2) + (tall ? 4 * hi + (s & 3) : 4 * (s & 3) + hi); };
    double qf[MT][K];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int s = 0; s < K; ++s) {
        int i = 16 * t + lo, j = slot(s);
        bool same = true;
        if (MT == 1 && fold > 0) {
          const int w = 4 - fold;
          same = i >> w == j >> w;
          i &= (1 << w) - 1;
          j &= (1 << w) - 1;
        }
        qf[t][s] = same ? s2[i * D::PD + j] * xs : 0.0;
      }
    int x_at[MT == 1 ? K : 1], x_lim[MT == 1 ? K : 1];
    if constexpr (MT == 1)
#pragma unroll
      for (int s = 0; s < K; ++s) x_at[s] = row_at(slot(s), x_lim[s]);
    auto load_cols = [&](int c, float (&x)[K]) {
#pragma unroll
      for (int s = 0; s < K; ++s) {
        const int col = c + lo;
        x[s] = 0.0f;
        if constexpr (MT == 1) {
          if (col < x_lim[s]) x[s] = thin_at(x0, x_at[s] + col * step_c);
        } else {
          const int row = slot(s);
          if (row < m && col < n1) x[s] = thin_at(x0, tall ? col * m + row : row * n + col);
        }
      }
    };
    // where register r of output tile t sits: columns by rows where a column's entries lie next to each other (X^T Q), else rows by
    // columns
    // (rows 4 r + hi of a tile of one: the slots' own)
    auto place = [&](int c, int t, int r, int& idx) {
      if (tall) {
        const int col = c + 4 * r + hi;
        idx = g_at[t] + col * step_c;
        return col < g_lim[t];
      }
      if constexpr (MT == 1) {
        idx = x_at[r] + c + lo;
        return c + lo < x_lim[r];
      }
      const int row = 16 * t + 4 * r + hi, col = c + lo;
      idx = row * n + col;
      return row < m && col < n1;
    };
    constexpr int kStep = kWaves * D::kGroup;
    float x[K], nx[K];
    int c = n0 + wave * D::kGroup;
    if (c < n1) load_cols(c, x);
    for (; c < n1; c += kStep) {
      if (c + kStep < n1) load_cols(c + kStep, nx);
      float w[MT][4];
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int idx;
          w[t][r] = 0.0f;
          if (last_run && place(c, t, r, idx)) w[t][r] = store == 0 ? thin_at(pb, idx) : load_stored(a.param, q.elem_off + idx, store);
        }
      v4d d[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) d[t] = v4d{0.0, 0.0, 0.0, 0.0};
      if constexpr (RUNS) {
#pragma unroll
        for (int s = 0; s < K; ++s) {
          const double y = (double)x[s];
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            const double e = 16 * t + lo == slot(s) ? q0 * xs : 0.0;
            d[t] = tall ? __builtin_amdgcn_mfma_f64_16x16x4f64(y, e, d[t], 0, 0, 0) : __builtin_amdgcn_mfma_f64_16x16x4f64(e, y, d[t], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int s = 0; s < K; ++s) {
        const double y = (double)x[s];
#pragma unroll
        for (int t = 0; t < MT; ++t)
          d[t] = tall ? __builtin_amdgcn_mfma_f64_16x16x4f64(y, qf[t][s], d[t], 0, 0, 0)
                      : __builtin_amdgcn_mfma_f64_16x16x4f64(qf[t][s], y, d[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int idx;
          if (!place(c, t, r, idx)) continue;
          const float v = (float)d[t][r];
          const float p = fmaf(nlr, (v * sc) * rm + wd * w[t][r], w[t][r]);
          thin_put(x0, idx, v);
          if (!last_run) continue;
          if (store == 0) thin_put(pb, idx, p);
          else store_stored(a.param, q.elem_off + idx, store, p);
        }
      if (c + kStep < n1) {
#pragma unroll
        for (int s = 0; s < K; ++s) x[s] = nx[s];
      }
    }
  }
  if (q.slabs > 1) {   // the last block of the matrix to get here leaves the counters as it found them
    __syncthreads();
    if (threadIdx.x == 0 &&
        __hip_atomic_fetch_add(sync + q.sync + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == q.slabs - 1) {
      __hip_atomic_store(sync + q.sync, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(sync + q.sync + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

}  // namespace pylo
