// Newton-Schulz, normaliser and update of small matrices (a smaller dim m of 33 to 128, and thinner ones lifted to their launch;
// k_ns_thin.h has the others) in one launch: a block (or a few) per matrix.
//
// The tiled products (k_ns_hf.h) are one launch per product for all matrices of a plan: sixteen dependent launches of
// 128 x 128 tiles with whole 128-row operands in memory.  A matrix whose smaller dim m is at most 128 pads that to several
// times its work and leaves most CUs idle, and what bounds its chain is launches, not products.  Here one block takes a
// matrix from the raw step to the parameter: norm, five iterations, RMS and update, its m x m matrices in LDS and
// registers throughout.
//
// Arithmetic is that of the tiled kernels: every operand is two fp16 planes of its entries times a power of two from
// ns_plane_exps, three v_mfma_f32_32x32x16_f16 per fp32 product, fp32 accumulation; iterations in pairs that share
// one Gram product and one update (T = A B', A' = B' T, B'' = p(A'), Q = B'' B', X'' = Q X).
//
// Layout.  MT = m rounded up to 32 over 32 (2 or 4); MT / RT x MT waves, each owning the 32 x 32 tiles (tr0 + i, tc), i <
// RT, of every m x m matrix and the tiles (tr0 + i, tc + MT j), j < J, of a chunk of NB = 32 MT J columns of X (m x n, n
// the longer dim, whatever way the tensor stores it), all as fp32 accumulators: register r of a lane is row 8 (r / 4) + 4 (lane / 32)
// + r % 4, its column is lane % 32.  Planes in LDS, the reduction index contiguous, rows padded by 16 bytes so that
// sixteen rows read 16 bytes each from sixteen different bank groups:
//   buffer 1   an m x m matrix          buffer 0   an m x m matrix, or a chunk of X as [m][n] (Gram) or [n][m] (update)
// A lane's four consecutive rows are one 8-byte store where the row index is the contiguous one: an m x m matrix is
// written as its transpose that way (they are symmetric, and products of them read rows of both operands).
//
// A matrix of more than one chunk keeps X in memory, in the raw step's place (a chunk belongs to one thread block and
// every element to one thread), and a long one is cut into slabs, a block each: the blocks of a matrix meet five times
// (norm, three Gram products, RMS), leaving their partial sums in the workspace and adding all of them in slab order.
// Blocks wait for blocks of their own matrix only.  The wait ends: a block draws its place in the item table when it
// starts, so that of all matrices with a block running at most one still has blocks to start -- as many as wait in
// it, at most 32 or 8 by class of the 512 or 256 that the chip holds (kSlabsMax), so that the launches that four
// hardware queues can run at once never fill it with them; all others have their blocks running, end, and make room.  After
// kSpinLimit polls a block gives up and leaves NaN in its part of the parameter.
// Measured: the kernel is a chain on one CU -- on 128 x 784 (seven blocks, 92 us) five products of an m x m pair phase
// take 13.7 us of which the matrix instructions are 1.3 us each, a meeting with its partial sums 8.5 us, a Gram or
// update product 3 us.  Whole ELO-CELO2 steps with it and with the tiled products alone: classifiers 784 -> 128 -> 128 -> 10
// 148 / 181 us, 784 -> 64 (x 4) -> 10 103 / 178, transformers of width 96 and 128 with twelve layers and two 4000 x width
// embeddings 267 / 272 and 302 / 301 us.
#pragma once

#include "k_ns_hf.h"

namespace pylo {

struct NsSmall {
  int tensor;
  int m, n, tall;        // tall: the tensor holds X^T (n rows of m)
  int slabs, chunks;     // blocks of the matrix; chunks per block
  long long elem_off;    // elements from the tensor's first
  long long part;        // floats into the partial-sum workspace: 2 x slabs x (32 MT)^2, slabs > 1 only
  int sums, sync;        // its 2 x slabs doubles and two counters (zero between calls)
  int fold;              // k_ns_thin: 2^fold columns side by side
};
struct NsSmallItem { int mat, slab; };

// scales of the planes and what turns accumulators into values (reciprocals of the operands' scales), per product
struct NsSmallStep {
  float x_s, a_s, b_s, t_s, q_s;
  float gram, poly, prod_t, prod_a, prod_q, upd_b, upd_q;
  float c0, c1, c2, eps;
  int n_chains, n_pairs; // chains of iterations; the first n_pairs take two each
};

template <int MT, int RT, int J>
struct SmDims {
  static constexpr int MP = 32 * MT, NB = 32 * MT * J, kWav = MT / RT * MT, kThr = 64 * kWav;
  static constexpr int PM = MP * 2 + 16, PN = NB * 2 + 16;                 // bytes of a plane's row
  static constexpr int kMM = 2 * MP * PM, kXs = 2 * MP * PN, kXl = 2 * NB * PM;
  static constexpr int kBuf0 = kMM > kXs ? (kMM > kXl ? kMM : kXl) : (kXs > kXl ? kXs : kXl);
  static constexpr int kLds = kBuf0 + kMM;
};

// Where lane's rows 32 tr + 8 g + 4 (lane / 32) .. + 3 of column `col` sit: `idx` the first one's element, `st` the
// distance to the next.
struct SmPlace { long long idx; int st; };
__device__ __forceinline__ SmPlace sm_place(const NsSmall& q, int row, int col) {
  return q.tall ? SmPlace{(long long)col * q.m + row, 1} : SmPlace{(long long)row * q.n + col, q.n};
}

// Everything a wave holds of a chunk: tiles (tr0 + i, tc + MT j).
template <int RT, int J>
struct SmX { v16f t[RT][J]; };

// The wave's tiles of the chunk that starts at column n0, from the tensor or whatever lies like it.  `ng[i]`: how many
// of the four groups of eight rows of row tile i hold rows of the matrix (the same for all lanes).  Every load is
// issued before any is waited for: nothing here depends on another.
template <int MT, int RT, int J>
__device__ __forceinline__ void sm_load(const NsSmall& q, const float* base, bool vec, int n0, int tr0, int tc,
                                        const int (&ng)[RT], SmX<RT, J>& x) {
  const int lo = threadIdx.x & 31, kg = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int col = n0 + 32 * (tc + MT * j) + lo;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int row = 32 * (tr0 + i) + 8 * g + 4 * kg;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (g < ng[i] && col < q.n && row < q.m) {
          const SmPlace p = sm_place(q, row, col);
          if (vec) {
            load_vec<4>(base + p.idx, v);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (row + r < q.m) v[r] = *(const gfloat*)(base + p.idx + (long long)r * p.st);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) x.t[i][j][4 * g + r] = v[r];
      }
    }
}

template <int MT, int RT, int J>
__device__ __forceinline__ void sm_store(const NsSmall& q, float* base, bool vec, int n0, int tr0, int tc,
                                         const int (&ng)[RT], const SmX<RT, J>& x) {
  const int lo = threadIdx.x & 31, kg = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int col = n0 + 32 * (tc + MT * j) + lo;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int row = 32 * (tr0 + i) + 8 * g + 4 * kg;
        if (g < ng[i] && col < q.n && row < q.m) {
          const SmPlace p = sm_place(q, row, col);
          const float v[4] = {x.t[i][j][4 * g], x.t[i][j][4 * g + 1], x.t[i][j][4 * g + 2], x.t[i][j][4 * g + 3]};
          if (vec) {
            store_vec<4>(base + p.idx, v);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (row + r < q.m) *(gfloat*)(base + p.idx + (long long)r * p.st) = v[r];
          }
        }
      }
    }
}

// acc[i] += (32 rows of P1 at a + i ra) (32 rows of P2 at b)^T over `ks` reduction steps of 16; `pl1`, `pl2`: distance of
// the planes
template <int RT>
__device__ __forceinline__ void sm_product(const PYLO_LDS char* a, int ra, int pl1, const PYLO_LDS char* b, int pl2, int ks,
                                           v16f (&acc)[RT]) {
  // the next step's fragments are read while the matrix instructions of this one run
  f16x8 fa[2][RT][2], fb[2][2];
  auto fetch = [&](int u, int k) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      fb[u][p] = __builtin_bit_cast(f16x8, *(const luint4*)(b + p * pl2 + 32 * k));
#pragma unroll
      for (int i = 0; i < RT; ++i) fa[u][i][p] = __builtin_bit_cast(f16x8, *(const luint4*)(a + i * ra + p * pl1 + 32 * k));
    }
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      constexpr int pa[3] = {1, 0, 0}, pb[3] = {0, 1, 0};
#pragma unroll
      for (int i = 0; i < RT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[u][i][pa[t]], fb[u][pb[t]], acc[i], 0, 0, 0);
    }
  };
  fetch(0, 0);
  int k = 0;
  for (; k + 2 <= ks; k += 2) {
    fetch(1, k + 1);
    multiply(0);
    fetch(0, k + 2 < ks ? k + 2 : k);
    multiply(1);
  }
  if (k < ks) multiply(0);
}

// A tile into planes whose contiguous index is the tile's row: element (row, col) at [col][row].  Groups of rows from
// `ng` on are zero and only the first `nz` are read as reduction steps.
__device__ __forceinline__ void sm_put_t(PYLO_LDS char* buf, int pitch, int plane, int row0, int col0, int ng, int nz,
                                         const v16f& v, float s) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef PYLO_LDS u32x2 lu2;
  const int lo = threadIdx.x & 31, kg = (threadIdx.x >> 5) & 1;
  PYLO_LDS char* p = buf + (col0 + lo) * pitch + (row0 + 4 * kg) * 2;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (g >= nz) break;
    u32x2 h = {0u, 0u}, l = {0u, 0u};
    if (g < ng) {
      unsigned h0, l0, h1, l1;
      hf_split2(v[4 * g] * s, v[4 * g + 1] * s, h0, l0);
      hf_split2(v[4 * g + 2] * s, v[4 * g + 3] * s, h1, l1);
      h = u32x2{h0, h1};
      l = u32x2{l0, l1};
    }
    *(lu2*)(p + 16 * g) = h;
    *(lu2*)(p + plane + 16 * g) = l;
  }
}
// ... and whose contiguous index is its column: element (row, col) at [row][col].  Rows from 8 `ng` on are left as they
// are: they only reach rows and columns of the product that nobody uses.
__device__ __forceinline__ void sm_put_n(PYLO_LDS char* buf, int pitch, int plane, int row0, int col0, int ng, const v16f& v,
                                         float s) {
  typedef PYLO_LDS hbits lhb;
  const int lo = threadIdx.x & 31, kg = (threadIdx.x >> 5) & 1;
  PYLO_LDS char* p = buf + (row0 + 4 * kg) * pitch + (col0 + lo) * 2;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (g >= ng) break;
#pragma unroll
    for (int r = 0; r < 4; r += 2) {
      unsigned h, l;
      hf_split2(v[4 * g + r] * s, v[4 * g + r + 1] * s, h, l);
      PYLO_LDS char* o = p + (8 * g + r) * pitch;
      *(lhb*)o = (hbits)h;
      *(lhb*)(o + plane) = (hbits)l;
      *(lhb*)(o + pitch) = (hbits)(h >> 16);
      *(lhb*)(o + pitch + plane) = (hbits)(l >> 16);
    }
  }
}

// The blocks of a matrix meet.  What they hand each other goes through agent-scope atomics on both sides (pylo_common.h):
// a fence would write back and invalidate the XCD's whole L2, which hundreds of blocks meeting five times each made the
// cost of everything else the launch reads.
__device__ __forceinline__ bool sm_meet(int* counter, int target, int* lds_flag) {
  __syncthreads();   // every exchange of this block has returned its old value
  if (threadIdx.x == 0) {
    __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int ok = coh_load(counter) >= target;
    for (int spin = 0; !ok && spin < kSpinLimit; ++spin) {
      __builtin_amdgcn_s_sleep(4);
      ok = coh_load(counter) >= target;
    }
    *lds_flag = ok;
  }
  __syncthreads();
  return *lds_flag != 0;
}
// The partial sums themselves are four floats an access: buffer accesses with the agent scope's cache bit (sc1, what an
// agent-scope atomic load or store carries), waited for before the block counts itself in.
constexpr int kSmAgent = 16;
typedef __amdgpu_buffer_rsrc_t SmBuf;
__device__ __forceinline__ SmBuf sm_buffer(float* p, int bytes) { return __builtin_amdgcn_make_buffer_rsrc(p, 0, bytes, 0x00020000); }
__device__ __forceinline__ void sm_leave(SmBuf b, int off, v4f v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), b, off, 0, kSmAgent);
}
__device__ __forceinline__ v4f sm_fetch(SmBuf b, int off) {
  return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, kSmAgent));
}

template <int RT>
struct SmM { v16f t[RT]; };   // a wave's tiles (tr0 + i, tc) of an m x m matrix

template <int MT, int RT, int J>
__global__ __launch_bounds__(64 * (MT / RT) * MT) void k_ns_small(
    const NsSmall* __restrict__ mats, const NsSmallItem* __restrict__ items, const TDesc* __restrict__ descs,
    const PyloTensorArgs* __restrict__ dyn, float* __restrict__ part, double* __restrict__ sums, int* __restrict__ sync,
    NsSmallStep st, int orth_call, int* __restrict__ tickets) {
  using D = SmDims<MT, RT, J>;
  extern __shared__ __attribute__((aligned(16))) char lds_[];
  PYLO_LDS char* buf0 = (PYLO_LDS char*)lds_;
  PYLO_LDS char* buf1 = buf0 + D::kBuf0;
  __shared__ double red[D::kWav];
  __shared__ int s_flag;
  int item = (int)blockIdx.x;
  if (tickets != nullptr) {
    if (threadIdx.x == 0) s_flag = __hip_atomic_fetch_add(tickets, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    item = __builtin_amdgcn_readfirstlane(s_flag);
    // the last block to draw leaves the counter at zero for the next launch
    if (item == (int)gridDim.x - 1 && threadIdx.x == 0)
      __hip_atomic_store(tickets, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const NsSmallItem it = items[item];
  const NsSmall q = mats[it.mat];
  const PyloTensorArgs a = dyn[q.tensor];
  if (a.grad == nullptr) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tr0 = wave / MT * RT, tc = wave % MT, lo = lane & 31, kg = lane >> 5;
  float* const base = a.step_out + q.elem_off;
  const bool vec = q.tall && (q.m & 3) == 0 && (reinterpret_cast<uintptr_t>(base) & 15) == 0;
  const int n0 = it.slab * q.chunks * D::NB;
  const int ks = (q.m + 15) >> 4;            // reduction steps over m
  int ng[RT], nz[RT];                        // groups of rows of the wave's tiles: with rows of the matrix; read by a reduction over m
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    ng[i] = min(max((q.m - 32 * (tr0 + i) + 7) >> 3, 0), 4);
    nz[i] = min(max(2 * ks - 4 * (tr0 + i), 0), 4);
  }
  const int n_ch = min(q.chunks, (q.n - n0 + D::NB - 1) / D::NB);
  const bool resident = q.chunks == 1;
  int meets = 0;
  bool good = true;
  // sum over the matrix of the block's sums `s` (per lane), the same for every block
  auto total = [&](double s) {
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < D::kWav; ++w) t += red[w];
    __syncthreads();
    if (q.slabs > 1) {
      double* o = sums + q.sums + (meets & 1) * q.slabs;
      if (threadIdx.x == 0) coh_store_wait(o + it.slab, t);
      ++meets;
      if (good) good = sm_meet(sync + q.sync, meets * q.slabs, &s_flag);
      t = wave_sum(lane < q.slabs ? coh_load(o + lane) : 0.0);   // at most 32 slabs; the same tree in every wave of every block
    }
    return t;
  };
  // the chunks of the block one after another, the next one's loads in flight; a single one stays in registers
  SmX<RT, J> x;
  auto each_chunk = [&](bool loaded, auto body) {
    if (!loaded) sm_load<MT, RT, J>(q, base, vec, n0, tr0, tc, ng, x);
    for (int c = 0; c < n_ch; ++c) {
      SmX<RT, J> nx;
      if (c + 1 < n_ch) sm_load<MT, RT, J>(q, base, vec, n0 + (c + 1) * D::NB, tr0, tc, ng, nx);
      body(c);
      if (c + 1 < n_ch) x = nx;
    }
  };
  // sums of squares: a lane's 32 values of a chunk in fp32, chunks, lanes and waves in fp64 (as k_celo2_sumsq, whose lanes
  // have 32 values too)
  static_assert(16 * RT * J == 32, "values of a lane and chunk");
  double sq = 0.0;
  auto square = [&]() {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) s = fmaf(x.t[i][j][r], x.t[i][j][r], s);
    sq += (double)s;
  };
  each_chunk(false, [&](int) { square(); });
  if (orth_call && (a.flags & kArgOrthogonalize)) {
    // X0 = raw / (||raw|| + eps): the factor rides on the planes' scale while X comes from memory
    float xs = 1.0f / ((float)sqrt(total(sq)) + st.eps);
    if (resident) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) x.t[i][j][r] *= xs;
      xs = 1.0f;
    }
    // a lane's 16 bytes of an operand row: row 32 t + lo, half kg of every step
    const int om = lo * D::PM + 16 * kg, on = lo * D::PN + 16 * kg;
    constexpr int kPlM = D::MP * D::PM, kPlN = D::MP * D::PN, kPlL = D::NB * D::PM;
    for (int ch = 0; ch < st.n_chains; ++ch) {
      const bool last = ch == st.n_chains - 1;
      const float sx = xs * st.x_s;
      SmM<RT> A;
      auto clear = [&](SmM<RT>& m) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) m.t[i][r] = 0.0f;
      };
      // A = X X^T
      clear(A);
      each_chunk(resident, [&](int) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < J; ++j)
            sm_put_n(buf0, D::PN, kPlN, 32 * (tr0 + i), 32 * (tc + MT * j), ng[i], x.t[i][j], sx);
        __syncthreads();
        sm_product<RT>(buf0 + 32 * tr0 * D::PN + on, 32 * D::PN, kPlN, buf0 + 32 * tc * D::PN + on, kPlN, D::NB / 16, A.t);
        __syncthreads();
      });
      // (rows and columns past m: zero, whatever the planes held there)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          A.t[i][r] = 32 * (tr0 + i) + 8 * (r >> 2) + 4 * kg + (r & 3) < q.m && 32 * tc + lo < q.m ? A.t[i][r] * st.gram : 0.0f;
      if (q.slabs > 1) {
        // [slab][tile][r / 4][thread][r % 4]: 16 bytes a thread, consecutive threads adjacent
        constexpr int kMM2 = D::MP * D::MP * 4;   // bytes
        const SmBuf pbuf = sm_buffer(part + q.part, 2 * q.slabs * kMM2);
        const int o = (meets & 1) * q.slabs * kMM2 + threadIdx.x * 16;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            if (g < ng[i])
              sm_leave(pbuf, o + it.slab * kMM2 + (i * 4 + g) * D::kThr * 16,
                       v4f{A.t[i][4 * g], A.t[i][4 * g + 1], A.t[i][4 * g + 2], A.t[i][4 * g + 3]});
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // they have been performed
        ++meets;
        if (good) good = sm_meet(sync + q.sync, meets * q.slabs, &s_flag);
        clear(A);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            if (g >= ng[i]) continue;
            constexpr int kAhead = RT == 2 ? 8 : 16;   // slabs whose values are asked for together
            for (int b0 = 0; b0 < q.slabs; b0 += kAhead) {
              v4f v[kAhead];
#pragma unroll
              for (int u = 0; u < kAhead; ++u)
                v[u] = b0 + u < q.slabs ? sm_fetch(pbuf, o + (b0 + u) * kMM2 + (i * 4 + g) * D::kThr * 16)
                                        : v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
              for (int u = 0; u < kAhead; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) A.t[i][4 * g + r] += v[u][r];
            }
          }
      }
      // the product of two m x m matrices in LDS, this wave's tiles of it
      auto mm = [&](const PYLO_LDS char* p1, const PYLO_LDS char* p2, float inv) {
        SmM<RT> d;
        clear(d);
        sm_product<RT>(p1 + 32 * tr0 * D::PM + om, 32 * D::PM, kPlM, p2 + 32 * tc * D::PM + om, kPlM, ks, d.t);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) d.t[i][r] *= inv;
        return d;
      };
      auto put = [&](PYLO_LDS char* b, const SmM<RT>& v, float s) {
#pragma unroll
        for (int i = 0; i < RT; ++i) sm_put_t(b, D::PM, kPlM, 32 * (tr0 + i), 32 * tc, ng[i], nz[i], v.t[i], s);
      };
      auto poly = [&](const PYLO_LDS char* pa) {   // c2 A A + c1 A + c0 I; rows and columns past m stay zero
        SmM<RT> d = mm(pa, pa, st.poly);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = 32 * (tr0 + i) + 8 * (r >> 2) + 4 * kg + (r & 3), col = 32 * tc + lo;
            d.t[i][r] = st.c2 * d.t[i][r] + st.c1 * A.t[i][r] + (row == col && row < q.m ? st.c0 : 0.0f);
          }
        return d;
      };
      put(buf0, A, st.a_s);
      __syncthreads();
      put(buf1, poly(buf0), st.b_s);                     // B'
      __syncthreads();
      const bool pair = ch < st.n_pairs;
      if (pair) {
        const SmM<RT> T = mm(buf0, buf1, st.prod_t);     // T = A B'
        __syncthreads();
        put(buf0, T, st.t_s);
        __syncthreads();
        A = mm(buf1, buf0, st.prod_a);                   // A' = B' T
        __syncthreads();
        put(buf0, A, st.a_s);
        __syncthreads();
        const SmM<RT> B2 = poly(buf0);                   // B'' = p(A')
        __syncthreads();
        put(buf0, B2, st.b_s);
        __syncthreads();
        const SmM<RT> Q = mm(buf0, buf1, st.prod_q);     // Q = B'' B'
        __syncthreads();
        put(buf1, Q, st.q_s);
      }
      // X <- Q X
      const float inv = pair ? st.upd_q : st.upd_b;
      if (last) sq = 0.0;
      each_chunk(resident, [&](int c) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < J; ++j)
            sm_put_t(buf0, D::PM, kPlL, 32 * (tr0 + i), 32 * (tc + MT * j), ng[i], nz[i], x.t[i][j], sx);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; ++j) {
          SmM<RT> d;
          clear(d);
          sm_product<RT>(buf1 + 32 * tr0 * D::PM + om, 32 * D::PM, kPlM, buf0 + 32 * (tc + MT * j) * D::PM + om, kPlL, ks, d.t);
#pragma unroll
          for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) x.t[i][j][r] = d.t[i][r] * inv;
        }
        if (last) square();
        if (!resident || last) sm_store<MT, RT, J>(q, base, vec, n0 + c * D::NB, tr0, tc, ng, x);
        __syncthreads();
      });
      xs = 1.0f;
    }
  }
  // step = X * rsqrt(1e-9 + mean X^2) * rmsmult; p <- p - lr (step + wd p)
  const float rm = a.step_mult, wd = a.weight_decay, nlr = -a.lr;
  const int store = descs[q.tensor].store;
  float* const pb = a.param + q.elem_off;
  const bool pvec = vec && (reinterpret_cast<uintptr_t>(pb) & 15) == 0;
  SmX<RT, J> p;   // the parameter's first chunk is asked for before the blocks meet
  if (store == 0) sm_load<MT, RT, J>(q, pb, pvec, n0, tr0, tc, ng, p);
  const double ss = total(sq);
  const float sc = good ? rsq(1e-9f + (float)(ss / ((double)q.m * (double)q.n))) : __builtin_nanf("");
  each_chunk(resident, [&](int c) {
    if (store == 0) {
      if (c > 0) sm_load<MT, RT, J>(q, pb, pvec, n0 + c * D::NB, tr0, tc, ng, p);
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            p.t[i][j][r] = fmaf(nlr, (x.t[i][j][r] * sc) * rm + wd * p.t[i][j][r], p.t[i][j][r]);
      sm_store<MT, RT, J>(q, pb, pvec, n0 + c * D::NB, tr0, tc, ng, p);
    } else {
      // the parameter in its storage type: widened, updated in fp32, rounded to nearest-even
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int col = n0 + c * D::NB + 32 * (tc + MT * j) + lo;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = 32 * (tr0 + i) + 8 * (r >> 2) + 4 * kg + (r & 3);
            if (col >= q.n || row >= q.m) continue;
            const long long e = q.elem_off + sm_place(q, row, col).idx;
            const float w = load_stored(a.param, e, store);
            store_stored(a.param, e, store, fmaf(nlr, (x.t[i][j][r] * sc) * rm + wd * w, w));
          }
        }
    }
  });
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
