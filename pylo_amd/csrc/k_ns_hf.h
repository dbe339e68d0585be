// Newton-Schulz products at fp32 accuracy on the fp16 matrix pipe.
//
// An fp32 number times a power of two is, to 2^-22 of its size, the sum of two fp16 numbers: x s = h + l with
// h = fp16(x s), l = fp16(x s - h) (11 + 11 significand bits), as long as h does not overflow (|x s| < 65 504) and l
// does not fall off the format's lower end (fp16 keeps subnormals down to 2^-24 and the matrix instructions take
// them as they are: l is exact to 2^-25 absolutely, i.e. entries below 1/8 lose relative, not absolute, accuracy).
// A product of two such numbers is four fp16 products; the smallest (l l, 2^-22 |x y|) is dropped with the
// remainders.  The other three are exact in fp32 and are accumulated in fp32 by v_mfma_f32_32x32x16_f16, which does
// sixteen times the multiply-adds of v_mfma_f32_32x32x2_f32 per instruction slot: three of them replace eight fp32
// instructions' worth of work.  An operand carries 23 significant bits where fp32 has 24: a product of the iteration
// is off by about 6e-8 of its entries' RMS, a quarter of what the fp32 accumulation of a reduction over 256 .. 4096
// terms adds anyway (a plain fp32 GEMM: 2.5e-7), but each entry of the result carries 1 .. 3e-7 of its own size where
// an fp32 product carries 6e-8.  With the reference's coefficients, which multiply rounding by up to 3.44 an
// iteration, the result is as far from the fp64 formula as the fp32 torch products are (0.4 .. 0.9 times, tests); with
// polynomials that do not amplify (1.5 x - 0.5 x^3, 2 x - x^3) it is 3 .. 12 times further, 1e-5 of its RMS at most.
// The scales: no entry of a matrix exceeds its largest singular value, and the singular values of everything the
// iteration forms follow from the coefficients alone once X0 has unit Frobenius norm (the host walks a grid of
// starting values through sigma -> sigma p(sigma^2), ns_plane_exps): X and A = X X^T stay below 1.5, B' = p(A)
// below c0, products of k such B' below c0^k.  Every kind of matrix gets the power of two that puts its bound at
// 12 000 .. 24 000; a product's accumulators are scaled back by the reciprocal of its operands' scales (exact) and
// what it writes is scaled by its own.  A value outside its bound -- there should be none -- is not clamped: it
// becomes an infinity and then a NaN, which stays visible.
//
// Operands therefore live as *planes*: two fp16 matrices (h, l) with the reduction index contiguous,
// written by the kernel that produces the matrix (never converted inside a product's main loop).
// With X of m x n or n x m (m the smaller dim), Xs = X as [m][n] and Xl = X as [n][m]:
//     A   = Xs Xs^T                      (reduction over n; symmetric, tiles on and above the diagonal)
//     B'  = c2 A A + c1 A + c0 I         (reduction over m; symmetric)
//     Xl' = Xl B'                        (reduction over m), written as planes of Xl' and of Xs' = Xl'^T,
//                                         or as fp32 in the tensor's own layout after the last iteration
// for wide and tall matrices alike (B' is symmetric, so (B' X)^T = X^T B').
//
// Two iterations can share the two products over the long dim.  Every B'_t is a polynomial in A_t, so it
// commutes with A_t and is symmetric, and A_{t+1} = X_{t+1} X_{t+1}^T = B'_t A_t B'_t needs no X:
//     A_t (Gram), B'_t = p(A_t) (Poly), T = A_t B'_t (Prod), A_{t+1} = B'_t T (ProdA), B'_{t+1} = p(A_{t+1}) (Poly),
//     Q = B'_{t+1} B'_t (Prod), X_{t+2} = Q X_t (Update)
// i.e. four products of m^3 / 2 multiply-adds in place of one Gram product (m^2 n / 2) and one update (m^2 n).
// What it costs in accuracy is bounded whatever the spectrum of X: A_t as computed is off by eps ||A_t|| in
// absolute terms, which A_{t+1} = B'_t A_t B'_t inherits relative to its small eigenvalues -- they grow by
// p(0)^2 = c0^2 in the step, so the error of p(A_{t+1}) in those directions is c1 c0^2 eps sigma_max^2, about
// 12 times that of p of a freshly formed Gram matrix and about 1e-6 of B' itself; a second chained step
// multiplies it by c0^2 again, which is why pairs are the default and the next pair starts from a Gram product
// of the X it was handed.  The host enqueues chains of any length L (one Gram product, 4 L - 3 products of
// m x m matrices rotating through four plane buffers, one update): PYLO_MI355_NS_CHAINS="3,2" in the environment
// trades accuracy for time (up to 1e-4 of the result's RMS on a dominant direction over a flat rest, where pairs
// are at 1.3e-5), PYLO_MI355_NS_PAIRS=0 keeps one Gram product and one update per iteration.
//
// Tile job: 128 x 128 (Gram, Poly, narrow updates) or 128 x 256 outputs (updates with m > 128) by 256 threads =
// 2 x 2 waves of 64 x 64 / 64 x 128 = 2 x 2 / 2 x 4 accumulators of 32 x 32; 16 reduction steps per stage,
// double buffered in LDS (32 / 48 KB), staged from global memory straight into LDS (global_load_lds_dwordx4: no
// staging registers, no LDS store instructions), one 16-byte read per lane, plane and 32-row block per stage.  A launch with
// less than a tile of 128 x 128 a CU takes 64 x 64 (a 32 x 32 a wave) and 64 steps a stage: such a job is a chain of loads
// that waits for memory once a stage, and four times as many blocks wait together.
// The planes are allocated with their rows rounded up to whole tiles and the padding holds zeros, so the main
// loop has no bounds checks; any two dims are taken (the raw step is read and the result written per element
// where the tensor's rows are not 16-byte aligned).
#pragma once

#include <type_traits>

#include "k_ns.h"

namespace pylo {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short hbits;   // one number of a plane in memory (an fp16)
constexpr int kNsPl = 2;                      // planes per matrix
constexpr int kNsRowB = 32 * kNsPl;           // bytes of one row in a block of 16 reduction steps
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4 luint4;

constexpr int kHfBK = 16;                     // reduction steps per stage
// LDS of a tile job with 64 WI rows and 64 WN columns: two stages of (64 WI + 64 WN) rows x 2 planes x 32 KS bytes
constexpr int hf_gemm_lds(int wi, int wn, int ks) { return 2 * ks * (64 * wi + 64 * wn) * kNsRowB; }

// Planes of one matrix with `rows` rows (a multiple of the tiles' rows; rows past the matrix hold zeros) and a (padded)
// reduction length: blocks of 16 reduction steps x 16 rows, [k / 16][row / 16], of 1 KB each, inside a block [half: k / 8 % 2]
// [plane][row % 16][k % 8].  The rows x 2 planes x 16 steps a tile job stages at a time are consecutive memory, a block is
// what one wave-wide 16-byte load or store moves in lane order, and in LDS, where a stage lies as in memory, sixteen lanes
// read the same piece of sixteen rows from 256 consecutive bytes.
struct HfPlanes {
  const hbits* base;
  int rows;
};
constexpr int kNsBlock = 16 * 16 * kNsPl;   // numbers of a block

// the block with row and reduction step (row, k), elements from the planes' first
__device__ __forceinline__ size_t hf_block(int rows, int row, int k) {
  return (size_t)(k >> 4) * rows * (16 * kNsPl) + (size_t)(row >> 4) * kNsBlock;
}

struct NsHfMat {
  int tensor;
  int R, C, m, n, tall;      // X is R x C row-major; m = min, n = max; tall: R > C
  int pad_m, pad_n;          // m and n rounded up to the 16 reduction steps of a stage (the padding holds zeros)
  int rows_m, rows_n;        // rows allocated for the planes whose rows are the m / n index (whole tiles)
  int n_slabs;
  long long off_xs;          // elements (hbits) into the plane workspace: planes of Xs (m rows, reduction n)
  long long off_xl[2];       // planes of Xl (n rows, reduction m), two buffers (a product reads one and writes the other)
  long long off_p, p_stride; // planes of the m x m matrices (m rows, reduction m): buffer b at off_p + b p_stride
  long long off_a, a_floats; // floats into the fp32 workspace: A (hf_a32); its size, and a partial matrix's
  long long off_part;        // floats: partial matrices of a split Gram product
  long long elem_off;        // elements from the tensor's raw step to this matrix (a slice of a tensor with more dims)
  int fpart0, n_fpart;       // its partial sums of squares of A (k_ns_hf_chain_sumsq): first, count
};

// the m x m plane buffers, and the two products on planes in and planes out (k_ns_hf_gemm's OP, after
// kNsGram / kNsPoly / kNsUpdate)
enum : int { kNsBufA = 0, kNsBufB = 1, kNsBufT = 2, kNsBufC = 3, kNsBufs = 4 };
enum : int { kNsProd = 3, kNsProdA = 4 };
// operand and result buffers of an m x m product (the update's B' is s1); what turns the accumulators into the
// product's values (the reciprocal of the operands' plane scales) and the scale of the planes written
struct NsBufs { int s1, s2, d; float acc_scale, out_scale; };

// The fp32 copy of a symmetric m x m matrix (and of the partial matrices that add up to it): the 128 x 128 tiles on and
// above the diagonal, row by row, each as the accumulators of the job that computes it, [wave][hi][hj][r / 4][lane][r % 4]
// -- the job that reads it again (Poly) is the same tile's, so both move 16 bytes a lane in lane order.
__host__ __device__ __forceinline__ int hf_tiles_upper(int m) {
  const int nt = (m + kNsTile - 1) / kNsTile;
  return nt * (nt + 1) / 2;
}
__device__ __forceinline__ int hf_tile_index(int m, int tm, int tn) {
  const int nt = (m + kNsTile - 1) / kNsTile;
  return tm * nt - tm * (tm - 1) / 2 + tn - tm;
}
constexpr int kNsTileFloats = kNsTile * kNsTile;
// floats from A's first to the lane's registers 4 q .. 4 q + 3 of sub-tile (hi, hj)
__device__ __forceinline__ size_t hf_a32(int tile, int wave, int hi, int hj, int q, int lane) {
  return ((((size_t)tile * 4 + wave) * 4 + hi * 2 + hj) * 4 + q) * 256 + lane * 4;
}

// Two values (times their plane scale already) as two dwords, one of each plane: x = h + l + what is left below 2^-22 |x|.
// No clamp: a matrix within the bounds the scales were chosen for stays below 24 000, and what is not -- a raw step with an
// infinity or a NaN, whose norm is neither -- has to stay visible.
__device__ __forceinline__ void hf_split2(float a, float b, unsigned& h, unsigned& l) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const h2 hh = __builtin_convertvector(f2{a, b}, h2);
  const h2 ll = __builtin_convertvector(f2{a - (float)hh[0], b - (float)hh[1]}, h2);
  h = __builtin_bit_cast(unsigned, hh);
  l = __builtin_bit_cast(unsigned, ll);
}

#define PYLO_LDS __attribute__((address_space(3)))
#define PYLO_GLB __attribute__((address_space(1)))

// A stage of ROWS rows of one operand from memory into LDS, as it lies there: one wave-wide load a block (the hardware
// puts lane l's 16 bytes at the instruction's LDS base + 16 l), blocks dealt to the waves in turn.  `g`: the stage's first
// byte plus 16 lane.  (NW: waves of the block)
template <int ROWS, int NW = 4>
__device__ __forceinline__ void hf_stage_issue(const char* g, PYLO_LDS char* lds, int wave) {
#pragma unroll
  for (int j = 0; j < ROWS * kNsRowB / (1024 * NW); ++j)
    __builtin_amdgcn_global_load_lds((const PYLO_GLB void*)(g + (j * NW + wave) * 1024), (PYLO_LDS void*)(lds + (j * NW + wave) * 1024), 16, 0, 0);
}

// The lane's fragment of row `row0 + lane % 32` (row0 a multiple of 16) in a stage in LDS: byte offset of plane 0, plane 1 is
// 256 bytes further, the row 32 further down 2048.
__device__ __forceinline__ int hf_frag(int row0, int lane) {
  const int lo = lane & 31, kg = lane >> 5;
  return (row0 + (lo & 16)) * kNsRowB + kg * 512 + (lo & 15) * 16;
}

// acc[hi][hj] += (rows i0.. of P1) x (rows j0.. of P2)^T over the reduction range [k0, k1) (multiples of 16);
// 16 NW WI rows of P1, 64 WN rows of P2, KS times 16 reduction steps a stage.  LDS: two stages of (16 NW WI + 64 WN) x 64 KS
// bytes.
// `compute` (the same for all lanes of a wave): false for a wave whose values nobody needs -- it stages and meets the
// barriers, and leaves the matrix pipe to the other waves of its SIMD.
template <int WI, int WN, int KS = 1, int NW = 4>
__device__ __forceinline__ void hf_tile_product(const HfPlanes& P1, int i0, const HfPlanes& P2, int j0, int k0, int k1,
                                                PYLO_LDS char* lds, v16f (&acc)[WI][WN], bool compute = true) {
  constexpr int RA = 16 * NW * WI, RB = 64 * WN, SA = RA * kNsRowB, STEP = SA + RB * kNsRowB, STAGE = KS * STEP;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = (wave >> 1) * 32 * WI, wj = (wave & 1) * 32 * WN;
  const char* ga = (const char*)P1.base + ((size_t)(k0 >> 4) * P1.rows + i0) * kNsRowB + 16 * lane;
  const char* gb = (const char*)P2.base + ((size_t)(k0 >> 4) * P2.rows + j0) * kNsRowB + 16 * lane;
  const size_t sa = (size_t)P1.rows * kNsRowB, sb = (size_t)P2.rows * kNsRowB;
  // a diagonal tile of X X^T or A A: both operands are the same rows, staged once
  const bool same = RA == RB && P1.base == P2.base && i0 == j0;
  auto issue = [&](int k, PYLO_LDS char* to) {   // the stage that starts at k
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (u > 0 && k + u * kHfBK >= k1) break;
      hf_stage_issue<RA, NW>(ga, to + u * STEP, wave);
      if (!same) hf_stage_issue<RB, NW>(gb, to + u * STEP + SA, wave);
      ga += sa;
      gb += sb;
    }
  };
  issue(k0, lds);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  const int oa = hf_frag(wi, lane), ob = (same ? 0 : SA) + hf_frag(wj, lane);
  auto multiply = [&](auto steps, const PYLO_LDS char* from) {
    constexpr int N = steps.value;
    f16x8 a[N][WI][kNsPl], b[N][WN][kNsPl];
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int q = 0; q < kNsPl; ++q) {
#pragma unroll
        for (int i = 0; i < WI; ++i)
          a[u][i][q] = __builtin_bit_cast(f16x8, *(const luint4*)(from + u * STEP + oa + i * 32 * kNsRowB + q * 256));
#pragma unroll
        for (int j = 0; j < WN; ++j)
          b[u][j][q] = __builtin_bit_cast(f16x8, *(const luint4*)(from + u * STEP + ob + j * 32 * kNsRowB + q * 256));
      }
    // smallest terms first: l h, h l, h h
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int term = 0; term < 3; ++term) {
        constexpr int pa[3] = {1, 0, 0}, pb[3] = {0, 1, 0};
#pragma unroll
        for (int hi = 0; hi < WI; ++hi)
#pragma unroll
          for (int hj = 0; hj < WN; ++hj)
            acc[hi][hj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[u][hi][pa[term]], b[u][hj][pb[term]], acc[hi][hj], 0, 0, 0);
      }
  };
  int cur = 0;
  for (int k = k0; k < k1; k += KS * kHfBK) {
    if (k + KS * kHfBK < k1) issue(k + KS * kHfBK, lds + (STAGE - cur));
    if (compute) {
      // (a whole stage's fragments are read before its first product: one wait for LDS, not one a step)
      if (KS == 1 || k + KS * kHfBK <= k1) multiply(std::integral_constant<int, KS>(), lds + cur);
      else
        for (int u = 0; k + u * kHfBK < k1; ++u) multiply(std::integral_constant<int, 1>(), lds + cur + u * STEP);
    }
    // the loads into the other stage have landed (they are counted like any other vector-memory load) and
    // every wave has read this one
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    cur = STAGE - cur;
  }
}

// The same product with the first operand's fragments loaded straight from memory into registers, two steps ahead (a
// lane's fragment of a row is 16 consecutive bytes of the planes): only the second operand goes through LDS, 48 KB
// of LDS traffic a step and block instead of 73.  128 rows of P1 (by 256 threads), 64 WN rows of P2; LDS: two
// stages of 64 WN x 64 bytes.  Benchmark instrumentation only (pylo_mi355_matrix_probe, mode 4): the bare loop is
// 8 - 12 % faster this way on one large operand, the update product inside whole steps 2.5 % slower (with four groups of matrices
// on four streams).
template <int WN>
__device__ __forceinline__ void hf_tile_product_direct(const HfPlanes& P1, int i0, const HfPlanes& P2, int j0, int k0, int k1,
                                                       PYLO_LDS char* lds, v16f (&acc)[2][WN]) {
  constexpr int RB = 64 * WN, STAGE = RB * kNsRowB;
  typedef PYLO_GLB u32x4 gu32x4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = (wave >> 1) * 64, wj = (wave & 1) * 32 * WN;
  const char* ga = (const char*)P1.base + ((size_t)(k0 >> 4) * P1.rows + i0) * kNsRowB + hf_frag(wi, lane);
  const char* gb = (const char*)P2.base + ((size_t)(k0 >> 4) * P2.rows + j0) * kNsRowB + 16 * lane;
  const size_t sa = (size_t)P1.rows * kNsRowB, sb = (size_t)P2.rows * kNsRowB;
  u32x4 an[2][2][kNsPl];   // the fragments of this step and the next (slot = step % 2), refilled for two steps on
  auto fetch_a = [&](auto slot, const char* g) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < kNsPl; ++q) an[slot.value][i][q] = *(const gu32x4*)(g + i * 32 * kNsRowB + q * 256);
  };
  typedef std::integral_constant<int, 0> S0;
  typedef std::integral_constant<int, 1> S1;
  hf_stage_issue<RB>(gb, lds, wave);
  fetch_a(S0(), ga);
  if (k0 + kHfBK < k1) fetch_a(S1(), ga + sa);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  const int ob = hf_frag(wj, lane);
  int cur = 0;
  ga += sa;
  auto step = [&](auto slot, int k) {
    f16x8 a[2][kNsPl], b[WN][kNsPl];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < kNsPl; ++q) a[i][q] = __builtin_bit_cast(f16x8, an[slot.value][i][q]);
    const bool more_b = k + kHfBK < k1, more_a = k + 2 * kHfBK < k1;
    if (more_b) {
      gb += sb;
      hf_stage_issue<RB>(gb, lds + (STAGE - cur), wave);
    }
    if (more_a) {
      ga += sa;
      fetch_a(slot, ga);
    }
#pragma unroll
    for (int q = 0; q < kNsPl; ++q)
#pragma unroll
      for (int j = 0; j < WN; ++j)
        b[j][q] = __builtin_bit_cast(f16x8, *(const luint4*)(lds + cur + ob + j * 32 * kNsRowB + q * 256));
#pragma unroll
    for (int term = 0; term < 3; ++term) {
      constexpr int pa[3] = {1, 0, 0}, pb[3] = {0, 1, 0};
#pragma unroll
      for (int hi = 0; hi < 2; ++hi)
#pragma unroll
        for (int hj = 0; hj < WN; ++hj)
          acc[hi][hj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[hi][pa[term]], b[hj][pb[term]], acc[hi][hj], 0, 0, 0);
    }
    // the second operand's next stage has landed and every wave has read this one; the fragments just asked for
    // (the newest loads: loads complete in order) may still be on their way.  The bare barrier: a __syncthreads()
    // would wait for them too.
    if (more_a) __builtin_amdgcn_s_waitcnt((2 * kNsPl) | (7 << 4));   // vmcnt <= 4, lgkmcnt 0
    else __builtin_amdgcn_s_waitcnt(7 << 4);                            // vmcnt 0, lgkmcnt 0
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    cur = STAGE - cur;
  };
  for (int k = k0; k < k1; k += 2 * kHfBK) {
    step(S0(), k);
    if (k + kHfBK < k1) step(S1(), k + kHfBK);
  }
}

// A wave's 32 HI x 32 WN values (accumulator layout) times `scale` into planes, in one or both orientations, every value
// split once.  Rows and columns past the matrix hold zeros (hf_mask_edge).
//   D   planes whose reduction index is the values' column: through the wave's own LDS patch, [column][16 rows] a plane,
//       sixteen rows at a time, read back transposed (ds_read_b64_tr_b16: of the 4 columns x 16 rows that sixteen lanes
//       address, lane i gets row i's four columns)
//   D4  (when not null) planes whose reduction index is the row: straight from the registers
// A lane's two quads of sixteen rows (8 g + 4 (lane / 32) ..) become eight consecutive ones by one swap between the
// halves of the wave: 16 bytes of a plane, LDS takes them as they are, and one more swap between neighbouring sixteens of
// lanes puts the pieces of sixteen columns into the order of a block: every store is 1 KB in lane order.  Before, the mirrored
// planes went out 8 bytes a lane, 64 apart, and the others 2 bytes a value into the patch.  GPT-2-small set, one stream,
// before / now: update 640 / 553 us, Gram 386 / 374, Poly (whose fp32 A was a dword a load) 161 / 113, A' 152 / 126, other
// m x m products 124 / 116, the split of the raw steps 328 / 277; whole ELO-CELO2 step 6.65 / 6.23 ms, CELO2 on ResNet-50
// 1.63 / 1.49 ms.
// Only the lanes of one wave meet in a patch (2 KB a 32 columns) and a wave's LDS instructions execute in order, so the
// passes need no barrier, just the compiler kept from moving the reads over the writes.
template <int HI, int WN>
__device__ __forceinline__ void hf_store_planes(PYLO_LDS char* patch, const v16f (&acc)[HI][WN], hbits* __restrict__ D,
                                                int rows_d, int wi, int wj, int n_rows, int n_cols,
                                                hbits* __restrict__ D4, int rows4, float scale) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef PYLO_LDS s16x4 ls4;
  const int lane = threadIdx.x & 63;
  PYLO_LDS char* const put = patch + (lane & 31) * 32 + (lane >> 5) * 16;
  // the block's piece that the lane stores: sixteen lanes a (half, plane)
  PYLO_LDS char* const get = patch + ((lane >> 4) & 1) * 1024 + (lane >> 5) * 256 + (lane & 15) * 8;
#pragma unroll
  for (int pass = 0; pass < 2 * HI; ++pass) {
    const int hi = pass >> 1, b = pass & 1, row = wi + 32 * hi + 16 * b;
    if (row >= n_rows) break;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the patch is free: the previous pass has read it
#pragma unroll
    for (int hj = 0; hj < WN; ++hj) {
      const v16f& v = acc[hi][hj];
      u32x4 h, l;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        unsigned h1, l1;
        hf_split2(v[8 * b + 2 * u] * scale, v[8 * b + 2 * u + 1] * scale, h1, l1);
        h[u] = h1;
        l[u] = l1;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const u32x2 a = __builtin_amdgcn_permlane32_swap(h[u], h[u + 2], false, false);
        const u32x2 c = __builtin_amdgcn_permlane32_swap(l[u], l[u + 2], false, false);
        h[u] = a[0]; h[u + 2] = a[1];
        l[u] = c[0]; l[u + 2] = c[1];
      }
      *(luint4*)(put + hj * 2048) = h;
      *(luint4*)(put + hj * 2048 + 1024) = l;
      if (D4 != nullptr) {
        const int col = wj + 32 * hj;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const u32x2 a = __builtin_amdgcn_permlane16_swap(h[u], l[u], false, false);
          h[u] = a[0];
          l[u] = a[1];
        }
        hbits* p = D4 + hf_block(rows4, col, row) + lane * 8;
        if (col < n_cols) *(u32x4*)p = h;
        if (col + 16 < n_cols) *(u32x4*)(p + kNsBlock) = l;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c = 0; c < 2 * WN; ++c) {     // 16 columns = one block
      const int col = wj + 16 * c;
      if (col >= n_cols) continue;
      const s16x4 w0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)(get + c * 512 + (c >> 1) * 1024));
      const s16x4 w1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)(get + c * 512 + (c >> 1) * 1024 + 128));
      const u32x2 x = __builtin_bit_cast(u32x2, w0), y = __builtin_bit_cast(u32x2, w1);
      *(u32x4*)(D + hf_block(rows_d, row, col) + lane * 8) = u32x4{x[0], x[1], y[0], y[1]};
    }
  }
}

// Values past the matrix's edge are products of padding: zeros, unless a NaN or an infinity met them.
template <int HI, int WN>
__device__ __forceinline__ void hf_mask_edge(v16f (&acc)[HI][WN], int wi, int wj, int n_rows, int n_cols) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < HI; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (wi + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3) >= n_rows || wj + 32 * j + (lane & 31) >= n_cols) acc[i][j][r] = 0.0f;
}

// One launch = one product of one iteration, for every tensor (see the head of this file).
//   kNsGram    A = Xs Xs^T as fp32 and planes, both halves; a slab of a split product: fp32 partial tile only
//   kNsPoly    c2 A A + c1 A + c0 I as planes (buffer bufs.d), both halves; A: buffer kNsBufA and its fp32 copy
//   kNsProd    (buffer s1) (buffer s2) as planes (buffer d), both halves
//   kNsProdA   the same, into buffer d and into the fp32 copy of A
//   kNsUpdate  Xl' = Xl (buffer s1): planes of Xl' (buffer 1 - par) and Xs', or fp32 X in place of the raw step (`last`)
// WI, WN: the tile has 64 WI rows and 64 WN columns: 2, 2; updates with enough of them 2, 4; 1, 1 where a launch has less
// than a 128 x 128 tile a CU (ns_tile_edge).  KS: reduction steps of 16 a stage.
// Registers: 64 / 128 accumulator registers plus what the epilogues need; tiles of 256 columns are held to two
// waves per SIMD (256 registers: left alone the epilogue takes 296 and a CU runs one job at a time).
// Which matrices a launch is for, when the chain length is chosen per matrix (k_ns_hf_chain_flag): all of them; those
// whose first chain is the longer one; the others; or all, the others with another first operand buffer and `last`.
enum : int { kNsAll = 0, kNsLongOnly = 1, kNsShortOnly = 2, kNsBoth = 3 };
struct NsPick {
  const int* flags;
  int sel, s1_short, last_short;
  float acc_scale_short;   // with s1_short: that buffer's planes have a scale of their own
};

template <int OP, int WI, int WN, int KS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WN == 4 ? 2 : 3))) void k_ns_hf_gemm(const NsHfMat* __restrict__ mats, const NsItem* __restrict__ items,
                                                    const PyloTensorArgs* __restrict__ dyn, float* __restrict__ ws,
                                                    hbits* __restrict__ pw, int par, int last, NsBufs bufs, float c0,
                                                    float c1, float c2, NsPick pick) {
  extern __shared__ __attribute__((aligned(16))) char lds_[];
  PYLO_LDS char* lds = (PYLO_LDS char*)lds_;
  const NsItem it = items[blockIdx.x];
  if (it.mat < 0) return;   // a filler job
  if (pick.sel != kNsAll) {
    const bool longer = pick.flags[it.mat] != 0;
    if ((pick.sel == kNsLongOnly && !longer) || (pick.sel == kNsShortOnly && longer)) return;
    if (pick.sel == kNsBoth && !longer) {
      bufs.s1 = pick.s1_short;
      bufs.acc_scale = pick.acc_scale_short;
      last = pick.last_short;
    }
  }
  const NsHfMat mt = mats[it.mat];
  const PyloTensorArgs a = dyn[mt.tensor];
  if (a.grad == nullptr || !(a.flags & kArgOrthogonalize)) return;
  const int m = mt.m, n = mt.n;
  v16f acc[WI][WN];
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  const int i0 = it.tm * 64 * WI, j0 = it.tn * 64 * WN;
  // A 128 x 128 tile on the diagonal of a symmetric product: the 64 x 64 quadrant below the diagonal is the mirror image of the
  // one above it, which its own wave (wave 1) writes to both places; wave 2 computes and stores nothing.
  const int wave_u = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool diag = OP != kNsUpdate && WI == 2 && it.tm == it.tn;
  const bool idle = diag && wave_u == 2;
  if (OP == kNsGram) {
    const HfPlanes X{pw + mt.off_xs, mt.rows_m};
    hf_tile_product<WI, WN, KS>(X, i0, X, j0, it.k0, it.k1, lds, acc, !idle);
  } else if (OP == kNsPoly) {
    const HfPlanes A{pw + mt.off_p, mt.rows_m};
    hf_tile_product<WI, WN, KS>(A, i0, A, j0, it.k0, it.k1, lds, acc, !idle);
  } else if (OP == kNsUpdate) {
    const HfPlanes X{pw + (par ? mt.off_xl[1] : mt.off_xl[0]), mt.rows_n};   // no run-time index: the struct stays in registers
    const HfPlanes B{pw + mt.off_p + bufs.s1 * mt.p_stride, mt.rows_m};
    hf_tile_product<WI, WN, KS>(X, i0, B, j0, it.k0, it.k1, lds, acc);
  } else {
    const HfPlanes P1{pw + mt.off_p + bufs.s1 * mt.p_stride, mt.rows_m};
    const HfPlanes P2{pw + mt.off_p + bufs.s2 * mt.p_stride, mt.rows_m};
    hf_tile_product<WI, WN, KS>(P1, i0, P2, j0, it.k0, it.k1, lds, acc, !idle);
  }
  if (idle) return;
  // the operands' planes hold their matrices times a power of two each
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] *= bufs.acc_scale;
  const int n_i = OP == kNsUpdate ? n : m;   // rows of the output; its columns are always m
  const bool partial = OP == kNsGram && it.slab >= 0;
  const bool mirror = OP != kNsUpdate && (it.tm != it.tn || (WI == 2 && wave_u == 1));
  const int lane = threadIdx.x & 63;
  const int wi = i0 + (wave_u >> 1) * 32 * WI, wj = j0 + (wave_u & 1) * 32 * WN;   // origin of the wave's values
  if (wi + 32 * WI > n_i || wj + 32 * WN > m) hf_mask_edge<WI, WN>(acc, wi, wj, n_i, m);
  if (OP == kNsGram || OP == kNsPoly || OP == kNsProdA) {
    // the fp32 A: written, or Poly's transform of the accumulators
    const size_t e = WI == 2 ? hf_a32(hf_tile_index(m, it.tm, it.tn), wave_u, 0, 0, 0, lane)
                             : hf_a32(hf_tile_index(m, it.tm >> 1, it.tn >> 1), (it.tm & 1) * 2 + (it.tn & 1), wave_u >> 1, wave_u & 1, 0, lane);
    float* A = ws + (partial ? mt.off_part + (size_t)it.slab * mt.a_floats : mt.off_a) + e;
#pragma unroll
    for (int hi = 0; hi < WI; ++hi)
#pragma unroll
      for (int hj = 0; hj < WN; ++hj)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          gv4f* p = (gv4f*)(A + ((hi * WN + hj) * 4 + q) * 256);
          if (OP == kNsPoly) {
            const v4f aij = *p;
            const int d = wj + hj * 32 + (lane & 31) - (wi + hi * 32 + 8 * q + 4 * (lane >> 5));   // the register on the diagonal, if 0 .. 3
            const bool in = wj + hj * 32 + (lane & 31) < m;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float x = acc[hi][hj][4 * q + r];
              x = c2 * x + c1 * aij[r] + (d == r && in ? c0 : 0.0f);
              acc[hi][hj][4 * q + r] = x;
            }
          } else {
            *p = v4f{acc[hi][hj][4 * q], acc[hi][hj][4 * q + 1], acc[hi][hj][4 * q + 2], acc[hi][hj][4 * q + 3]};
          }
        }
    if (partial) return;
  }
  if (OP == kNsUpdate && last) {
    // fp32 X in place of the raw step
    float* xout = a.step_out + mt.elem_off;
    if (!mt.tall && (mt.C & 3) == 0) {
      // X = Xs, m x n, 16-byte aligned rows: 32 x 32 values through the wave's LDS patch (rows of 36 floats), so that eight
      // lanes store 128 consecutive bytes of a row
      typedef PYLO_LDS v4f lv4f;
      PYLO_LDS char* patch = lds + wave_u * (32 * 144);
#pragma unroll
      for (int hi = 0; hi < WI; ++hi)
#pragma unroll
        for (int hj = 0; hj < WN; ++hj) {
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *(lv4f*)(patch + (lane & 31) * 144 + 32 * q + 16 * (lane >> 5)) =
                v4f{acc[hi][hj][4 * q], acc[hi][hj][4 * q + 1], acc[hi][hj][4 * q + 2], acc[hi][hj][4 * q + 3]};
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int cl = 8 * q + (lane >> 3), col = wj + hj * 32 + cl, row = wi + hi * 32 + 4 * (lane & 7);
            const v4f v = *(lv4f*)(patch + cl * 144 + 16 * (lane & 7));
            if (col < m && row < n) *(gv4f*)(xout + (size_t)col * n + row) = v;
          }
        }
    } else {
#pragma unroll
      for (int hi = 0; hi < WI; ++hi)
#pragma unroll
        for (int hj = 0; hj < WN; ++hj) {
          const int col = wj + hj * 32 + (lane & 31);
          if (col >= m) continue;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = wi + hi * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (row < n) xout[mt.tall ? (size_t)row * m + col : (size_t)col * n + row] = acc[hi][hj][r];
          }
        }
    }
    return;
  }
  // planes: A and B' in both halves (the mirrored tile is the other orientation), Xl' and Xs'
  PYLO_LDS char* patch = lds + wave_u * (2048 * WN);
  if (OP == kNsUpdate) {
    hf_store_planes<WI, WN>(patch, acc, pw + (par ? mt.off_xl[0] : mt.off_xl[1]), mt.rows_n, wi, wj, n, m, pw + mt.off_xs, mt.rows_m,
                           bufs.out_scale);
  } else {
    hbits* D = pw + mt.off_p + (OP == kNsGram ? (int)kNsBufA : bufs.d) * mt.p_stride;
    hf_store_planes<WI, WN>(patch, acc, D, mt.rows_m, wi, wj, m, m, mirror ? D : nullptr, mt.rows_m, bufs.out_scale);
  }
}

// A = sum over the slabs' partial matrices, in slab order, as fp32 and as planes (both halves): a wave for each 32 x 32 of
// the tiles on and above the diagonal.
__global__ __launch_bounds__(64) void k_ns_hf_gram_reduce(const NsHfMat* __restrict__ mats, const int* __restrict__ split_mats,
                                                          const PyloTensorArgs* __restrict__ dyn, float* __restrict__ ws,
                                                          hbits* __restrict__ pw, NsPick pick, float out_scale) {
  __shared__ __attribute__((aligned(16))) char patch[2048];
  if (pick.sel == kNsShortOnly && pick.flags[split_mats[blockIdx.y]] != 0) return;
  const NsHfMat mt = mats[split_mats[blockIdx.y]];
  const PyloTensorArgs a = dyn[mt.tensor];
  if (a.grad == nullptr || !(a.flags & kArgOrthogonalize)) return;
  const int m = mt.m, nt = (m + kNsTile - 1) / kNsTile, lane = threadIdx.x;
  const int tile = blockIdx.x >> 4, wave = (blockIdx.x >> 2) & 3, hi = (blockIdx.x >> 1) & 1, hj = blockIdx.x & 1;
  if (tile >= hf_tiles_upper(m)) return;
  int tm = 0, left = tile;
  while (left >= nt - tm) left -= nt - tm++;
  const int tn = tm + left;
  if (tm == tn && wave == 2) return;   // the mirror image of wave 1's
  const int wi = tm * kNsTile + (wave >> 1) * 64 + hi * 32, wj = tn * kNsTile + (wave & 1) * 64 + hj * 32;
  const size_t e = hf_a32(tile, wave, hi, hj, 0, lane);
  const float* p = ws + mt.off_part + e;
  v16f acc[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.0f;
  for (int s0 = 0; s0 < mt.n_slabs; s0 += 4) {
    v4f v[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[u][q] = s0 + u < mt.n_slabs ? *(const gv4f*)(p + (size_t)(s0 + u) * mt.a_floats + q * 256) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][0][r] += v[u][r >> 2][r & 3];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *(gv4f*)(ws + mt.off_a + e + q * 256) = v4f{acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2], acc[0][0][4 * q + 3]};
  hbits* P = pw + mt.off_p;   // buffer A
  hf_store_planes<1, 1>((PYLO_LDS char*)patch, acc, P, mt.rows_m, wi, wj, m, m, tm != tn || wave == 1 ? P : nullptr, mt.rows_m, out_scale);
}

// X0 = raw * s (s = 1 / (||raw|| + eps), scale[mat]) as planes in both layouts.  One block = one 64 x 64
// tile of the raw step (R x C): the planes in which the tensor's rows stay rows are written straight from
// the loaded values, the transposed planes through LDS.
// The length of a matrix's first chain.  With X scaled to unit Frobenius norm, ||A||_F (A = X X^T as computed) bounds
// the largest eigenvalue of A from above; what a chain of three iterations adds to the error of the result is
// proportional to it, 196 eps_A lambda_max against 16 eps_A lambda_max for a pair (head of this file), so three
// iterations are taken where ||A||_F^2 <= tau^2, with tau = 16 / 196: no worse there than a pair is on any matrix.
// Two launches, sums in a fixed order: 64 x 64 elements of A per block, then one block per matrix.
// items[b] = {matrix, 64 x 64 part (tile x 4 + wave) of its fp32 A}: parts off the diagonal count twice
__global__ __launch_bounds__(256) void k_ns_hf_chain_sumsq(const NsHfMat* __restrict__ mats, const Item* __restrict__ items,
                                                           const PyloTensorArgs* __restrict__ dyn, const float* __restrict__ ws,
                                                           float* __restrict__ part) {
  __shared__ float red[4];
  const Item it = items[blockIdx.x];
  const NsHfMat mt = mats[it.tensor];
  const PyloTensorArgs a = dyn[mt.tensor];
  if (a.grad == nullptr || !(a.flags & kArgOrthogonalize)) return;
  const int nt = (mt.m + kNsTile - 1) / kNsTile, wave = it.a & 3;
  int tm = 0, left = it.a >> 2;
  while (left >= nt - tm) left -= nt - tm++;
  // the mirror image of wave 1's, and parts past the matrix: nobody writes them
  if ((left == 0 && wave == 2) || (tm + left) * kNsTile + (wave & 1) * 64 >= mt.m) {
    if (threadIdx.x == 0) part[mt.fpart0 + it.a] = 0.0f;
    return;
  }
  const float* A = ws + mt.off_a + (size_t)it.a * 4096;
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const v4f v = *(const gv4f*)(A + 1024 * i + 4 * threadIdx.x);
    s = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, s))));
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[mt.fpart0 + it.a] = (left > 0 || wave == 1 ? 2.0f : 1.0f) * ((red[0] + red[1]) + (red[2] + red[3]));
}

__global__ __launch_bounds__(64) void k_ns_hf_chain_flag(const NsHfMat* __restrict__ mats, const int* __restrict__ list,
                                                         const PyloTensorArgs* __restrict__ dyn, const float* __restrict__ part,
                                                         float tau2, int* __restrict__ flags) {
  const int q = list[blockIdx.x];
  const NsHfMat mt = mats[q];
  const PyloTensorArgs a = dyn[mt.tensor];
  if (a.grad == nullptr || !(a.flags & kArgOrthogonalize)) return;
  float s = 0.0f;
  for (int b = threadIdx.x; b < mt.n_fpart; b += 64) s += part[mt.fpart0 + b];
  s = wave_sum(s);
  if (threadIdx.x == 0) flags[q] = s <= tau2 ? 1 : 0;
}

struct NsTileItem { int mat, tr, tc; };

__global__ __launch_bounds__(256) void k_ns_hf_split(const NsHfMat* __restrict__ mats, const NsTileItem* __restrict__ items,
                                                     const PyloTensorArgs* __restrict__ dyn, const float* __restrict__ scale,
                                                     hbits* __restrict__ pw, float plane_scale) {
  constexpr int RP = 72;   // numbers per row of the tile in LDS: 64 + 8, rows stay 16-byte aligned
  __shared__ __attribute__((aligned(16))) hbits tile[kNsPl][64][RP];
  const NsTileItem it = items[blockIdx.x];
  const NsHfMat mt = mats[it.mat];
  const PyloTensorArgs a = dyn[mt.tensor];
  if (a.grad == nullptr || !(a.flags & kArgOrthogonalize)) return;
  const float s = scale[it.mat] * plane_scale;
  const int R = mt.R, C = mt.C;
  const float* raw = a.step_out + mt.elem_off;
  const bool vec_in = (C & 3) == 0;
  // direct planes: the tensor's rows are the planes' rows; transposed planes: its columns are
  hbits* direct = pw + (mt.tall ? mt.off_xl[0] : mt.off_xs);
  hbits* transp = pw + (mt.tall ? mt.off_xs : mt.off_xl[0]);
  const int rows_d = mt.tall ? mt.rows_n : mt.rows_m, rows_t = mt.tall ? mt.rows_m : mt.rows_n;
  const int r0 = it.tr * 64, c0 = it.tc * 64;
  const int t = threadIdx.x;
  // Eight consecutive columns of one row a lane and pass: 32 bytes read, 16 bytes per plane into the tile in LDS.  Columns and
  // rows past the matrix are zeros, which land in the planes' padding.
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int u = pass * 256 + t, lr = u >> 3, lc = 8 * (u & 7);
    const int r = r0 + lr, c = c0 + lc;
    float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (r < R && c < C) {
      const float* src = raw + (size_t)r * C + c;
      if (vec_in) {
        const v4f x = *(const gv4f*)src;
        v[0] = x.x * s; v[1] = x.y * s; v[2] = x.z * s; v[3] = x.w * s;
        if (c + 4 < C) {
          const v4f y = *(const gv4f*)(src + 4);
          v[4] = y.x * s; v[5] = y.y * s; v[6] = y.z * s; v[7] = y.w * s;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c + e < C) v[e] = *(const gfloat*)(src + e) * s;
      }
    }
    u32x4 h, l;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      unsigned h1, l1;
      hf_split2(v[2 * q], v[2 * q + 1], h1, l1);
      h[q] = h1;
      l[q] = l1;
    }
    *(luint4*)&tile[0][lr][lc] = h;
    *(luint4*)&tile[1][lr][lc] = l;
  }
  __syncthreads();
  // Sixteen blocks of each orientation, four a wave (those of sixteen rows of the tile), every store a block in lane order:
  // sixteen lanes a (half, plane).  Transposed pieces are read with ds_read_b64_tr_b16 (lane i of sixteen gets column i of four rows).
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef PYLO_LDS s16x4 ls4;
  const int lane = t & 63, rb = 16 * (t >> 6), plane = (lane >> 4) & 1, half = lane >> 5, i = lane & 15;
  if (r0 + rb >= R) return;
#pragma unroll
  for (int cb = 0; cb < 64; cb += 16) {
    if (c0 + cb >= C) break;
    *(u32x4*)(direct + hf_block(rows_d, r0 + rb, c0 + cb) + lane * 8) = *(const luint4*)&tile[plane][rb + i][cb + 8 * half];
    const s16x4 w0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)&tile[plane][rb + 8 * half + (i >> 2)][cb + 4 * (i & 3)]);
    const s16x4 w1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)&tile[plane][rb + 8 * half + 4 + (i >> 2)][cb + 4 * (i & 3)]);
    const u32x2 x = __builtin_bit_cast(u32x2, w0), y = __builtin_bit_cast(u32x2, w1);
    *(u32x4*)(transp + hf_block(rows_t, c0 + cb, r0 + rb) + lane * 8) = u32x4{x[0], x[1], y[0], y[1]};
  }
}

}  // namespace pylo
