// ELO-CELO2 / CELO2 MLP tensors whose feature normalisers are not tensor-wide: tensors with more
// than two dims (the naive class normalises every feature over the last two dims only,
// ELO_CELO2_naive.py:217-218, so each slice of the last two dims has its own 30 normalisers) and
// tensors with fewer than two dims on the MLP path (use_adamw_for_1d=False: per-element Adafactor
// accumulator, the first nine feature groups only, :166-169,180-191).  The row / column vectors of an
// N-D tensor still span the whole tensor and come from the P0 / V0 passes; everything after that is
// local to a slice, so one pass does statistics, MLP and the accumulator writes.
//
// Short slices of tensors with more than two dims (conv kernels: 1 .. 32 elements) are packed, as many whole ones as fit, into a
// wave of one lane an element (k_celo2_slices_wave).  All others are walked twice (sum of squares, then apply) by k_celo2_slices,
// by one lane when the slice is short and by one wave otherwise: written for correctness on any shape (patch embeddings, biases).
#pragma once

#include "k_velo.h"

namespace pylo {

constexpr int kSliceLaneMax = 32;  // slices up to this length are packed into waves, or walked by a single lane
// launches of k_celo2_slices_wave: slices of one element, of nine (3 x 3), of any other length; and those whose row and
// column channels are not the same for all slices that meet a vector's entries (slice_runs)
enum : int { kSliceOne = 0, kSliceNine = 1, kSliceAny = 2, kSliceGather = 3, kSliceWaveClasses = 4 };
// raw CELO2 MLP block: w_in (30,8) | b_in 8 | w_h (8,8) | b_h 8 | w_out (8,3) | b_out 3, all (in, out)
constexpr int kC2RawBI = 240, kC2RawWH = 248, kC2RawBH = 312, kC2RawWO = 320, kC2RawBO = 344;

// Accumulators of element idx advanced, and its feature channels in the reference's 30-channel order.
template <bool VEC>
__device__ __forceinline__ void slice_element(const TDesc& d, const PyloTensorArgs& a, long long idx,
                                              const EmaConsts& e, const PyloDecays& dec,
                                              const float* __restrict__ fac_tab, float (&f)[30], float (&m)[3],
                                              float& rms, float (&fv)[3]) {
  float f18[kNStat];
  if constexpr (VEC) {
    const long long n = d.n;
    const float g = cond_grad(*(const gfloat*)(a.grad + idx), d.gscale, a.clip_val, d.nan0);
    const float p = *(const gfloat*)(a.param + idx);
    rms = *(const gfloat*)(a.rms + idx);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      m[k] = *(const gfloat*)(a.mom + k * n + idx);
      fv[k] = *(const gfloat*)(a.fac_v + k * n + idx);
    }
    vec_update(e, dec, g, m, rms, fv);
    float rf[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) rf[k] = rsq(fmaxf(fv[k] + 1e-9f, 1e-9f));
    lo_features(g, p, m, rms, rf, 1e-8f, f18);
#pragma unroll
    for (int c = 0; c < 15; ++c) f[c] = f18[c];
#pragma unroll
    for (int c = 15; c < 30; ++c) f[c] = 0.0f;
  } else {
    ElemIn<1> x;
    lo_load<1, true>(d, a, idx, fac_tab, x);
    ema_update(e, x.g[0], x.m[0], x.rms[0]);
    lo_features(x.g[0], x.p[0], x.m[0], x.rms[0], x.rfcf[0], 1e-8f, f18);
#pragma unroll
    for (int c = 0; c < 15; ++c) f[c] = f18[c];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float fr = *(const gfloat*)(a.fac_r + (size_t)k * d.len[0] + x.i0);  // vector 0 is the row vector
      const float fc = *(const gfloat*)(a.fac_c + (size_t)k * d.len[1] + x.i1);
      f[15 + k] = fr;
      f[18 + k] = fc;
      f[21 + k] = rsq(fr + 1e-8f);
      f[24 + k] = rsq(fc + 1e-8f);
      f[27 + k] = f18[15 + k];
      m[k] = x.m[0][k];
    }
    rms = x.rms[0];
  }
}

// direction * exp(magnitude * exp_mult) from the normalised features (ELO_CELO2_naive.py:219-229)
template <int NC>
__device__ __forceinline__ float slice_mlp(const float (&f)[30], const float (&s)[30], const cfloat* w, float exp_mult) {
  float h0[8], h1[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) h0[j] = w[kC2RawBI + j];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const float x = f[c] * s[c];
#pragma unroll
    for (int j = 0; j < 8; ++j) h0[j] = fmaf(x, w[c * 8 + j], h0[j]);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) h1[j] = w[kC2RawBH + j];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float hk = fmaxf(h0[k], 0.0f);
#pragma unroll
    for (int j = 0; j < 8; ++j) h1[j] = fmaf(hk, w[kC2RawWH + k * 8 + j], h1[j]);
  }
  float o0 = w[kC2RawBO + 0], o1 = w[kC2RawBO + 1];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float hk = fmaxf(h1[k], 0.0f);
    o0 = fmaf(hk, w[kC2RawWO + k * 3 + 0], o0);
    o1 = fmaf(hk, w[kC2RawWO + k * 3 + 1], o1);
  }
  return o0 * expf(o1 * exp_mult);
}

// One slice: elements first + j for j = j0, j0 + dj, ... < S.  LANE: the lane owns the slice (no
// reduction across lanes); else the 64 lanes of the wave share it.
template <bool VEC, bool LANE>
__device__ __forceinline__ void slice_run(const TDesc& d, const PyloTensorArgs& a, long long first, int S,
                                          const EmaConsts& e, const PyloDecays& dec,
                                          const float* __restrict__ fac_tab, const cfloat* w) {
  constexpr int NC = VEC ? 15 : 30;
  const int j0 = LANE ? 0 : (threadIdx.x & 63), dj = LANE ? 1 : 64;
  float acc[30];
#pragma unroll
  for (int c = 0; c < 30; ++c) acc[c] = 0.0f;
  for (int j = j0; j < S; j += dj) {
    float f[30], m[3], rms, fv[3];
    slice_element<VEC>(d, a, first + j, e, dec, fac_tab, f, m, rms, fv);
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = fmaf(f[c], f[c], acc[c]);
  }
  float s[30];
#pragma unroll
  for (int c = 0; c < 30; ++c) {
    const float tot = (LANE || c >= NC) ? acc[c] : wave_sum(acc[c]);
    s[c] = rsq(1e-9f + tot / (float)S);
  }
  const long long n = d.n;
  for (int j = j0; j < S; j += dj) {
    const long long idx = first + j;
    float f[30], m[3], rms, fv[3];
    slice_element<VEC>(d, a, idx, e, dec, fac_tab, f, m, rms, fv);
    const float step = slice_mlp<NC>(f, s, w, a.exp_mult);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      *(gfloat*)(a.mom + k * n + idx) = m[k];
      if constexpr (VEC) *(gfloat*)(a.fac_v + k * n + idx) = fv[k];
    }
    *(gfloat*)(a.rms + idx) = rms;
    *(gfloat*)(a.step_out + idx) = step;
  }
}

// What an element of a tensor with more than two dims reads of the factored statistics: the products of the table
// (row and column) and the two accumulators themselves, three decays each.  Gathered apart from the arithmetic so
// that a walk over a slice can have the next element's loads in flight while it works on this one.
struct SliceFac { float4 fa, fb; float fr[3], fc[3]; };
__device__ __forceinline__ SliceFac slice_gather_nd(const TDesc& d, const PyloTensorArgs& a, long long idx,
                                                    const float* __restrict__ fac_tab) {
  const unsigned u = (unsigned)idx;
  const unsigned s0 = (unsigned)d.nd_stride[0], s1 = (unsigned)d.nd_stride[1];
  const int i0 = (int)(fd_div(u, d.nd_div_blk[0]) * s0 + (u - fd_div(u, d.nd_div_st[0]) * s0));
  const int i1 = (int)(fd_div(u, d.nd_div_blk[1]) * s1 + (u - fd_div(u, d.nd_div_st[1]) * s1));
  SliceFac x;
  x.fa = load_f4(fac_tab + d.fac_off[0] + (size_t)i0 * 4);
  x.fb = load_f4(fac_tab + d.fac_off[1] + (size_t)i1 * 4);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    x.fr[k] = *(const gfloat*)(a.fac_r + (size_t)k * d.len[0] + i0);  // vector 0 is the row vector
    x.fc[k] = *(const gfloat*)(a.fac_c + (size_t)k * d.len[1] + i1);
  }
  return x;
}

// The feature channels of one element of a tensor with more than two dims from its inputs and accumulators as
// they stand after this step's update (what slice_element computes after loading and updating them).
__device__ __forceinline__ void slice_features_nd(const SliceFac& x, float g, float p, const float (&m)[3], float rms,
                                                  float (&f)[30]) {
  const float rfcf[3] = {x.fa.x * x.fb.x, x.fa.y * x.fb.y, x.fa.z * x.fb.z};
  float f18[kNStat];
  lo_features(g, p, m, rms, rfcf, 1e-8f, f18);
#pragma unroll
  for (int c = 0; c < 15; ++c) f[c] = f18[c];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    f[15 + k] = x.fr[k];
    f[18 + k] = x.fc[k];
    f[21 + k] = rsq(x.fr[k] + 1e-8f);
    f[24 + k] = rsq(x.fc[k] + 1e-8f);
    f[27 + k] = f18[15 + k];
  }
}

// The raw MLP block as the lane-local matrix instruction wants it (mfma_w4: four weights of one input from four
// neighbouring lanes): 96 groups of four floats in six registers a lane.  w_in, b_in, w_h, b_h are already rows of
// eight = two groups; a row of w_out (three outputs) and b_out become a group each, padded with a zero.
constexpr int kC2GrpBI = 60, kC2GrpWH = 62, kC2GrpBH = 78, kC2GrpWO = 80, kC2GrpBO = 88;
__device__ __forceinline__ void slice_mlp_weights(const float* __restrict__ mlp, float (&wreg)[6]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    const int q = 64 * r + lane, g = q >> 2, j = q & 3;
    int src = q;                                   // w_in | b_in | w_h | b_h: as stored
    if (g >= kC2GrpBO) src = g == kC2GrpBO && j < 3 ? kC2RawBO + j : -1;
    else if (g >= kC2GrpWO) src = j < 3 ? kC2RawWO + 3 * (g - kC2GrpWO) + j : -1;
    wreg[r] = src >= 0 ? *(const gfloat*)(mlp + src) : 0.0f;
  }
}

// direction * exp(magnitude * exp_mult) from the normalised features, on the matrix pipe: every lane of the wave
// must get here (lanes without an element pass zeros and drop the result).
__device__ __forceinline__ float slice_mlp_mfma(const float (&f)[30], const float (&s)[30], const float (&wreg)[6],
                                                float exp_mult) {
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  v4f ha = mfma_w4(wreg[kC2GrpBI / 16], 1.0f, zero, kC2GrpBI % 16);
  v4f hb = mfma_w4(wreg[(kC2GrpBI + 1) / 16], 1.0f, zero, (kC2GrpBI + 1) % 16);
#pragma unroll
  for (int c = 0; c < 30; ++c) {
    const float x = f[c] * s[c];
    ha = mfma_w4(wreg[(2 * c) / 16], x, ha, (2 * c) % 16);
    hb = mfma_w4(wreg[(2 * c + 1) / 16], x, hb, (2 * c + 1) % 16);
  }
  v4f ga = mfma_w4(wreg[kC2GrpBH / 16], 1.0f, zero, kC2GrpBH % 16);
  v4f gb = mfma_w4(wreg[(kC2GrpBH + 1) / 16], 1.0f, zero, (kC2GrpBH + 1) % 16);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float hk = relu(k < 4 ? ha[k] : hb[k - 4]);
    ga = mfma_w4(wreg[(kC2GrpWH + 2 * k) / 16], hk, ga, (kC2GrpWH + 2 * k) % 16);
    gb = mfma_w4(wreg[(kC2GrpWH + 2 * k + 1) / 16], hk, gb, (kC2GrpWH + 2 * k + 1) % 16);
  }
  v4f o = mfma_w4(wreg[kC2GrpBO / 16], 1.0f, zero, kC2GrpBO % 16);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float hk = relu(k < 4 ? ga[k] : gb[k - 4]);
    o = mfma_w4(wreg[(kC2GrpWO + k) / 16], hk, o, (kC2GrpWO + k) % 16);
  }
  return o[0] * expf(o[1] * exp_mult);
}

// The same where the row and column channels' part of the first layer comes from the term tables (ta, tb: vector 0 with the bias,
// vector 1): the eighteen channels of an element alone.
__device__ __forceinline__ float slice_mlp_terms(const float (&f)[kNStat], const float (&s)[kNStat], const v4f (&ta)[2], const v4f (&tb)[2],
                                                 const float (&wreg)[6], float exp_mult) {
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  v4f ha = ta[0] + tb[0], hb = ta[1] + tb[1];
#pragma unroll
  for (int q = 0; q < kNStat; ++q) {
    const int c = q < 15 ? q : q + 12;
    const float x = f[q] * s[q];
    ha = mfma_w4(wreg[(2 * c) / 16], x, ha, (2 * c) % 16);
    hb = mfma_w4(wreg[(2 * c + 1) / 16], x, hb, (2 * c + 1) % 16);
  }
  v4f ga = mfma_w4(wreg[kC2GrpBH / 16], 1.0f, zero, kC2GrpBH % 16);
  v4f gb = mfma_w4(wreg[(kC2GrpBH + 1) / 16], 1.0f, zero, (kC2GrpBH + 1) % 16);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float hk = relu(k < 4 ? ha[k] : hb[k - 4]);
    ga = mfma_w4(wreg[(kC2GrpWH + 2 * k) / 16], hk, ga, (kC2GrpWH + 2 * k) % 16);
    gb = mfma_w4(wreg[(kC2GrpWH + 2 * k + 1) / 16], hk, gb, (kC2GrpWH + 2 * k + 1) % 16);
  }
  v4f o = mfma_w4(wreg[kC2GrpBO / 16], 1.0f, zero, kC2GrpBO % 16);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float hk = relu(k < 4 ? ga[k] : gb[k - 4]);
    o = mfma_w4(wreg[(kC2GrpWO + k) / 16], hk, o, (kC2GrpWO + k) % 16);
  }
  return o[0] * expf(o[1] * exp_mult);
}

// Short slices (1 .. 32 elements) of tensors with more than two dims: a wave takes the 64 / S whole slices that fit it, a
// lane an element, consecutive in every array, so that all loads and stores are coalesced, every input is read and every
// output written once, and an element's features are computed once.  The sums over a slice go through the wave's own
// LDS: f^2 in as [channel][lane], then a lane sums a (slice, channel) at a time -- in the slice's order -- and leaves its
// normaliser, which the slice's lanes read back.
// TERMS: a factored vector's entries lie in runs of S that the slices meet whole (slice_runs), so the twelve channels that
// depend on the row or the column only have one normaliser a run: k_v0b has normalised them and pushed them through the
// first layer, [entry][8] in the term tables, and 24 of the 89 rank-1 updates of an element's MLP and 18 of its reciprocal
// roots go.  Else (small tensors whose factored dims are dims of the slice) they are gathered and normalised like the others.
// What bounds it: instruction issue -- some 370 instructions a trip, 63 of them rank-1 updates and 19 reciprocal roots -- where the
// bytes would take half the time.  ResNet-50's kernels, a lane walking its slice twice through LDS before / now: 12.1 M
// elements of 1 x 1 227 / 145 us (3.7 TB/s), 11.3 M of 3 x 3 300 / 161; whole CELO2 step 1.19 / 0.98 ms.
// Item: tensor, first slice of the block, trips (of 64 / S slices) a wave.  LEN: the slice length, 0: any.
constexpr int kSliceLd = 65;       // floats per channel of the squares in LDS
template <int LEN, bool TERMS>
__global__ __launch_bounds__(kThreads) void k_celo2_slices_wave(const TDesc* __restrict__ descs,
                                                                const PyloTensorArgs* __restrict__ dyn,
                                                                const Item* __restrict__ items,
                                                                const float* __restrict__ fac_tab,
                                                                const float* __restrict__ term_tab,
                                                                const Globals* __restrict__ gl, PyloDecays dec,
                                                                const float* __restrict__ mlp) {
  constexpr int NC = TERMS ? kNStat : 30, NCP = TERMS ? 20 : 32;   // channels, and the pitch of a slice's normalisers
  // squares, then the normalisers of at most 32 slices and of the lanes past the last whole one
  __shared__ float lds[kWaves][LEN == 1 ? 1 : NC * kSliceLd + 33 * NCP];
  const Item it = items[blockIdx.x];
  TDesc d = descs[it.tensor];
  const PyloTensorArgs a = dyn[it.tensor];
  if (a.grad == nullptr) return;
  set_grad_scale(d, a, gl, it.tensor);
  const EmaConsts e = make_ema(dec);
  const int S = LEN ? LEN : d.slice_len, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int spw = 64 / S, per = spw * S, sl = lane / S;
  const long long n = d.n;
  const float inv_s = 1.0f / (float)S;
  float* sq = lds[wave];
  float* nrm = sq + NC * kSliceLd;
  // the lane's (slice, channel) pairs: its slice, its first channel, and how many channels the wave sums at a time
  const int pc0 = lane / spw, ps = lane - pc0 * spw, pcs = 64 / spw;
  float wreg[6];
  slice_mlp_weights(mlp, wreg);
  struct In { float g, p, m[3], r; };
  auto fetch = [&](long long first, unsigned off) {   // (the wave's first element, the lane's from there)
    In x;
    x.g = *(const gfloat*)(a.grad + first + off);
    x.p = *(const gfloat*)(a.param + first + off);
    x.m[0] = *(const gfloat*)(a.mom + first + off);
    x.m[1] = *(const gfloat*)(a.mom + n + first + off);
    x.m[2] = *(const gfloat*)(a.mom + 2 * n + first + off);
    x.r = *(const gfloat*)(a.rms + first + off);
    return x;
  };
  // Lanes past the last whole slice of the wave or of the tensor work on the wave's first element and store nothing (the
  // matrix instructions want the whole wave).
  long long e0 = ((long long)it.a + (long long)wave * it.b * spw) * S;
  if (e0 >= n) return;
  auto mine = [&](long long first) { return lane < per && first + lane < n; };
  In cur = fetch(e0, mine(e0) ? lane : 0);
  for (int trip = 0; trip < it.b && e0 < n; ++trip, e0 += per) {
    const bool live = mine(e0);
    const unsigned off = live ? lane : 0;
    const long long idx = e0 + off;
    const long long next = trip + 1 < it.b && e0 + per < n ? e0 + per : e0;
    const In nxt = fetch(next, mine(next) ? lane : 0);
    float f[NC], sc[NC], m[3] = {cur.m[0], cur.m[1], cur.m[2]}, rms = cur.r;
    const float g = cond_grad(cur.g, d.gscale, a.clip_val, d.nan0);
    v4f ta[2], tb[2];
    if constexpr (TERMS) {
      const unsigned u = (unsigned)idx;
      const unsigned s0 = (unsigned)d.nd_stride[0], s1 = (unsigned)d.nd_stride[1];
      const size_t i0 = fd_div(u, d.nd_div_blk[0]) * s0 + (u - fd_div(u, d.nd_div_st[0]) * s0);
      const size_t i1 = fd_div(u, d.nd_div_blk[1]) * s1 + (u - fd_div(u, d.nd_div_st[1]) * s1);
      const float4 fa = load_f4(fac_tab + d.fac_off[0] + i0 * 4), fb = load_f4(fac_tab + d.fac_off[1] + i1 * 4);
      const gv4f* t0 = (const gv4f*)(term_tab + d.term_off[0] + i0 * 8);
      const gv4f* t1 = (const gv4f*)(term_tab + d.term_off[1] + i1 * 8);
      ta[0] = t0[0]; ta[1] = t0[1];
      tb[0] = t1[0]; tb[1] = t1[1];
      ema_update(e, g, m, rms);
      const float rfcf[3] = {fa.x * fb.x, fa.y * fb.y, fa.z * fb.z};
      lo_features(g, cur.p, m, rms, rfcf, 1e-8f, f);
    } else {
      const SliceFac fac = slice_gather_nd(d, a, idx, fac_tab);
      ema_update(e, g, m, rms);
      slice_features_nd(fac, g, cur.p, m, rms, f);
    }
    if constexpr (LEN == 1) {
#pragma unroll
      for (int c = 0; c < NC; ++c) sc[c] = rsq(1e-9f + f[c] * f[c]);
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the previous trip's reads are done
#pragma unroll
      for (int c = 0; c < NC; ++c) sq[c * kSliceLd + lane] = f[c] * f[c];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int c = pc0; c < NC && pc0 < pcs; c += pcs) {
        const float* q = sq + c * kSliceLd + ps * S;
        float t = 0.0f;
        if constexpr (LEN != 0) {
#pragma unroll
          for (int j = 0; j < LEN; ++j) t += q[j];
        } else {
          for (int j = 0; j < S; ++j) t += q[j];
        }
        nrm[ps * NCP + c] = rsq(1e-9f + t * inv_s);   // the mean by the reciprocal
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int c = 0; c < NC; ++c) sc[c] = nrm[(lane < per ? sl : 0) * NCP + c];
    }
    float step;
    if constexpr (TERMS) step = slice_mlp_terms(f, sc, ta, tb, wreg, a.exp_mult);
    else step = slice_mlp_mfma(f, sc, wreg, a.exp_mult);
    if (live) {
      *(gfloat*)(a.mom + e0 + off) = m[0];
      *(gfloat*)(a.mom + n + e0 + off) = m[1];
      *(gfloat*)(a.mom + 2 * n + e0 + off) = m[2];
      *(gfloat*)(a.rms + e0 + off) = rms;
      *(gfloat*)(a.step_out + e0 + off) = step;
    }
    cur = nxt;
  }
}

// Item: tensor, first slice of the block.  A block covers 256 slices (one per lane) or 4 (one per wave)."
__global__ __launch_bounds__(kThreads) void k_celo2_slices(const TDesc* __restrict__ descs,
                                                           const PyloTensorArgs* __restrict__ dyn,
                                                           const Item* __restrict__ items,
                                                           const float* __restrict__ fac_tab,
                                                           const Globals* __restrict__ gl, PyloDecays dec,
                                                           const float* __restrict__ mlp) {
  const Item it = items[blockIdx.x];
  TDesc d = descs[it.tensor];
  const PyloTensorArgs a = dyn[it.tensor];
  if (a.grad == nullptr) return;
  set_grad_scale(d, a, gl, it.tensor);
  const EmaConsts e = make_ema(dec);
  const cfloat* w = launder(mlp);
  const int S = d.slice_len;
  const long long n_slices = d.n / S;
  const bool vec = d.mode == kModeVec;
  if (S <= kSliceLaneMax) {
    const long long sl = (long long)it.a + threadIdx.x;
    if (sl >= n_slices) return;
    if (vec) slice_run<true, true>(d, a, sl * S, S, e, dec, fac_tab, w);
    else slice_run<false, true>(d, a, sl * S, S, e, dec, fac_tab, w);
  } else {
    const long long sl = (long long)it.a + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (sl >= n_slices) return;
    if (vec) slice_run<true, false>(d, a, sl * S, S, e, dec, fac_tab, w);
    else slice_run<false, false>(d, a, sl * S, S, e, dec, fac_tab, w);
  }
}

}  // namespace pylo
