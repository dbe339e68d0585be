// Fused learned-optimizer step for MI355X (gfx950): the C ABI of include/pylo_mi355.h.
//
// Pipeline of one ELO-CELO2 step over all tensors of a plan (6 launches, no host sync):
//   k_p0 (pass 0)   row / column sums of g^2 per tile, sum g^2 and clamp flag per block     4 B/elem
//   k_gnorm         global gradient norm, clamp flag
//   k_p0 (pass 1)   exits at once unless some |g| exceeded the clamp: redoes the sums exactly
//   k_v0a           fac_r / fac_c EMAs per 64 vector entries, partial sums of their statistics
//   k_v0b           row / column factor tables; the 12 row-only / column-only feature channels
//                   normalised and folded into 8-float first-layer terms per row / column
//   k_celo2_elem    one launch, items ordered slab by slab (k_celo2.h):
//     statistics    sum of squares of the 18 per-element channels (accumulators advanced in
//                   registers, nothing written); AdamW tensors are fully updated here      24 B/elem
//     fold          per tensor, by its last statistics block: normalisation scales folded into the
//                   first-layer weights
//     apply         accumulators advanced and written, features, MLP, step_out             44 B/elem
//   (PYLO_MI355_SLAB_ELEMS=0: k_celo2_stats, k_stat_segsum, k_celo2_fold, k_celo2_apply as launches
//   of their own, each over all tensors)
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "k_celo2.h"
#include "k_gradstats.h"
#include "k_adafac.h"
#include "k_single.h"
#include "k_velo.h"
#include "k_celo2_slices.h"
#include "k_ns.h"
#include "k_ns_hf.h"
#include "k_ns_small.h"
#include "k_ns_thin.h"
#include "k_slice_finish.h"
#include "k_cast.h"
#include "pylo_common.h"
#include "pylo_mi355_bench.h"

// =============================================================================================
// Host side: plan construction and the C ABI
// =============================================================================================
using namespace pylo;

namespace {

thread_local std::string g_err;

int fail(const std::string& m) {
  g_err = m;
  return 1;
}

#define HIP_TRY(expr)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess) return fail(std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

size_t align_up(size_t x, size_t a = 256) { return (x + a - 1) / a * a; }
long long round4(long long x) { return (x + 3) / 4 * 4; }

// (dc, dr): index of the 2nd-largest and largest dim, ties keep index order
// (pylo/optim/CELO2_naive.py:42-47); VeLO swaps an equal pair except 4-D (0,1)
// (pylo/optim/velo_cuda.py:121-131).
bool factored_dims(int kind, const PyloTensorShape& s, int* dc, int* dr) {
  if (s.ndim < 2) return false;
  std::vector<int> order(s.ndim);
  for (int i = 0; i < s.ndim; ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return s.shape[x] < s.shape[y]; });
  int a = order[s.ndim - 2], b = order[s.ndim - 1];
  if (kind == PYLO_KIND_VELO && s.shape[a] == s.shape[b] && !(s.ndim == 4 && a == 0 && b == 1)) std::swap(a, b);
  *dc = a;
  *dr = b;
  return true;
}

// One group of matrices of the split-fp16 Newton-Schulz kernels: its ranges in the job tables.
struct NsGroup {
  int gram0, n_gram, poly0, n_poly, upd0, n_upd, upd40, n_upd4, split0, n_split, split_max_m;
  int gram_edge, poly_edge, upd_edge;   // output tiles of the three tables: 64 or 128 (upd4: 128 x 256)
  int list0, n_list;       // its matrices (ns_list)
  int sitem0, n_sitems;    // its tiles of the pass that splits the raw steps into planes
  int fitem0, n_fitems;    // its blocks of the pass that sums the squares of A (chain length per matrix)
  int fin0, n_fin;         // its blocks of the finishing pass
  int unit0, n_units;      // ... and their units
};
// One batch of matrices: those whose operand planes share the plane workspace at one time.
struct NsBatch { int mat0, n_mats, group0, n_groups; long long plane_elems; };

constexpr int kNsSmallClasses = 4;
struct Layout {
  std::vector<Item> mx_items;   // ELO-CELO2, VeLO: statistics and apply items in slab order (k_celo2_elem, k_velo_elem)
  bool fused = false;           // ... whatever tensors are in them
  // ... and the streamed tensors: their blocks, the same last to first, the segments of their rows of sums, and the tensors
  std::vector<Item> big_items, big_apply, big_seg;
  std::vector<int> big_list;
  bool split = false;           // element blocks smaller than 8192 elements (split_for)
  size_t off_mx_items = 0, off_big_items = 0, off_big_apply = 0, off_big_seg = 0, off_big_list = 0, off_sync = 0;
  size_t off_newsum = 0, off_piv = 0, off_wmix = 0;   // VeLO: sums carried to the next step, pivots, un-folded MLPs
  // ELO-CELO2: Newton-Schulz on the 2-D tensors (k_ns.h)
  std::vector<NsMat> ns_mats;
  std::vector<NsItem> ns_gram, ns_poly, ns_upd;
  std::vector<NsItem> ns_upd4;        // split-fp16 kernels: update jobs with 256-column tiles
  std::vector<NsGroup> ns_groups;     // split-fp16 kernels: ranges of the job tables, one per group of matrices
  std::vector<NsBatch> ns_batches;    // split-fp16 kernels: batches of matrices that run one after another
  std::vector<int> ns_split;          // matrices whose Gram product is split (k_ns_gram_reduce)
  std::vector<long long> ns_xalt;     // per tensor: offset of its second X buffer, -1 without one
  std::vector<int> ns_of_tensor;      // per tensor: index into ns_mats, -1
  std::vector<int> ns_group_of_tensor;  // split-fp16 kernels, per tensor: its group (index into ns_groups), -1
  std::vector<int> ns_list;           // the groups' matrices, group after group
  int fin_rest0 = 0, n_fin_rest = 0, unit_rest0 = 0, n_unit_rest = 0;   // finishing pass: what belongs to no group
  size_t off_ns_list = 0;
  // ELO-CELO2: tensors with more than two dims, finished per slice of the last two dims (k_slice_finish.h)
  std::vector<SliceMat> slice_mats;
  // blocks of the lane-owned slices (in registers: 1 x 1, 3 x 3, 5 x 5, 7 x 7; in LDS: up to 12, 28, 64 KB a wave),
  // of the wave-owned and of the block-owned ones
  std::vector<Item> slice_items_l[kSliceLaneSets], slice_items_w, slice_items_b;
  std::vector<int> slice_of_tensor;   // per tensor: index into slice_mats, -1
  std::vector<FinUnit> fin_units;     // ELO-CELO2 finishing pass: what each normaliser runs over
  size_t off_fin_units = 0;
  int slice_lds_l[kSliceLaneSets] = {}, slice_lds_w = 0, slice_lds_b = 0;
  size_t off_slice_mats = 0, off_slice_items_l[kSliceLaneSets] = {}, off_slice_items_w = 0, off_slice_items_b = 0;
  int ns_max_m = 0;
  // Newton-Schulz: matrices that one launch takes from the raw step to the parameter (k_ns_thin.h, k_ns_small.h), by class (m up to
  // 16, 32, 64, 128)
  std::vector<NsSmall> sm_mats;
  std::vector<NsSmallItem> sm_items[kNsSmallClasses];
  std::vector<char> small_of_tensor;  // per tensor: its matrices are in sm_mats (2: they are multiples of four elements long)
  long long sm_part_floats = 0;
  int sm_sums = 0, sm_sync = 0, sm_ticket0 = 0;
  bool sm_meets[kNsSmallClasses] = {};   // the class has matrices of several blocks
  size_t off_sm_mats = 0, off_sm_items[kNsSmallClasses] = {}, off_sm_part = 0, off_sm_sums = 0, off_sm_sync = 0;
  std::vector<Item> ns_flag_items;    // split-fp16 kernels: {matrix, chunk of its A} of k_ns_hf_chain_sumsq, group after group
  int ns_fpart_total = 0;
  size_t off_ns_flags = 0, off_ns_fpart = 0, off_ns_flag_items = 0;
  // Newton-Schulz on the fp16 matrix pipe (two-way split operands): tables of their own
  bool ns_hf = false;
  std::vector<NsHfMat> nsb_mats;
  std::vector<NsTileItem> nsb_split_items;
  size_t off_nsb_mats = 0, off_nsb_split_items = 0, off_ns_pw = 0, off_ns_upd4 = 0;
  long long nsb_plane_elems = 0;
  size_t off_ns_mats = 0, off_ns_gram = 0, off_ns_poly = 0, off_ns_upd = 0, off_ns_split = 0, off_ns_xalt = 0,
         off_ns_scale = 0, off_ns_ws = 0;
  // tensors whose grad / param are not fp32 (PYLO_F_STORE_*): fp32 staging, pieces of the cast kernels
  bool typed = false;
  bool in_place = false;   // some tensor of 16-bit storage is read in place (TDesc::direct)
  std::vector<StageOfs> stage_ofs;
  std::vector<Item> cast_items;
  long long stage_floats = 0;
  size_t off_dyn_user = 0, off_stage_ofs = 0, off_cast_items = 0, off_stage = 0;
  std::vector<TDesc> descs;
  std::vector<Item> sl_wave_items;    // ELO-CELO2: blocks of k_celo2_slices_wave, one class after another
  std::vector<Item> sl_wave_cls[kSliceWaveClasses];
  int sl_wave_n[kSliceWaveClasses] = {};
  bool slice_runs = false;            // some tensor's (TDesc::slice_runs)
  size_t off_sl_wave_items = 0;
  std::vector<Item> p0_items, nd_items, sl_items, seg_items, el_items, ap_items, pp_items, ga_items, fin_items, v0a_items, v0b_items;
  std::vector<int> fac_list;
  std::vector<int> dc, dr;
  int H = 8;  // width of the first MLP layer (terms per row / column)
  int Tpad = 0;
  bool lin_matrix = false;   // AdafacLO: ga_items are k_adafac_apply_lin's (else k_adafac_apply's)
  bool global_norm = false;  // AdafacLO kind: every tensor has P0 items, the call may clip by global norm
  bool tensor_norm = false;  // ... or every tensor by its own norm (PYLO_F_TENSOR_NORM)
  size_t off_descs, off_dyn, off_p0_items, off_nd_items, off_sl_items, off_seg_items, off_segtot, off_el_items, off_ap_items, off_pp_items, off_ga_items, off_fin_items, off_finpart, off_finscale, off_tscale, off_v0a_items, off_v0b_items, off_fac_list,
      off_part, off_gsq, off_flag, off_globals, off_fac, off_term, off_v0part, off_bscale, off_stats, off_wfold,
      off_chan_ms, off_totals, off_xfeat, off_lossfeat, off_xT, off_mixbuf, off_pmax, off_canon, off_frac, total;
};

int first_layer_width(int kind) { return kind == PYLO_KIND_CELO2 ? 8 : kind == PYLO_KIND_VELO ? 4 : 32; }

// The hidden layers of ELO-CELO2 run as lane-local 4x4x1 fp32 outer products on the matrix pipe and
// wide 2-D tensors are walked column-resident; PYLO_MI355_VALU_MLP=1 in the environment keeps the
// earlier all-VALU kernels over linear chunks (same results up to rounding; for A/B measurements).
bool env_matrix_pipe() {
  const char* v = std::getenv("PYLO_MI355_VALU_MLP");
  return !(v && v[0] == '1');
}

// AdafacLO's element MLP on the fp16 matrix instructions (two-plane operands); PYLO_MI355_ADAFAC_F32=1 keeps
// the fp32 matrix instructions.
bool env_adafac_hf() {
  const char* v = std::getenv("PYLO_MI355_ADAFAC_F32");
  return !(v && v[0] == '1');
}

// Elements per slab of the fused element pass of ELO-CELO2 (k_celo2_elem).  While the apply items of one
// slab run, the statistics items of the third slab after it do, with the slabs between them resident
// as well: four slabs of 24 bytes per element plus the 20 bytes per element the apply items write
// must fit the 256 MB memory-side cache (measured on the GPT-2-small set: 1.2 M elements 1.51 ms a step,
// 2.4 M 1.48, 3.6 M 1.48, 4.8 M 1.72).  PYLO_MI355_SLAB_ELEMS=0 in the environment (read at plan
// creation) runs each pass over all tensors as a launch of its own instead.
long long env_slab_elems() {
  const char* v = std::getenv("PYLO_MI355_SLAB_ELEMS");
  if (v && v[0]) return std::atoll(v);
  return 2400000;
}
// Slabs of statistics items between a slab's statistics and its apply items (measured: ELO-CELO2 on the
// GPT-2-small set 1.49 / 1.48 ms a step with 2 / 3, VeLO on the ViT-B/16 set 1.06 / 1.00 / 1.04 ms with 1 / 2 / 3).
int env_slab_depth(int kind) {
  const char* v = std::getenv("PYLO_MI355_SLAB_DEPTH");
  return (v && v[0]) ? std::max(1, std::atoi(v)) : (kind == PYLO_KIND_VELO ? 2 : 3);
}
long long env_keep_elems() {   // largest tensor whose inputs are still expected in the cache when its apply items run
  const char* v = std::getenv("PYLO_MI355_KEEP_ELEMS");
  return (v && v[0]) ? std::atoll(v) : 8000000;
}

// How finely the element passes of a plan are cut: a block's 8192 elements (four wave tasks of 16 rows, or a chunk of
// eight trips) are divided by this.  A block of a small plan is a serial chain of memory round trips while most
// CUs have no block at all, so blocks are halved until there is one for each of the 256 CUs or a wave task is down to one
// row.  Measured on a 118 000-parameter classifier, 1 against 16: k_celo2_elem 49 -> 21 us, k_velo_elem 48 -> 26 us,
// AdafacLO's statistics and apply launches 49 -> 24 us together.  From 2.1 M elements on nothing is divided: with
// 512 or 1024 blocks asked for, VeLO on 2.8 M elements went from 137 to 140 and 149 us, AdafacLO from 172 to 173
// and 178 us (every block derives pivots and weights for itself and leaves a row of partial sums to add up).
int split_for(long long elems) {
  int f = 1;
  while (f < kTileRows && elems * f < 256ll * 8192) f *= 2;
  return f;
}
int tile_rows_for(int kind, int split) {
  const char* v = std::getenv("PYLO_MI355_TILE_ROWS");
  if (kind == PYLO_KIND_CELO2 && v && v[0] && std::atoi(v) > 0) return std::atoi(v);
  return kTileRows / split;
}

// Items of k_celo2_elem.  Slabs are runs of whole tensors, last tensors first (their gradients are what
// k_p0 read last).  A tensor too large to stay cached gains nothing from one launch and pays for the hand-over in every block (the
// memory-side round trips of its sums, of the flag and of the weights): its statistics are a launch of the plain kernel in
// front of this one and its apply items one behind it, last item first, since they start on what was read last.  VeLO on one tensor of
// 131 M elements 1704 / 1519 us.
void build_elem_items(Layout& L, int T, int kind) {
  struct Piece { int st0, st1, ap0, ap1; bool keep; };   // statistics items [st0, st1); apply items [ap0, ap1) or none
  const long long cap = env_slab_elems(), keep_max = env_keep_elems();
  if (cap <= 0) return;
  std::vector<Piece> pieces;
  long long elems = 0;
  int el_hi = -1, el_lo = -1;
  auto close = [&]() {
    if (el_hi > el_lo) pieces.push_back(Piece{el_lo, el_hi, el_lo, el_hi, true});
    el_hi = el_lo = -1;
    elems = 0;
  };
  for (int t = T - 1; t >= 0; --t) {
    const TDesc& d = L.descs[t];
    if (d.nblk == 0) continue;
    if (d.n > keep_max) close();   // a run of items has no gaps
    if (d.n > keep_max && d.mode != kModeFlat) {
      L.big_list.push_back(t);
      for (int i = d.blk0; i < d.blk0 + d.nblk; ++i) L.big_items.push_back(L.el_items[i]);
      for (int i = d.seg0; i < d.seg0 + d.nseg; ++i) L.big_seg.push_back(L.seg_items[i]);
      continue;
    }
    if (d.n > keep_max) {   // AdamW: finished by what would be its statistics items, which nobody waits for
      pieces.push_back(Piece{d.blk0, d.blk0 + d.nblk, 0, 0, false});
      continue;
    }
    if (elems > 0 && elems + d.n > cap) close();
    if (el_hi < 0) el_hi = d.blk0 + d.nblk;
    el_lo = d.blk0;   // tensors are visited in descending order: the run grows downwards
    elems += d.n;
  }
  close();
  L.fused = true;
  L.big_apply.assign(L.big_items.rbegin(), L.big_items.rend());
  const int np = (int)pieces.size(), depth = env_slab_depth(kind);
  auto push = [&](int i0, int i1, bool apply, bool keep) {
    for (int i = i0; i < i1; ++i) {
      Item it = L.el_items[i];
      if (apply && L.descs[it.tensor].mode == kModeFlat) continue;   // AdamW tensors are finished by their statistics items
      it.b = i;
      it.c = apply ? kElemApply : (keep ? kElemKeep : 0);
      L.mx_items.push_back(it);
    }
  };
  for (int k = 0; k < np + depth; ++k) {
    if (k < np) push(pieces[k].st0, pieces[k].st1, false, pieces[k].keep);
    if (k >= depth) push(pieces[k - depth].ap0, pieces[k - depth].ap1, true, pieces[k - depth].keep);
  }
}

// PYLO_MI355_NS_F32=1 keeps the Newton-Schulz products on the fp32 matrix instructions (k_ns.h) instead of
// the split-fp16 ones (k_ns_hf.h); read at plan creation.
bool env_ns_xcd() {
  const char* e = getenv("PYLO_MI355_NS_XCD");
  return !(e && e[0] == '0');
}

// PYLO_MI355_NS_GROUPS: into how many groups (streams) the matrices of a plan are dealt, 1 to 4; read at plan creation.  Three
// unless it says otherwise.  A process has four hardware queues here; the runtime gives a new stream one of those that have the
// fewest streams, and two groups that share one wait for each other.  Streams made in threes land on three queues
// whatever streams the program has (which is why a plan of two groups makes three as well), and no group rides on the
// caller's stream, whose queue a group of another plan may share.  Whole ELO-CELO2 step on the GPT-2-small set, the
// first, second and third plan of a process: three groups 6.02, 6.04, 6.00 ms, four 6.61, 6.00, 6.00, two on two
// streams 6.09, 6.79, 6.06; with one of three on the caller's stream 6.04 to 6.30.
int env_ns_groups() {
  const char* e = getenv("PYLO_MI355_NS_GROUPS");
  const int g = e ? atoi(e) : 3;
  return std::max(1, std::min(g, 4));
}

// PYLO_MI355_NS_WORKSPACE_MB: what the operand planes of the matrices that are orthogonalised at one time may take
// (in fp16 elements here); read at plan creation.
long long env_ns_budget_elems() {
  const char* e = getenv("PYLO_MI355_NS_WORKSPACE_MB");
  const long long mb = e ? atoll(e) : 8192;
  return std::max(1ll, mb) * (1ll << 20) / 2;
}

// How the Newton-Schulz iterations share their products over the long dim (k_ns_hf.h): a chain of L iterations takes
// one Gram product, one update and 4 L - 3 products of m x m matrices.  PYLO_MI355_NS_CHAINS="2,3" gives the chain
// lengths in order (they must add up to the iteration count, else the default applies); PYLO_MI355_NS_PAIRS=0 means
// chains of one: one Gram product and one update per iteration, as the formula is written.  Read when the products
// are enqueued.
std::vector<int> ns_chains(int iters) {
  std::vector<int> out;
  const char* p = getenv("PYLO_MI355_NS_PAIRS");
  if (p && p[0] == '0') {
    out.assign(iters, 1);
    return out;
  }
  if (const char* e = getenv("PYLO_MI355_NS_CHAINS")) {
    int sum = 0;
    for (const char* c = e; *c;) {
      const int v = atoi(c);
      if (v < 1) break;
      out.push_back(v);
      sum += v;
      while (*c && *c != ',') ++c;
      if (*c == ',') ++c;
    }
    if (sum == iters) return out;
    out.clear();
  }
  // default: pairs (five iterations: 2, 2, 1).  Longer chains are faster and less accurate: "3,2" takes the
  // GPT-2-small step from 6.4 to 5.7 ms and stays at the formula's own fp32 error on most inputs, but reaches 1e-4
  // of the result's RMS (against 1.3e-5 for pairs) on matrices with a dominant direction over a flat rest.
  for (int left = iters; left > 0;) {
    const int l = std::min(left, 2);
    out.push_back(l);
    left -= l;
  }
  return out;
}

// PYLO_MI355_NS_ADAPTIVE=1: a first chain of three iterations for the matrices whose spectrum allows it
// (k_ns_hf_chain_flag), pairs for the others -- unless the environment fixes the chains (PYLO_MI355_NS_CHAINS,
// PYLO_MI355_NS_PAIRS=0).  Off by default: raw steps with a direction that holds more than 8 % of their squared norm
// never qualify (an untrained MLP's steps, with their common offset, are such), and the test costs 0.04 ms a step.
// Read when the products are enqueued.
bool ns_adaptive() {
  const char* a = getenv("PYLO_MI355_NS_ADAPTIVE");
  if (!(a && a[0] == '1')) return false;
  const char* p = getenv("PYLO_MI355_NS_PAIRS");
  if (p && p[0] == '0') return false;
  const char* c = getenv("PYLO_MI355_NS_CHAINS");
  return !(c && c[0]);
}

// The planes of the Newton-Schulz products are fp16 numbers: every matrix is stored times a power of two that puts its
// largest possible entry at 12 000 .. 24 000 (the format ends at 65 504), so that the second plane keeps its bits on
// entries five decades smaller.  No entry exceeds the matrix's largest singular value, and those follow from the
// coefficients alone: X0 has unit Frobenius norm, so its singular values lie in [0, 1], and every iteration maps
// sigma to sigma p(sigma^2), p(l) = c2 l^2 + c1 l + c0.  Bounds over all iterations, from a grid of starting values:
// X (sigma), A = X X^T (sigma^2), B' = p(A), T = A B', and the products of k consecutive B' (q[k], k >= 1).
struct NsExps {
  int x, a, b, t;
  std::vector<int> q;
};
inline float pow2(int e) { return std::ldexp(1.0f, e); }
NsExps ns_plane_exps(float c0, float c1, float c2, int iters) {
  constexpr int kGrid = 2048;
  const int n = std::max(iters, 1);
  double bx = 1.0, ba = 1.0, bb = std::fabs((double)c0), bt = 0.0;
  std::vector<double> bq(n + 1, 0.0), pv(n);
  for (int g = 0; g <= kGrid; ++g) {
    double sig = (double)g / kGrid;
    for (int t = 0; t < n; ++t) {
      const double l = sig * sig, pl = (double)c2 * l * l + (double)c1 * l + (double)c0;
      pv[t] = std::fabs(pl);
      ba = std::max(ba, l);
      bb = std::max(bb, pv[t]);
      bt = std::max(bt, l * pv[t]);
      sig *= pl;
      bx = std::max(bx, std::fabs(sig));
    }
    for (int t0 = 0; t0 < n; ++t0) {
      double prod = 1.0;
      for (int k = 1; t0 + k <= n; ++k) {
        prod *= pv[t0 + k - 1];
        bq[k] = std::max(bq[k], prod);
      }
    }
  }
  auto exp_of = [](double bound) {
    if (!(bound > 0.0) || !std::isfinite(bound)) return -60;   // (coefficients that diverge: nothing to keep)
    const int e = (int)std::floor(std::log2(30000.0 / (1.25 * bound)));
    return std::max(-60, std::min(e, 14));
  };
  NsExps ex;
  ex.x = exp_of(bx); ex.a = exp_of(ba); ex.b = exp_of(bb); ex.t = exp_of(bt);
  ex.q.resize(n + 1);
  for (int k = 1; k <= n; ++k) ex.q[k] = exp_of(bq[k]);
  ex.q[0] = ex.b;
  return ex;
}

// PYLO_MI355_SLICES_LDS=0: the short slices of ELO-CELO2 tensors with more than two dims stay on the kernel that walks
// them twice (k_celo2_slices); read at plan creation.
bool env_slices_lds() {
  const char* e = getenv("PYLO_MI355_SLICES_LDS");
  return !(e && e[0] == '0');
}

bool env_ns_hf() {
  const char* e = getenv("PYLO_MI355_NS_F32");
  return !(e && e[0] == '1');
}

// Workgroups go to the eight XCDs in turn (block b runs on XCD b % 8) and every XCD has an L2 of its own:
// tile jobs that read the same operands should share an XCD.  `units` are runs of jobs that belong together
// (count, work per job); the run sequence is cut into eight stretches of about equal work, stretch x becomes
// the jobs 8 i + x.  Stretches are filled up with jobs that do nothing (mat = -1).
constexpr int kXcds = 8;
void xcd_interleave(std::vector<NsItem>& items, const std::vector<std::pair<int, long long>>& units) {
  long long total = 0;
  for (const auto& u : units) total += u.first * u.second;
  std::vector<std::vector<NsItem>> lane(kXcds);
  long long done = 0;
  size_t pos = 0;
  int x = 0;
  for (const auto& u : units) {
    // a unit goes to the stretch in which its middle falls
    const long long mid = done + u.first * u.second / 2;
    x = std::max(x, (int)std::min<long long>(kXcds - 1, total > 0 ? mid * kXcds / total : 0));
    for (int i = 0; i < u.first; ++i) lane[x].push_back(items[pos + i]);
    pos += u.first;
    done += u.first * u.second;
  }
  size_t longest = 0;
  for (const auto& l : lane) longest = std::max(longest, l.size());
  std::vector<NsItem> out;
  out.reserve(longest * kXcds);
  for (size_t i = 0; i < longest; ++i)
    for (int q = 0; q < kXcds; ++q) out.push_back(i < lane[q].size() ? lane[q][i] : NsItem{-1, 0, 0, 0, 0, -1});
  items.swap(out);
}

// PYLO_MI355_NS_SMALL=0: small matrices go through the tiled products like all others; read at plan creation.
bool env_ns_small() {
  const char* e = getenv("PYLO_MI355_NS_SMALL");
  return !(e && e[0] == '0');
}

// The products of an m x n matrix in the unit of the rules below: five iterations in pairs are three Gram products on
// the upper blocks, three updates and eleven m x m products.
double ns_work(int m, int n) { return (double)m * m * (4.6 * n + 5.9 * m); }
// ... as the tiled launches do it, in whole tiles (a thousand 130 x 130, 176 G and not 23: 2000 us on two streams, 2177 on one)
double ns_tiled_work(int m, int n) {
  auto up = [](int x) { return (x + kNsTile - 1) / kNsTile * kNsTile; };
  return ns_work(up(m), up(n));
}

// Into how many groups (streams) the matrices of a plan are dealt: as many as have eight of its matrices each, those that
// go aside to k_ns_small counted (which launch takes them says nothing about the others), and 55 G of work each.  Below that a
// group's launches are bound by their number, and more streams only add to it.  Whole steps, 1 / 2 / 3 groups (with two
// embeddings of 4000 rows):
//   width 256, 4, 12 layers (9, 21 G) 408 / 480 / 492 us, 668 / 691 / 718      384, 8 (47 G) 1101 / 1108 / 1151, 12 (68 G)
//   1404 / 1391 / 1456      512, 4 (60 G) 1086 / 1136 / 1229, 6 (84 G) 1435 / 1425 / 1439, 8 (109 G) 1774 / 1721 / 1778, 12 (157 G)
//   2514 / 2438 / 2403      768, 2 (110 G) 1586 / 1583 / 1669, 4 (192 G) 2481 / 2341 / 2307      1024, 2 (247 G, fourteen matrices)
//   2648 / 2471 / 2489, 3 (344 G) 3397 / 3325 / 3336, 8 (830 G) 7773 / 7436 / 7425
//   64 of 256 x 256 (11 G) 383 / 385 / 459, 40 of 512 x 512 (56 G) 883 / 918 / 951, 500 of 200 x 200 (88 G) 1664 / 1541 / 1544
int ns_group_count(int mats, double work) {
  return (int)std::min<double>(std::min(env_ns_groups(), std::max(mats / 8, 1)), 1.0 + std::floor(work / 55e9));
}

using SmMid = SmDims<2, 1, 2>;
using SmLarge = SmDims<4, 2, 1>;
// 0, 1: k_ns_thin<1>, <2>; 2, 3: k_ns_small<2, 1, 2>, <4, 2, 1>
int ns_small_class(int m) { return m <= ThinDims<1>::MP ? 0 : m <= ThinDims<2>::MP ? 1 : m <= SmMid::MP ? 2 : 3; }
int ns_small_chunk(int cls) { return cls < 2 ? kThinChunk : cls == 2 ? SmMid::NB : SmLarge::NB; }
// floats of partial sums that a block of a matrix of several leaves: G in fp64, or A in fp32 twice
int ns_small_part(int cls) { return cls == 0 ? ThinDims<1>::NT * 512 : cls == 1 ? ThinDims<2>::NT * 512 : 2 * (cls == 2 ? SmMid::MP * SmMid::MP : SmLarge::MP * SmLarge::MP); }

// Which matrices the one-launch kernel takes: a smaller dim of at most 128 (its m x m matrices fit a CU's LDS) and a
// longer one up to where its few blocks, each walking chunks of the long dim one after another, fall behind tiles of 64 x 64
// on all CUs.  Where that is depends on how many a plan has: few long ones leave CUs idle that tiles would use, sixteen and
// more fill them either way and need half the launches here.  The line for few: 24576 for m of 49 to 64, for m > 64 1024 at
// m = 128, 2147 at 100, 5753 at 72, and n / 30 times that in a plan of n > 30 matrices with m > 64, whose launch the long ones
// end under; `many[c]`: the plan has four of the former (c = 0) or sixteen of the latter (c = 1) beyond it.
// Whole steps on matrices of m x n, here / by tiles, us:
//   m = 128, 1, 8, 16, 32, 64 of them: n = 1100 197 / 180, 224 / 215, 249 / 250, 272 / 304, 479 / 447      4096 282 / 199,
//     344 / 292, 469 / 447, 535 / 623, 899 / 1089      8192 440 / 253, 610 / 475, 781 / 716, 916 / 1075, 1719 / 2032
//   m = 96: 2048 175 / 169, 213 / 220, 244 / 271, 296 / 374, 466 / 579      8192 374 / 252, 467 / 409, 680 / 664, 814 / 964,
//     1490 / 1834
//   m = 72: 3000 177 / 181, 212 / 240, 246 / 285, 305 / 412, 504 / 668      6000 257 / 211, 299 / 288, 387 / 436, 516 / 645,
//     1092 / 1157
//   m = 64, 1, 4, 16, 64 of them: 16384 213 / 232, 258 / 314, 737 / 786, 1974 / 2457      32768 317 / 284, 446 / 497, 1219 / 1453,
//     4028 / 4528
//   m = 48: 24000 229 / 248, 286 / 342, 823 / 874, 2573 / 2806      32768 267 / 271, 358 / 418, 1043 / 1299, 3110 / 3748
//   m = 32 (k_ns_thin, no line below its limits: from one matrix to 256 of any length it is the faster): 1024 101 / 172, 104 / 182,
//     110 / 192, 145 / 262      16384 110 / 222, 154 / 279, 335 / 515, 850 / 1499      32768 141 / 255, 206 / 327, 549 / 965, 1622 / 2659
//   m = 16, 1, 16 of them: 8192 100 / 205, 146 / 289      32768 104 / 235, 354 / 745      65536 131 / 257, 571 / 1200
//   m = 4: 65536 101 / 237, 271 / 963
//   decoders of width 128 with two embeddings: 12 layers (74 matrices) 2000 239 / 266, 4000 324 / 291; 24 (146) 2000 287 / 345,
//     4000 374 / 402, 8000 549 / 472; 40 (242) 4000 424 / 559, 8000 571 / 688
struct NsSmallRule {
  double stretch = 1.0;
  bool many[2] = {true, true};
};
bool ns_small_long(int m, int n, const NsSmallRule& r) {
  return m > SmMid::MP ? (double)m * m * m * n > r.stretch * (1ll << 31) : m > 48 && n > 24576;
}
bool ns_small_takes(int R, int C, const NsSmallRule& r) {
  const int m = std::min(R, C), n = std::max(R, C);
  if (m > SmLarge::MP || n > (m <= 16 ? 65536 : m <= SmMid::MP ? 32768 : 8192)) return false;
  return !ns_small_long(m, n, r) || r.many[m > SmMid::MP];
}

// Whether a plan's small matrices go aside to their own launches, or with the larger ones through the tiled launches that
// run anyway.  Aside they cost a fork and a join (10 us and more of a chain on one stream) and, in the largest class, a CU
// a block; in the tiled launches they are a few more tiles, free while the launches leave CUs idle.  So they stay with larger
// matrices that are one group, if these are less than 22 G of work (or the small one is alone) and the small ones add
// no more than 512 update tiles, two a CU.  Whole steps, tiled / aside:
//   classifier 784 -> 1024 -> 1024 -> 10 (19 G) 442 / 468 us, 784 -> 384 -> 384 -> 10 250 / 269, 784 -> 2048 (x 4) -> 10
//     (373 G, one small) 3103 / 3135
//   one 512 x 512 (1.4 G) and 8, 32, 64 of 16 x 1024 262 / 283, 346 / 353, 389 / 413
//   decoder of width 256 with k, v of 32, 1, 4, 12 layers (4, 7, 17 G) 293 / 317, 379 / 412, 642 / 610; width 384, 48, 1 layer 404 / 430
//   four 1024 x 1024 (45 G) and 8, 16, 64 of 16 x 1024 715 / 753, 756 / 791, 937 / 888
//   two 1024 x 1024 (23 G) and 4, 16 of 64 x 2000 467 / 478, 613 / 548
//   decoder of width 512 with k, v of 64, 2 layers (30 G) 727 / 723, 8 (86 G, two groups) 1496 / 1480
//   decoder of width 1024 with k, v of 128, 1, 2 layers (127, 202 G) 1648 / 1634, 2230 / 2205
bool ns_small_aside(int n_large, double work_large, int n_small, long long small_tiles) {
  if (n_large == 0 || small_tiles > 512 || ns_group_count(n_large + n_small, work_large) > 1) return true;
  return n_small > 1 && work_large >= 22e9;
}

// Slabs (blocks) of each small matrix and the items of the launches.
void build_small_items(Layout& L) {
  // how many blocks a launch of the class is cut into at most -- what 256 CUs hold at a time (LDS), for the thin ones fewer: every
  // block of a matrix goes through its m x m products (sixteen of 17 x 32768, blocks up to 256 / 512 / 1024: 164 / 128 / 161 us,
  // three hundred of 32 x 1024 124 / 98 / 121) -- and the most blocks one matrix may have waiting (k_ns_small.h)
  constexpr int kHolds[kNsSmallClasses] = {1024, 512, 512, 256}, kSlabsMax[kNsSmallClasses] = {64, 64, 32, 8};
  constexpr int kChunksMin[kNsSmallClasses] = {8, 4, 1, 1};   // what a block takes before a matrix is cut
  auto cls_of = [](const NsSmall& b) { return ns_small_class(b.m); };
  int lift[kNsSmallClasses] = {0, 1, 2, 3};
  // A plan with few small matrices takes them in the class of the largest, one launch: the small ones end under it,
  // unless the fewer and larger blocks of that class walk more than eight chunks each, what its own longest matrix walks
  // (a chunk is 15 to 25 us of a block's chain).  Whole steps, a class of 65 x 65 or 100 x 100 next to others, lifted /
  // in their own classes: 784 -> 128 -> 128 -> 10 148 / 177 us, 784 -> 64 (x 4) -> 10 112 / 121, twenty of 64 x 8192 (eight
  // chunks) 548 / 613; 16 x 65536 (64 chunks) 1028 / 397, 64 x 32768 (32) 1092 / 405, 63 of 16 x 65536 (126) 4319 / 3000.
  if ((int)L.sm_mats.size() <= 64) {
    int top = 0;
    for (const NsSmall& b : L.sm_mats) top = std::max(top, cls_of(b));
    const int nb = ns_small_chunk(top);
    for (int c = top - 1; c >= 0; --c) {
      long long total = 0, most = 0;
      for (const NsSmall& b : L.sm_mats) {
        if (lift[cls_of(b)] != top && cls_of(b) != c) continue;
        total += (b.n + nb - 1) / nb;
        if (cls_of(b) == c) most = std::max<long long>(most, (b.n + nb - 1) / nb);
      }
      if (std::max(total / kHolds[top], (most + kSlabsMax[top] - 1) / kSlabsMax[top]) <= 8) lift[c] = top;
    }
  }
  for (int cls = 0; cls < kNsSmallClasses; ++cls) {
    std::vector<int> of;
    const int nb = ns_small_chunk(cls);
    if (cls == 0)
      for (int q = 0; q < (int)L.sm_mats.size(); ++q)
        if (lift[cls_of(L.sm_mats[q])] == 0)
          for (NsSmall& b = L.sm_mats[q]; (2 << b.fold) * b.m <= ThinDims<1>::MP;) ++b.fold;
    auto chunks = [&](int q) { return (L.sm_mats[q].n + (nb << L.sm_mats[q].fold) - 1) / (nb << L.sm_mats[q].fold); };
    long long total = 0;
    for (int q = 0; q < (int)L.sm_mats.size(); ++q)
      if (lift[cls_of(L.sm_mats[q])] == cls) {
        of.push_back(q);
        total += chunks(q);
      }
    // one slab a chunk while no more blocks are started than twice what runs at once, longer ones when there are more
    const int per = (int)std::max<long long>(kChunksMin[cls], total / kHolds[cls]);
    for (int q : of) {
      NsSmall& b = L.sm_mats[q];
      const int c = chunks(q);
      b.chunks = std::max(per, (c + kSlabsMax[cls] - 1) / kSlabsMax[cls]);
      b.slabs = (c + b.chunks - 1) / b.chunks;
      if (b.slabs == 1) { b.chunks = c; continue; }
      b.chunks = (c + b.slabs - 1) / b.slabs;      // even slabs
      b.slabs = (c + b.chunks - 1) / b.chunks;
      b.part = L.sm_part_floats;
      L.sm_part_floats += (long long)b.slabs * ns_small_part(cls);
      b.sums = L.sm_sums;
      L.sm_sums += 2 * b.slabs;
      b.sync = L.sm_sync;
      L.sm_sync += 2;
      L.sm_meets[cls] = true;
    }
    // the blocks that meet first (they start together), then the longest
    std::stable_sort(of.begin(), of.end(), [&](int x, int y) {
      const NsSmall &a = L.sm_mats[x], &b = L.sm_mats[y];
      if ((a.slabs > 1) != (b.slabs > 1)) return a.slabs > 1;
      return a.chunks > b.chunks;
    });
    for (int q : of)
      for (int sl = 0; sl < L.sm_mats[q].slabs; ++sl) L.sm_items[cls].push_back(NsSmallItem{q, sl});
  }
  L.sm_ticket0 = L.sm_sync;
  L.sm_sync += kNsSmallClasses;
}

// The output tiles of a launch with `jobs` tiles of 128 x 128: those, or 64 x 64 where they are fewer than the CUs.  A tile job
// is a chain of stages that wait for memory; few long ones leave most of the part idle and each of them half of its CU.
// The m x m products' bare loop, 128 x 128 / 64 x 64 tiles (four steps a stage): one 1024 x 1024 with 63 steps (36 / 136 jobs)
// 28.0 / 12.2 us, four 512 x 512 (40 / 144) 12.9 / 6.3, six 384 x 384 (36 / 126) 10.2 / 5.2, twelve 768 x 768 (252 / 936)
// 24.9 / 24.6, forty-eight (1008 / 3744) 76.9 / 92.0.  Finishing calls before (all 128 x 128 and 128 x 256) / now: one
// 1000 x 2048 738 / 319 us, a layer of width 256 366 / 154, four of width 512 916 / 644, twenty 200 x 200 312 / 141, 4000 x 512
// 495 / 214; whole CELO2 step on ResNet-50 1.49 / 1.21 ms.
int ns_tile_edge(long long jobs) { return jobs < 256 ? 64 : kNsTile; }

// Newton-Schulz tables: every 2-D MLP tensor (the fp32 kernels: those whose rows (C) and whose smaller dim are
// multiples of 4).  `ws_floats` returns the floats of workspace behind off_ns_ws.
void build_ns_tables(Layout& L, const PyloTensorShape* shapes, int T, long long& ws_floats) {
  ws_floats = 0;
  L.ns_xalt.assign(T, -1);
  L.ns_of_tensor.assign(T, -1);
  L.ns_group_of_tensor.assign(T, -1);
  L.small_of_tensor.assign(T, 0);
  auto take = [&](long long n) { const long long o = ws_floats; ws_floats += (n + 63) / 64 * 64; return o; };
  // The matrices of a tensor: R x C, n_sl of them; none if the products do not take it.
  auto matrices = [&](int t, int& R, int& C, int& n_sl) {
    const TDesc& d = L.descs[t];
    if (d.n == 0 || (shapes[t].flags & PYLO_F_NO_ORTHOGONALIZE)) return false;
    // two dims; or more, as one matrix per slice of the last two, where the per-slice launches do not take the
    // slices (k_slice_finish.h) -- the split-fp16 kernels only, whose tables carry a matrix's place in its tensor
    const bool slices = d.mode == kModeFacND && L.ns_hf && L.slice_of_tensor[t] < 0;
    if (d.mode != kModeFac2D && !slices) return false;
    R = slices ? (int)shapes[t].shape[shapes[t].ndim - 2] : d.R0;
    C = slices ? (int)shapes[t].shape[shapes[t].ndim - 1] : d.C0;
    // the fp32 kernels load 16 bytes at a time along the contiguous dim of X, A and B'
    if (!L.ns_hf && (C % 4 != 0 || std::min(R, C) % 4 != 0)) return false;
    n_sl = slices ? (int)(d.n / ((long long)R * C)) : 1;
    return true;
  };
  int R = 0, C = 0, n_sl = 0;
  // Chains of other lengths than pairs and singles, where the environment asks for them, are the tiled products' only.
  const char* chains = getenv("PYLO_MI355_NS_CHAINS");
  NsSmallRule rule;
  bool small = L.ns_hf && env_ns_small() && !(chains && chains[0]) && !ns_adaptive();
  if (small) {
    int n_large = 0, n_small = 0, n_cls = 0, n_long[2] = {0, 0};
    double work = 0.0;
    long long tiles = 0;
    for (int t = 0; t < T; ++t)
      if (matrices(t, R, C, n_sl) && std::min(R, C) > SmMid::MP && ns_small_takes(R, C, rule)) n_cls += n_sl;
    rule.stretch = std::max(1.0, n_cls / 30.0);
    for (int t = 0; t < T; ++t)
      if (matrices(t, R, C, n_sl) && ns_small_takes(R, C, rule) && ns_small_long(std::min(R, C), std::max(R, C), rule))
        n_long[std::min(R, C) > SmMid::MP] += n_sl;
    rule.many[0] = n_long[0] >= 4;
    rule.many[1] = n_long[1] >= 16;
    for (int t = 0; t < T; ++t) {
      if (!matrices(t, R, C, n_sl)) continue;
      if (ns_small_takes(R, C, rule)) {
        n_small += n_sl;
        tiles += (long long)n_sl * ((std::max(R, C) + kNsTile - 1) / kNsTile);
      } else {
        n_large += n_sl;
        work += n_sl * ns_tiled_work(std::min(R, C), std::max(R, C));
      }
    }
    small = ns_small_aside(n_large, work, n_small, tiles);
  }
  for (int t = 0; t < T; ++t) {
    if (!matrices(t, R, C, n_sl)) continue;
    if (small && ns_small_takes(R, C, rule)) {
      L.small_of_tensor[t] = (long long)R * C % 4 == 0 ? 2 : 1;
      for (int sl = 0; sl < n_sl; ++sl) {
        NsSmall b{};
        b.tensor = t;
        b.m = std::min(R, C);
        b.n = std::max(R, C);
        b.tall = R > C;
        b.elem_off = (long long)sl * R * C;
        L.sm_mats.push_back(b);
      }
      continue;
    }
    for (int sl = 0; sl < n_sl; ++sl) {
    NsMat mt{};
    mt.tensor = t;
    mt.unit = sl;        // the finishing pass's tables come later: build_fin_tables adds the tensor's first unit
    mt.elem_off = (long long)sl * R * C;
    mt.R = R; mt.C = C;
    mt.tall = R > C;
    mt.m = std::min(R, C);
    const int K = mt.tall ? mt.R : mt.C;
    mt.n_slabs = K >= kNsSplitMin ? (K + kNsSlabK - 1) / kNsSlabK : 1;
    mt.slab_k = kNsSlabK;
    mt.off_x1 = take((long long)R * C);
    mt.off_a = take((long long)mt.m * mt.m);
    mt.off_b = take((long long)mt.m * mt.m);
    mt.off_part = mt.n_slabs > 1 ? take((long long)mt.n_slabs * mt.m * mt.m) : 0;
    const int q = (int)L.ns_mats.size();
    if (sl == 0) {
      L.ns_of_tensor[t] = q;
      L.ns_xalt[t] = mt.off_x1;
    }
    L.ns_max_m = std::max(L.ns_max_m, mt.m);
    const int nt = (mt.m + kNsTile - 1) / kNsTile;
    for (int tm = 0; tm < nt; ++tm)
      for (int tn = tm; tn < nt; ++tn) {
        if (mt.n_slabs > 1) {
          for (int sb = 0; sb < mt.n_slabs; ++sb)
            L.ns_gram.push_back(NsItem{q, tm, tn, sb * kNsSlabK, std::min(K, (sb + 1) * kNsSlabK), sb});
        } else {
          L.ns_gram.push_back(NsItem{q, tm, tn, 0, K, -1});
        }
        L.ns_poly.push_back(NsItem{q, tm, tn, 0, mt.m, -1});
      }
    const int ni = ((mt.tall ? mt.R : mt.m) + kNsTile - 1) / kNsTile, nj = ((mt.tall ? mt.m : mt.C) + kNsTile - 1) / kNsTile;
    for (int tm = 0; tm < ni; ++tm)
      for (int tn = 0; tn < nj; ++tn) L.ns_upd.push_back(NsItem{q, tm, tn, 0, mt.m, -1});
    if (mt.n_slabs > 1) L.ns_split.push_back(q);
    L.ns_mats.push_back(mt);
    }
  }
  build_small_items(L);
  if (L.ns_hf) {
    // A plan with few matrices (a convolutional net's one classifier, a small MLP) has fewer Gram tile jobs than the
    // part has CUs, each a long reduction: split them along it, up to eight ways, until there are two jobs a CU.
    {
      long long jobs = 0;
      for (const int edge : {kNsTile, 64}) {
        jobs = 0;
        for (const NsMat& f : L.ns_mats) {
          const long long nt = (f.m + edge - 1) / edge;
          jobs += nt * (nt + 1) / 2 * f.n_slabs;
        }
        if (ns_tile_edge(jobs) == kNsTile) break;
      }
      if (jobs > 0 && jobs < kNsFewJobs) {
        const int ways = (int)std::min<long long>(8, (kNsFewJobs + jobs - 1) / jobs);
        for (NsMat& f : L.ns_mats) {
          if (f.n_slabs > 1) continue;
          const int K = f.tall ? f.R : f.C;
          const int sk = std::max(256, ((K + ways - 1) / ways + 15) / 16 * 16);
          if ((K + sk - 1) / sk > 1) {
            f.slab_k = sk;
            f.n_slabs = (K + sk - 1) / sk;
          }
        }
      }
    }
    // same matrices, operands as fp16 planes; the item tables are rebuilt for the uniform (n x m) orientation
    L.ns_gram.clear(); L.ns_poly.clear(); L.ns_upd.clear(); L.ns_upd4.clear();
    ws_floats = 0;
    long long pw = 0;
    auto take_p = [&](long long n) { const long long o = pw; pw += (n + 63) / 64 * 64; return o; };
    auto up = [](int x, int q) { return (x + q - 1) / q * q; };
    auto up16 = [&](int x) { return up(x, kHfBK); };
    // Planes and fp32 matrices of every matrix.  The planes are only live during a matrix's own products, so
    // the matrices are cut into batches (in tensor order) whose planes fit PYLO_MI355_NS_WORKSPACE_MB (8192 by
    // default); the batches run one after another in the same memory.  A plan whose matrices fit in one batch
    // has its planes' padding zeroed once, at plan creation; with several batches every batch starts by zeroing
    // the region (one fill at HBM write speed: the padding of one batch's planes lies in another's data).
    const long long budget = env_ns_budget_elems();
    long long pw_max = 0, ws_max = 0;
    std::vector<int> batch_of;
    L.ns_batches.clear();
    NsBatch batch{};
    auto mats_of_tensor = [&](size_t q) {
      size_t e = q;
      while (e < L.ns_mats.size() && L.ns_mats[e].tensor == L.ns_mats[q].tensor) ++e;
      return (long long)(e - q);
    };
    for (size_t q = 0; q < L.ns_mats.size(); ++q) {
      const NsMat& f = L.ns_mats[q];
      NsHfMat b{};
      b.tensor = f.tensor; b.R = f.R; b.C = f.C; b.m = f.m; b.n = std::max(f.R, f.C); b.tall = f.tall;
      b.pad_m = up16(b.m);
      b.pad_n = up16(b.n);
      // update tiles of 256 columns where that does not compute much more padding than tiles of 128 would
      const bool wide_tiles = up(b.m, 256) <= 1.06 * up(b.m, 128);
      b.rows_m = up(b.m, wide_tiles ? 256 : kNsTile);
      b.rows_n = up(b.n, kNsTile);
      b.a_floats = (long long)hf_tiles_upper(b.m) * kNsTileFloats;
      b.n_slabs = f.n_slabs;
      b.p_stride = ((long long)kNsPl * b.rows_m * b.pad_m + 63) / 64 * 64;
      // (the matrices of one tensor -- the slices of one with more than two dims -- stay in one batch)
      const bool first_of_tensor = q == 0 || L.ns_mats[q - 1].tensor != f.tensor;
      const long long need = ((long long)kNsPl * b.rows_m * b.pad_n + 2ll * kNsPl * b.rows_n * b.pad_m + kNsBufs * b.p_stride + 4 * 64) *
                             (first_of_tensor ? mats_of_tensor(q) : 1);
      if (pw > 0 && first_of_tensor && pw + need > budget) {   // this tensor opens the next batch
        batch.plane_elems = pw;
        L.ns_batches.push_back(batch);
        batch = NsBatch{};
        batch.mat0 = (int)q;
        pw = 0;
        ws_floats = 0;
      }
      b.off_xs = take_p((long long)kNsPl * b.rows_m * b.pad_n);
      b.off_xl[0] = take_p((long long)kNsPl * b.rows_n * b.pad_m);
      b.off_xl[1] = take_p((long long)kNsPl * b.rows_n * b.pad_m);
      b.off_p = take_p(kNsBufs * b.p_stride);
      b.off_a = take(b.a_floats);
      b.off_part = b.n_slabs > 1 ? take((long long)b.n_slabs * b.a_floats) : 0;
      b.elem_off = f.elem_off;
      L.ns_mats[q].off_a = b.off_a;   // the fp32 tables stay consistent for k_ns_scale (tensor index only)
      L.nsb_mats.push_back(b);
      batch_of.push_back((int)L.ns_batches.size());
      batch.n_mats = (int)q + 1 - batch.mat0;
      pw_max = std::max(pw_max, pw);
      ws_max = std::max(ws_max, ws_floats);
    }
    if (batch.n_mats > 0) {
      batch.plane_elems = pw;
      L.ns_batches.push_back(batch);
    }
    pw = pw_max;
    ws_floats = ws_max;
    L.nsb_plane_elems = pw;
    std::fill(L.ns_xalt.begin(), L.ns_xalt.end(), -1);   // the result always replaces the raw step
    // Groups of matrices.  The products of one matrix depend on each other, those of different matrices do not:
    // each group runs its chain of launches on a stream of its own, so that the blocks of one group's launch
    // fill the CUs that the tail of the other's leaves idle.  Matrices are dealt to the groups heaviest first.
    L.ns_groups.clear();
    L.ns_split.clear();
    L.ns_list.clear();
    L.nsb_split_items.clear();
    L.ns_flag_items.clear();
    L.ns_fpart_total = 0;
    for (NsBatch& bt : L.ns_batches) {
    double batch_work = 0.0;
    for (int q = bt.mat0; q < bt.mat0 + bt.n_mats; ++q) batch_work += ns_tiled_work(L.nsb_mats[q].m, L.nsb_mats[q].n);
    // (one of the four hardware queues is left to the small matrices where there are any: 3 / 4 groups next to them, 1024
    // wide 8117 / 8162 us, 512 wide 3203 / 3281)
    const int n_groups = std::min({L.sm_mats.empty() ? 4 : 3, bt.n_mats,
                                   ns_group_count(bt.n_mats + (int)L.sm_mats.size(), batch_work)});
    std::vector<std::vector<int>> members(n_groups);
    {
      // (tensor by tensor: the slices of a tensor with more than two dims share a group, which also finishes it)
      struct Run { int q0, q1; double work; };
      std::vector<Run> runs;
      for (int q = bt.mat0; q < bt.mat0 + bt.n_mats; ++q) {
        const NsHfMat& b = L.nsb_mats[q];
        const double w = ns_work(b.m, b.n);
        if (!runs.empty() && L.nsb_mats[runs.back().q0].tensor == b.tensor) { runs.back().q1 = q + 1; runs.back().work += w; }
        else runs.push_back(Run{q, q + 1, w});
      }
      std::stable_sort(runs.begin(), runs.end(), [](const Run& x, const Run& y) { return x.work > y.work; });
      std::vector<double> load(n_groups, 0.0);
      for (const Run& r : runs) {
        const int g = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        for (int q = r.q0; q < r.q1; ++q) members[g].push_back(q);
        load[g] += r.work;
      }
      for (auto& mm : members) std::sort(mm.begin(), mm.end());   // neighbours in memory stay neighbours in the tables
    }
    bt.group0 = (int)L.ns_groups.size();
    bt.n_groups = n_groups;
    // the tiles of the batch's launches (those of its groups run next to each other)
    long long gram_jobs = 0, poly_jobs = 0, upd_jobs = 0, upd4_jobs = 0;
    auto wide_tiles = [&](const NsHfMat& b) { return b.rows_m % 256 == 0 && up(b.m, 256) <= 1.06 * up(b.m, 128); };
    for (int q = bt.mat0; q < bt.mat0 + bt.n_mats; ++q) {
      const NsHfMat& b = L.nsb_mats[q];
      const long long nt = (b.m + kNsTile - 1) / kNsTile, ni = (b.n + kNsTile - 1) / kNsTile;
      gram_jobs += nt * (nt + 1) / 2 * b.n_slabs;
      poly_jobs += nt * (nt + 1) / 2;
      (wide_tiles(b) ? upd4_jobs : upd_jobs) += ni * (wide_tiles(b) ? (b.m + 255) / 256 : nt);
    }
    const int gram_edge = ns_tile_edge(gram_jobs), poly_edge = ns_tile_edge(poly_jobs);
    const bool any_wide = upd4_jobs + upd_jobs >= 256;      // else those of 128 x 256 are cut in two
    const int upd_edge = ns_tile_edge(any_wide ? upd4_jobs + upd_jobs : 2 * upd4_jobs + upd_jobs);
    for (int g = 0; g < n_groups; ++g) {
      // job runs that read the same operands: per matrix (slab), and finer, per row of tiles, for sets of few matrices
      std::vector<std::pair<int, long long>> gram_units, poly_units, upd_units, upd4_units, gram_rows, poly_rows;
      std::vector<NsItem> gram, poly, upd, upd4;
      NsGroup grp{};
      grp.split0 = (int)L.ns_split.size();
      grp.list0 = (int)L.ns_list.size();
      grp.sitem0 = (int)L.nsb_split_items.size();
      grp.fitem0 = (int)L.ns_flag_items.size();
      grp.gram_edge = gram_edge;
      grp.poly_edge = poly_edge;
      grp.upd_edge = upd_edge;
      for (int q : members[g]) {
        {
          NsHfMat& bw = L.nsb_mats[q];
          bw.fpart0 = L.ns_fpart_total;
          bw.n_fpart = 4 * hf_tiles_upper(bw.m);
          L.ns_fpart_total += bw.n_fpart;
          for (int c = 0; c < bw.n_fpart; ++c) L.ns_flag_items.push_back(Item{q, c, 0, 0});
        }
        const NsHfMat& b = L.nsb_mats[q];
        L.ns_list.push_back(q);
        L.ns_group_of_tensor[b.tensor] = (int)L.ns_groups.size();
        for (int tr = 0; tr < (b.R + 63) / 64; ++tr)
          for (int tc = 0; tc < (b.C + 63) / 64; ++tc) L.nsb_split_items.push_back(NsTileItem{q, tr, tc});
        // Gram: the tiles of one matrix (of one slab of it) read the same rows of Xs; Poly: the same A
        auto upper = [&](std::vector<NsItem>& items, std::vector<std::pair<int, long long>>& units,
                         std::vector<std::pair<int, long long>>& rows, int edge, int k0, int k1, int slab) {
          const int nt = (b.m + edge - 1) / edge;
          for (int tm = 0; tm < nt; ++tm) {
            for (int tn = tm; tn < nt; ++tn) items.push_back(NsItem{q, tm, tn, k0, k1, slab});
            rows.push_back({nt - tm, (long long)(k1 - k0)});
          }
          units.push_back({nt * (nt + 1) / 2, (long long)(k1 - k0)});
        };
        for (int sl = 0; sl < b.n_slabs; ++sl) {
          const int slab_k = L.ns_mats[q].slab_k;
          const int k0 = b.n_slabs > 1 ? sl * slab_k : 0;
          const int k1 = b.n_slabs > 1 ? up16(std::min(b.n, (sl + 1) * slab_k)) : up16(b.n);
          upper(gram, gram_units, gram_rows, gram_edge, k0, k1, b.n_slabs > 1 ? sl : -1);
        }
        upper(poly, poly_units, poly_rows, poly_edge, 0, up16(b.m), -1);
        // Update: the tiles of one row block read the same rows of Xl, all of them the same B'
        const bool wide = any_wide && wide_tiles(b);
        const int ei = wide ? kNsTile : upd_edge, ej = wide ? 256 : upd_edge;
        std::vector<NsItem>& u = wide ? upd4 : upd;
        std::vector<std::pair<int, long long>>& units = wide ? upd4_units : upd_units;
        for (int tm = 0; tm < (b.n + ei - 1) / ei; ++tm) {
          const int ntu = (b.m + ej - 1) / ej;
          for (int tn = 0; tn < ntu; ++tn) u.push_back(NsItem{q, tm, tn, 0, up16(b.m), -1});
          units.push_back({ntu, (long long)up16(b.m)});
        }
        if (b.n_slabs > 1) {
          L.ns_split.push_back(q);
          grp.split_max_m = std::max(grp.split_max_m, b.m);
        }
      }
      if (env_ns_xcd()) {
        // with fewer runs than a few per XCD the stretches would be uneven: take the finer runs, or leave the order
        auto pick = [](std::vector<NsItem>& items, const std::vector<std::pair<int, long long>>& coarse,
                       const std::vector<std::pair<int, long long>>& fine) {
          if (coarse.size() >= 4 * kXcds) xcd_interleave(items, coarse);
          else if (fine.size() >= 4 * kXcds) xcd_interleave(items, fine);
        };
        pick(gram, gram_units, gram_rows);
        pick(poly, poly_units, poly_rows);
        pick(upd, upd_units, upd_units);
        pick(upd4, upd4_units, upd4_units);
      }
      auto append = [](std::vector<NsItem>& all, const std::vector<NsItem>& part, int& first, int& count) {
        first = (int)all.size();
        count = (int)part.size();
        all.insert(all.end(), part.begin(), part.end());
      };
      append(L.ns_gram, gram, grp.gram0, grp.n_gram);
      append(L.ns_poly, poly, grp.poly0, grp.n_poly);
      append(L.ns_upd, upd, grp.upd0, grp.n_upd);
      append(L.ns_upd4, upd4, grp.upd40, grp.n_upd4);
      grp.n_split = (int)L.ns_split.size() - grp.split0;
      grp.n_list = (int)L.ns_list.size() - grp.list0;
      grp.n_sitems = (int)L.nsb_split_items.size() - grp.sitem0;
      grp.n_fitems = (int)L.ns_flag_items.size() - grp.fitem0;
      L.ns_groups.push_back(grp);
    }
    }
    return;
  }
  // longest jobs first: the launch ends when its last block does
  auto longer = [](const NsItem& x, const NsItem& y) { return x.k1 - x.k0 > y.k1 - y.k0; };
  std::stable_sort(L.ns_gram.begin(), L.ns_gram.end(), longer);
  std::stable_sort(L.ns_poly.begin(), L.ns_poly.end(), longer);
  std::stable_sort(L.ns_upd.begin(), L.ns_upd.end(), longer);
}

// ELO-CELO2 tensors with more than two dims on the MLP path: the slices of their last two dims, where one fits the
// LDS of the lanes that would own it (k_slice_finish.h).
void build_slice_tables(Layout& L, const PyloTensorShape* shapes, int T) {
  L.slice_of_tensor.assign(T, -1);
  L.slice_mats.clear(); L.slice_items_w.clear(); L.slice_items_b.clear();
  for (int k = 0; k < kSliceLaneSets; ++k) { L.slice_items_l[k].clear(); L.slice_lds_l[k] = 0; }
  L.slice_lds_w = L.slice_lds_b = 0;
  for (int t = 0; t < T; ++t) {
    const TDesc& d = L.descs[t];
    const PyloTensorShape& sh = shapes[t];
    if (d.mode != kModeFacND || d.n == 0 || sh.ndim < 3) continue;
    SliceMat sm{};
    sm.tensor = t;
    sm.R = (int)sh.shape[sh.ndim - 2];
    sm.C = (int)sh.shape[sh.ndim - 1];
    sm.slices = d.n / ((long long)sm.R * sm.C);
    sm.no_orth = (sh.flags & PYLO_F_NO_ORTHOGONALIZE) != 0;
    if (!slice_geometry(sm)) continue;
    const int per_block = sm.lanes == 1 ? 64 : 256 / sm.lanes;
    const long long blocks = (sm.slices + per_block - 1) / per_block;
    if (blocks >= (1ll << 31)) continue;
    const int q = (int)L.slice_mats.size();
    L.slice_of_tensor[t] = q;
    // lane-owned slices: one launch per register size, and per LDS size class of the others (a wave's LDS share
    // decides how many waves a CU holds)
    int set = 0;
    if (sm.lanes == 1) {
      const long long need = slice_lane_lds(sm.m, sm.n);
      set = slice_in_registers(sm.m, sm.n) ? sm.m / 2 : need <= 12 * 1024 ? 4 : need <= 28 * 1024 ? 5 : 6;
    }
    std::vector<Item>& items = sm.lanes == 1 ? L.slice_items_l[set] : sm.lanes == 256 ? L.slice_items_b : L.slice_items_w;
    int& lds = sm.lanes == 1 ? L.slice_lds_l[set] : sm.lanes == 256 ? L.slice_lds_b : L.slice_lds_w;
    lds = std::max(lds, sm.lanes == 1 ? (int)slice_lane_lds(sm.m, sm.n) : (int)sizeof(float) * sm.per_floats * per_block);
    for (long long b = 0; b < blocks; ++b) items.push_back(Item{q, (int)b, 0, 0});
    L.slice_mats.push_back(sm);
  }
}

// Units and blocks of ELO-CELO2's finishing pass (after Newton-Schulz): a unit is what one normaliser runs over, cut
// into linear 8192-element blocks.  MLP tensors of up to two dims are one unit; a tensor with more dims whose slices
// the per-slice launches do not take (k_slice_finish.h) is one unit per slice of its last two dims.  The tables
// hold the tensors of each group of Newton-Schulz matrices together (a group finishes its own tensors on its own
// stream), then the tensors of no group.
int build_fin_tables(Layout& L, const PyloTensorShape* shapes, int T) {
  L.fin_units.clear(); L.fin_items.clear();
  auto add = [&](int t) {
    TDesc& d = L.descs[t];
    d.fin_unit0 = (int)L.fin_units.size();
    d.fin_units = 0;
    if (d.mode == kModeFlat || d.n == 0 || L.small_of_tensor[t]) return;
    long long slices = 1, len = d.n;
    if (d.mode == kModeFacND) {
      if (L.slice_of_tensor[t] >= 0) return;
      len = shapes[t].shape[shapes[t].ndim - 2] * shapes[t].shape[shapes[t].ndim - 1];
      slices = d.n / len;
    }
    for (long long sl = 0; sl < slices; ++sl) {
      FinUnit u{};
      u.tensor = t;
      u.off = sl * len;
      u.n = len;
      u.vec = len % 4 == 0;
      u.blk0 = (int)L.fin_items.size();
      const int unit = (int)L.fin_units.size();
      for (long long c = 0; c * kFinElems < len; ++c) L.fin_items.push_back(Item{unit, (int)c, 0, 0});
      u.nblk = (int)L.fin_items.size() - u.blk0;
      L.fin_units.push_back(u);
    }
    d.fin_units = (int)slices;
  };
  for (size_t g = 0; g < L.ns_groups.size(); ++g) {
    NsGroup& grp = L.ns_groups[g];
    grp.fin0 = (int)L.fin_items.size();
    grp.unit0 = (int)L.fin_units.size();
    for (int t = 0; t < T; ++t)
      if (L.ns_group_of_tensor[t] == (int)g) add(t);
    grp.n_fin = (int)L.fin_items.size() - grp.fin0;
    grp.n_units = (int)L.fin_units.size() - grp.unit0;
    if (L.fin_items.size() >= (1u << 30)) return fail("plan: too many blocks in the finishing pass");
  }
  L.fin_rest0 = (int)L.fin_items.size();
  L.unit_rest0 = (int)L.fin_units.size();
  for (int t = 0; t < T; ++t)
    if (L.ns_group_of_tensor[t] < 0) add(t);
  L.n_fin_rest = (int)L.fin_items.size() - L.fin_rest0;
  L.n_unit_rest = (int)L.fin_units.size() - L.unit_rest0;
  if (L.fin_items.size() >= (1u << 30)) return fail("plan: too many blocks in the finishing pass");
  for (NsMat& m : L.ns_mats) m.unit += L.descs[m.tensor].fin_unit0;
  return 0;
}

int build_layout(int kind, const PyloTensorShape* shapes, int T, Layout& L, int velo_hidden) {
  if (kind != PYLO_KIND_CELO2 && kind != PYLO_KIND_VELO && kind != PYLO_KIND_ADAFAC)
    return fail("plan: unknown optimizer kind");
  if (T <= 0 || shapes == nullptr) return fail("plan: no tensors");
  L.H = first_layer_width(kind);
  L.descs.assign(T, TDesc{});
  L.dc.assign(T, -1);
  L.dr.assign(T, -1);
  long long part = 0, fac = 0, term = 0;
  std::vector<int> lin_tensors;   // AdafacLO: tensors of the linear apply pass
  long long v0a_blocks = 0;
  const int H = L.H;
  long long total_elems = 0;
  for (int t = 0; t < T; ++t) {
    long long n = 1;
    for (int i = 0; i < std::max(0, std::min(shapes[t].ndim, PYLO_MAX_DIMS)); ++i) n *= std::min<long long>(std::max<long long>(shapes[t].shape[i], 0), 1ll << 31) , n = std::min(n, 1ll << 31);
    total_elems += n;
  }
  const int split = split_for(total_elems);
  L.split = split > 1;
  // Rows of a wave task of AdafacLO's walks: a wave's set-up (weights split into planes, column terms, three dependent loads
  // before the first row) costs about as much as a row, so rows are doubled up to 64 while 16384 tasks, five rounds of what
  // runs at once, are left.  Whole steps, 16 / 32 / 64 rows: 22 M elements 505 / 505 / 520 us, 86 M 1769 / 1741 / 1733, 124 M
  // 2476 / 2418 / 2404, 355 M 6872 / 6700 / 6611.
  int apply_rows = tile_rows_for(kind, split);
  while (apply_rows >= kTileRows && apply_rows < kApplyRowsMax && total_elems >= 16384ll * 64 * 2 * apply_rows) apply_rows *= 2;
  L.tensor_norm = (shapes[0].flags & PYLO_F_TENSOR_NORM) != 0;
  L.global_norm = (shapes[0].flags & PYLO_F_GLOBAL_NORM) != 0 || L.tensor_norm;
  // Short slices (k_celo2_slices_wave): trips a wave, as many as leave sixteen waves a CU and no more than eight
  // (the set-up of a wave, its weights, costs about as much as a trip).
  long long slice_elems = 0;
  for (int t = 0; t < T && kind == PYLO_KIND_CELO2; ++t) {
    const PyloTensorShape& s = shapes[t];
    if (s.ndim < 3 || s.ndim > PYLO_MAX_DIMS || s.shape[s.ndim - 2] * s.shape[s.ndim - 1] > kSliceLaneMax) continue;
    long long n = 1;
    for (int i = 0; i < s.ndim; ++i) n *= s.shape[i];
    slice_elems += n;
  }
  const int slice_trips = (int)std::max<long long>(1, std::min<long long>(8, slice_elems / (64 * 16 * 256)));
  auto short_slices = [&](const TDesc& d) { return d.mode == kModeFacND && d.slice_len <= kSliceLaneMax && env_slices_lds(); };
  for (int t = 0; t < T; ++t) {
    const PyloTensorShape& s = shapes[t];
    if (s.ndim < 0 || s.ndim > PYLO_MAX_DIMS) return fail("plan: bad ndim");
    long long n = 1;
    int rank = 0;
    for (int i = 0; i < s.ndim; ++i) {
      if (s.shape[i] < 0) return fail("plan: negative dim");
      n *= s.shape[i];
      rank += s.shape[i] > 1;
    }
    if (n >= (1ll << 31)) return fail("plan: tensors of 2^31 or more elements are not supported");
    TDesc& d = L.descs[t];
    d.n = n;
    d.iters = std::max(1, kElemIters / split);
    d.gscale = 1.0f;
    if ((s.flags & (PYLO_F_NAN_TO_NUM | PYLO_F_WD_PRESTEP | PYLO_F_GLOBAL_NORM | PYLO_F_TENSOR_NORM)) &&
        kind != PYLO_KIND_ADAFAC)
      return fail("plan: PYLO_F_NAN_TO_NUM / PYLO_F_WD_PRESTEP / PYLO_F_GLOBAL_NORM / PYLO_F_TENSOR_NORM belong to "
                  "AdafacLO plans");
    if (((s.flags & PYLO_F_TENSOR_NORM) != 0) != L.tensor_norm)
      return fail("plan: PYLO_F_TENSOR_NORM must be set on every tensor of the plan or on none");
    if (L.tensor_norm && (s.flags & (PYLO_F_GLOBAL_NORM | PYLO_F_NAN_TO_NUM)))
      return fail("plan: PYLO_F_TENSOR_NORM does not combine with PYLO_F_GLOBAL_NORM or PYLO_F_NAN_TO_NUM");
    if (!L.tensor_norm && ((s.flags & PYLO_F_GLOBAL_NORM) != 0) != L.global_norm)
      return fail("plan: PYLO_F_GLOBAL_NORM must be set on every tensor of the plan or on none");
    d.own_norm = L.tensor_norm ? 1 : 0;
    d.nan0 = (s.flags & PYLO_F_NAN_TO_NUM) != 0;
    d.store = (s.flags & PYLO_F_STORE_MASK) >> 8;
    d.wd_prestep = (s.flags & PYLO_F_WD_PRESTEP) != 0;
    d.fac_slot = -1;
    d.rank = rank < 4 ? rank : 4;
    int dc = -1, dr = -1;
    const bool can_factor = factored_dims(kind, s, &dc, &dr);
    if (kind == PYLO_KIND_CELO2) {
      const bool adam = (s.flags & (PYLO_F_ADAM | PYLO_F_ADAM_INDEP)) != 0;
      d.adam_indep = (s.flags & PYLO_F_ADAM_INDEP) != 0;
      if (adam) d.mode = kModeFlat;
      else if (!can_factor) d.mode = kModeVec;  // the MLP on a tensor with fewer than two dims
      else d.mode = s.ndim == 2 ? kModeFac2D : kModeFacND;
      if (d.mode == kModeVec) d.slice_len = (int)std::max<long long>(n, 1);
      if (d.mode == kModeFacND) d.slice_len = (int)std::max<long long>(s.shape[s.ndim - 2] * s.shape[s.ndim - 1], 1);
    } else {
      d.mode = !can_factor ? kModeVec : (s.ndim == 2 ? kModeFac2D : kModeFacND);
    }
    // Geometry is laid out over the dims that matter: dims of size 1 other than the two factored ones
    // change neither strides nor sums, so a (O, I, 1, 1) convolution kernel or a (1, 1, C) token is a
    // plain 2-D tensor for the kernels (vectorised loads, column-resident walk).  Not for CELO2, whose
    // normalisers run over slices of the last two dims as given.
    PyloTensorShape e = s;
    int edc = dc, edr = dr;
    if (can_factor && kind != PYLO_KIND_CELO2 && n > 0) {
      e.ndim = 0;
      for (int i = 0; i < s.ndim; ++i) {
        if (s.shape[i] == 1 && i != dc && i != dr) continue;
        if (i == dc) edc = e.ndim;
        if (i == dr) edr = e.ndim;
        e.shape[e.ndim++] = s.shape[i];
      }
      d.mode = e.ndim == 2 ? kModeFac2D : kModeFacND;
    }
    if (d.mode == kModeFlat || d.mode == kModeVec) {
      d.vec = (n % 4 == 0) ? 4 : 1;
    } else {
      L.dc[t] = dc;
      L.dr[t] = dr;
      if (d.mode == kModeFac2D) {
        d.R0 = (int)e.shape[0];
        d.C0 = (int)e.shape[1];
        d.vec = (d.C0 % 4 == 0) ? 4 : 1;
        d.vec0_is_r = (edr == 1) ? 1 : 0;  // vector 0 (indexed by dim 0) results from summing over dim 1
        d.len[0] = d.R0; d.len[1] = d.C0;
        d.sumlen[0] = d.C0; d.sumlen[1] = d.R0;
        // (16-bit gradients that k_p0 reads itself are taken in the usual tiles)
        const bool typed16 = d.store == kStoreF16 || d.store == kStoreBF16;
        d.p0_thin = typed16 ? 0 : d.R0 <= kP0Thin && d.C0 > 64 * d.vec ? 1 : d.C0 <= kP0Thin && d.R0 > kP0Rows ? 2 : 0;
        const int tile_r = d.p0_thin == 2 ? kP0Long : kP0Rows, tile_c = d.p0_thin == 1 ? kP0Long : 64 * d.vec;
        d.n_strips = (d.R0 + tile_r - 1) / tile_r;
        d.n_colblk = (d.C0 + tile_c - 1) / tile_c;
        d.npart[0] = d.n_colblk * (d.p0_thin == 1 ? 2 : 1); d.npart[1] = d.n_strips * (d.p0_thin == 2 ? 2 : 1);   // p0_thin_total: two
        d.nd_div_blk[0] = make_fastdiv((unsigned)std::max(d.C0, 1));   // element -> row (k_adafac_apply_lin)
      } else {
        d.vec = 1;
        d.vec0_is_r = 1;
        const int rem[2] = {edr, edc};  // the dim each vector lost
        for (int w = 0; w < 2; ++w) {
          long long stride = 1;
          for (int i = rem[w] + 1; i < e.ndim; ++i) stride *= e.shape[i];
          d.nd_size[w] = (int)e.shape[rem[w]];
          d.nd_stride[w] = (int)stride;
          d.nd_div_blk[w] = make_fastdiv((unsigned)std::max<long long>(e.shape[rem[w]] * stride, 1));
          d.nd_div_st[w] = make_fastdiv((unsigned)std::max<long long>(stride, 1));
          d.len[w] = d.nd_size[w] > 0 ? (int)(n / d.nd_size[w]) : 0;
          d.sumlen[w] = d.nd_size[w];
          d.npart[w] = std::max(1, (d.nd_size[w] + kNdX - 1) / kNdX);
        }
        // the dc axis as it sits inside the row vector (the tensor without dim dr)
        d.rcm_size = d.nd_size[1];
        d.rcm_stride = edc > edr ? d.nd_stride[1] : d.nd_stride[1] / std::max(d.nd_size[0], 1);
      }
      for (int w = 0; w < 2; ++w) {
        d.pitch[w] = (int)round4(d.len[w]);
        d.part_off[w] = part;
        part += round4((long long)d.npart[w] * d.len[w]);
        d.fac_off[w] = fac;              // [entry][4]
        fac += (long long)d.len[w] * 4;
        d.term_off[w] = term;            // [entry][H]
        term += round4((long long)d.len[w] * H);
      }
      if (n > 0) {
        d.fac_slot = (int)L.fac_list.size();
        L.fac_list.push_back(t);
        for (int w = 0; w < 2; ++w) {
          v0a_blocks += (d.len[w] + kV0aEnt - 1) / kV0aEnt;
          for (int c = 0; c * kV0bEnt < d.len[w]; ++c) L.v0b_items.push_back(Item{t, c, w, 0});
          if (d.mode == kModeFacND)
            for (int c = 0; c * kV0aEnt < d.len[w]; ++c)
              for (int q = 0; q < d.npart[w]; ++q) L.nd_items.push_back(Item{t, c, w, q});
        }
      }
    }
    const long long chunk = (long long)kThreads * d.vec * d.iters;
    // P0 items: tiles of 2-D factored tensors; flat chunks only where a global norm is needed
    // (CELO2's AdamW tensors, every other tensor of a PYLO_F_GLOBAL_NORM plan)
    d.p0_first = (int)L.p0_items.size();
    if (n > 0) {
      if (d.mode == kModeFac2D) {
        for (int st = 0; st < d.n_strips; ++st)
          for (int cb = 0; cb < d.n_colblk; ++cb) L.p0_items.push_back(Item{t, st, cb, 0});
      } else if (kind == PYLO_KIND_CELO2 || L.global_norm) {
        for (long long c = 0; c * chunk < n; ++c) L.p0_items.push_back(Item{t, (int)c, 0, 0});
      }
    }
    d.p0_n = (int)L.p0_items.size() - d.p0_first;
    d.blk0 = (int)L.el_items.size();
    const bool wide = d.mode == kModeFac2D && n > 0 && env_matrix_pipe();
    if (kind == PYLO_KIND_CELO2 && (d.mode == kModeFacND || d.mode == kModeVec)) {
      // one pass per slice of the last two dims (k_celo2_slices): 256 slices a block, or 4
      const long long n_slices = n / d.slice_len, per = d.slice_len <= kSliceLaneMax ? kThreads : kWaves;
      if (n_slices >= (1ll << 31)) return fail("plan: too many slices");
      if (short_slices(d)) {
        // short slices of a tensor with more than two dims: packed into waves (k_celo2_slices_wave)
        d.slice_runs = d.nd_stride[0] % d.slice_len == 0 && d.nd_stride[1] % d.slice_len == 0;
        L.slice_runs = L.slice_runs || d.slice_runs;
        const int cls = !d.slice_runs ? kSliceGather : d.slice_len == 1 ? kSliceOne : d.slice_len == 9 ? kSliceNine : kSliceAny;
        const long long per_wave = 64 / d.slice_len;
        for (long long s0 = 0; s0 < n_slices && n > 0; s0 += kWaves * per_wave * slice_trips)
          L.sl_wave_cls[cls].push_back(Item{t, (int)s0, slice_trips, 0});
      } else
      for (long long s0 = 0; s0 < n_slices && n > 0; s0 += per) L.sl_items.push_back(Item{t, (int)s0, 0, 0});
    } else if (wide && d.C0 % kTileCols == 0) {
      d.tile_nct = d.C0 / kTileCols;
      d.tile_rows = tile_rows_for(kind, split);
      d.tile_ntask = d.tile_nct * ((d.R0 + d.tile_rows - 1) / d.tile_rows);
      d.direct = (kind != PYLO_KIND_ADAFAC || env_adafac_hf()) && (d.store == kStoreF16 || d.store == kStoreBF16);
      L.in_place = L.in_place || d.direct;
      for (int b = 0; b * 4 < d.tile_ntask; ++b) L.el_items.push_back(Item{t, b, 0, 0});
    } else {
      for (long long c = 0; c * chunk < n; ++c) L.el_items.push_back(Item{t, (int)c, 0, 0});
    }
    d.nblk = (int)L.el_items.size() - d.blk0;
    if (d.nblk > kSegMin) {  // two-stage reduction of the statistics partials (k_stat_segsum)
      d.seg0 = (int)L.seg_items.size();
      for (int r = 0; r < d.nblk; r += kSegRows) L.seg_items.push_back(Item{t, r, std::min(kSegRows, d.nblk - r), (int)L.seg_items.size()});
      d.nseg = (int)L.seg_items.size() - d.seg0;
    }
    // blocks of AdafacLO's apply pass: one column per lane where the tensor allows it (ap_items,
    // k_adafac_apply_tile), linear chunks otherwise (ga_items, k_adafac_apply)
    if (kind == PYLO_KIND_ADAFAC) {
      // an (O, I, k, ..) tensor factored over its two leading dims (convolution kernels) is the matrix (O, I * P)
      // for this pass, P = product of the trailing dims (pp_items)
      bool periodic = false;
      if (d.mode == kModeFacND && n > 0 && env_matrix_pipe() && env_adafac_hf() && e.ndim >= 3 &&
          ((edr == 0 && edc == 1) || (edr == 1 && edc == 0))) {
        long long P = 1;
        for (int i = 2; i < e.ndim; ++i) P *= e.shape[i];
        if ((e.shape[1] * P) % 64 == 0) {
          periodic = true;
          d.aper = (int)P;
          d.aper_col = edr == 0 ? 0 : 1;   // vector 0 lost dim edr: it is indexed by the column if that dim is O
          d.R0 = (int)e.shape[0];
          d.C0 = (int)(e.shape[1] * P);
        }
      }
      if ((wide && d.C0 % 64 == 0) || periodic) {
        d.atile_nct = d.C0 / 64;
        // The walk's offsets inside a task are 32-bit byte offsets: 4 C0 a row into the tensor, and, where the row side has an
        // entry per column mod P, 128 P a row into its first-layer terms, the larger ones for I < 32.  (P, the product of up to
        // six dims none of which exceeds the two leading ones, stays below 2^24 in a tensor of 2^31 elements: one row always fits.)
        long long rows_max = (1ll << 30) / d.C0;
        if (periodic) rows_max = std::min<long long>(rows_max, (1ll << 31) / ((long long)sizeof(float) * kAH * d.aper));
        d.atile_rows = (int)std::max<long long>(1, std::min<long long>(apply_rows, rows_max));
        d.atile_ntask = d.atile_nct * ((d.R0 + d.atile_rows - 1) / d.atile_rows);
        for (int b = 0; b * 4 < d.atile_ntask; ++b) (periodic ? L.pp_items : L.ap_items).push_back(Item{t, b, 0, 0});
      } else {
        lin_tensors.push_back(t);
      }
    }
  }
  // Blocks of k_v0a: four times the entries where there are more of them than the chip holds at a time (2048)
  for (int t : L.fac_list) {
    TDesc& d = L.descs[t];
    for (int w = 0; w < 2; ++w) {
      const bool wide = v0a_blocks > 4096 && d.npart[w] <= kV0aParts && d.len[w] > kV0aEnt;
      const int ent = wide ? kV0aWide : kV0aEnt;
      d.v0a_first[w] = (int)L.v0a_items.size();
      for (int c = 0; c * ent < d.len[w]; ++c) L.v0a_items.push_back(Item{t, c, w, wide ? 1 : 0});
      d.v0a_n[w] = (int)L.v0a_items.size() - d.v0a_first[w];
    }
  }
  // Blocks of AdafacLO's linear apply pass: on the matrix pipe Item::b trips of 256 elements each, as many as leave
  // every SIMD the two waves it holds and no more than 16 (the set-up of a wave, its weights,
  // costs about as much as a trip); else 8192- / 2048-element chunks.
  L.lin_matrix = env_matrix_pipe();
  long long lin_elems = 0;
  for (int t : lin_tensors) lin_elems += L.descs[t].n;
  const int trips = (int)std::max<long long>(1, std::min<long long>(16, lin_elems / (2 * 256 * kThreads)));
  for (int t : lin_tensors) {
    const long long chunk = L.lin_matrix ? (long long)kThreads * trips : (long long)kThreads * L.descs[t].vec * kElemIters;
    for (long long c = 0; c * chunk < L.descs[t].n; ++c) L.ga_items.push_back(Item{t, (int)c, L.lin_matrix ? trips : 0, 0});
  }
  for (int i = 0; i < (int)L.el_items.size(); ++i) L.el_items[i].b = i;   // rows of the partial sums
  if (kind == PYLO_KIND_CELO2 || kind == PYLO_KIND_VELO) build_elem_items(L, T, kind);
  long long ns_floats = 0;
  if (kind == PYLO_KIND_CELO2) {
    L.ns_hf = env_ns_hf();
    build_slice_tables(L, shapes, T);
    build_ns_tables(L, shapes, T, ns_floats);
    if (int rc = build_fin_tables(L, shapes, T)) return rc;
  }
  // fp32 staging of tensors in other storage types (k_cast.h)
  for (int t = 0; t < T; ++t) {
    const TDesc& d = L.descs[t];
    L.stage_ofs.push_back(StageOfs{-1, -1});
    if (d.store == kStoreF32 || d.n == 0) continue;
    L.typed = true;
    if (d.direct) continue;
    const long long pitch = (d.n + 63) / 64 * 64;
    L.stage_ofs.back() = StageOfs{L.stage_floats, L.stage_floats + pitch};
    L.stage_floats += 2 * pitch;
    for (long long c = 0; c * kCastElems < d.n; ++c) L.cast_items.push_back(Item{t, (int)c, 0, 0});
  }
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off = align_up(off + std::max<size_t>(bytes, 16));
    return o;
  };
  const size_t nfac = std::max<size_t>(L.fac_list.size(), 1);
  L.off_descs = take(sizeof(TDesc) * T);
  L.off_dyn = take(sizeof(PyloTensorArgs) * T);
  L.off_dyn_user = L.typed ? take(sizeof(PyloTensorArgs) * T) : L.off_dyn;
  L.off_stage_ofs = take(L.typed ? sizeof(StageOfs) * T : 0);
  L.off_cast_items = take(sizeof(Item) * L.cast_items.size());
  L.off_stage = take(sizeof(float) * (size_t)L.stage_floats);
  L.off_p0_items = take(sizeof(Item) * L.p0_items.size());
  L.off_nd_items = take(sizeof(Item) * L.nd_items.size());
  L.off_sl_items = take(sizeof(Item) * L.sl_items.size());
  for (int c = 0; c < kSliceWaveClasses; ++c) {
    L.sl_wave_n[c] = (int)L.sl_wave_cls[c].size();
    L.sl_wave_items.insert(L.sl_wave_items.end(), L.sl_wave_cls[c].begin(), L.sl_wave_cls[c].end());
    L.sl_wave_cls[c] = std::vector<Item>();
  }
  L.off_sl_wave_items = take(sizeof(Item) * L.sl_wave_items.size());
  L.off_seg_items = take(sizeof(Item) * L.seg_items.size());
  L.off_segtot = take(sizeof(double) * kStatW * L.seg_items.size());
  L.off_el_items = take(sizeof(Item) * L.el_items.size());
  L.off_ap_items = take(sizeof(Item) * L.ap_items.size());
  L.off_pp_items = take(sizeof(Item) * L.pp_items.size());
  L.off_ga_items = take(sizeof(Item) * L.ga_items.size());
  L.off_fin_items = take(sizeof(Item) * L.fin_items.size());
  L.off_finpart = take(sizeof(double) * L.fin_items.size());
  L.off_finscale = take(sizeof(float) * L.fin_units.size());
  L.off_fin_units = take(sizeof(FinUnit) * L.fin_units.size());
  L.off_v0a_items = take(sizeof(Item) * L.v0a_items.size());
  L.off_v0b_items = take(sizeof(Item) * L.v0b_items.size());
  L.off_fac_list = take(sizeof(int) * nfac);
  L.off_part = take(sizeof(float) * part);
  L.off_gsq = take(sizeof(double) * L.p0_items.size());
  L.off_flag = take(sizeof(int) * L.p0_items.size());
  L.off_globals = take(sizeof(Globals));
  L.off_tscale = take(sizeof(float) * (L.tensor_norm ? T : 0));
  L.off_fac = take(sizeof(float) * fac);
  L.off_term = take(sizeof(float) * term);
  L.off_v0part = take(sizeof(double) * kNV0 * L.v0a_items.size());
  L.off_bscale = take(sizeof(BScale) * nfac);
  L.off_stats = take(sizeof(double) * kStatW * L.el_items.size());
  L.off_wfold = take(sizeof(float) * (kind == PYLO_KIND_CELO2 ? kC2Fold * nfac
                                      : kind == PYLO_KIND_VELO ? (size_t)kVFold * T : (size_t)kAFold * T));
  L.off_chan_ms = take(sizeof(float) * kNStat * nfac);
  L.off_totals = take(sizeof(double) * kStatW * T);
  L.Tpad = (T + kGateBT - 1) / kGateBT * kGateBT;
  L.off_xfeat = take(sizeof(float) * kXW * T);
  L.off_lossfeat = take(sizeof(float) * 16);
  L.off_xT = take(kind == PYLO_KIND_VELO ? sizeof(float) * 2 * (size_t)velo_hidden * L.Tpad : 0);
  L.off_mixbuf = take(kind == PYLO_KIND_VELO ? sizeof(float) * 2 * (size_t)velo_hidden * T : 0);
  L.off_pmax = take(kind == PYLO_KIND_VELO ? sizeof(float) * (size_t)velo_hidden * ((T + kMixRows - 1) / kMixRows) : 0);
  L.off_canon = take(kind == PYLO_KIND_VELO ? sizeof(float) * kVCanon * (size_t)T : 0);
  L.off_frac = take(kind == PYLO_KIND_VELO ? sizeof(float) * 9 * PYLO_MAX_GROUPS : 0);
  L.off_mx_items = take(sizeof(Item) * L.mx_items.size());
  L.off_big_items = take(sizeof(Item) * L.big_items.size());
  L.off_big_apply = take(sizeof(Item) * L.big_apply.size());
  L.off_big_seg = take(sizeof(Item) * L.big_seg.size());
  L.off_big_list = take(sizeof(int) * L.big_list.size());
  // (VeLO: behind the counters, the guard of the carried sums: flag address, padding, T doubles -- k_velo.h)
  L.off_sync = take(sizeof(int) * (size_t)((2 * T + 3) & ~3) + (kind == PYLO_KIND_VELO ? 16 + sizeof(double) * (size_t)T : 0));
  L.off_newsum = take(kind == PYLO_KIND_VELO ? sizeof(double) * kNewSumW * L.el_items.size() : 0);
  L.off_piv = take(kind == PYLO_KIND_VELO ? sizeof(float) * 4 * (size_t)T : 0);
  L.off_wmix = take(kind == PYLO_KIND_VELO ? sizeof(float) * 160 * (size_t)T : 0);
  if (kind == PYLO_KIND_CELO2) {
    L.off_ns_mats = take(sizeof(NsMat) * L.ns_mats.size());
    L.off_ns_gram = take(sizeof(NsItem) * L.ns_gram.size());
    L.off_ns_poly = take(sizeof(NsItem) * L.ns_poly.size());
    L.off_ns_upd = take(sizeof(NsItem) * L.ns_upd.size());
    L.off_ns_upd4 = take(sizeof(NsItem) * L.ns_upd4.size());
    L.off_ns_split = take(sizeof(int) * L.ns_split.size());
    L.off_ns_xalt = take(sizeof(long long) * (size_t)T);
    L.off_ns_scale = take(sizeof(float) * L.ns_mats.size());
    L.off_ns_flags = take(sizeof(int) * L.ns_mats.size());
    L.off_ns_fpart = take(sizeof(float) * (size_t)L.ns_fpart_total);
    L.off_ns_flag_items = take(sizeof(Item) * L.ns_flag_items.size());
    L.off_ns_ws = take(sizeof(float) * (size_t)ns_floats);
    L.off_nsb_mats = take(sizeof(NsHfMat) * L.nsb_mats.size());
    L.off_nsb_split_items = take(sizeof(NsTileItem) * L.nsb_split_items.size());
    L.off_ns_list = take(sizeof(int) * L.ns_list.size());
    L.off_ns_pw = take(sizeof(hbits) * (size_t)L.nsb_plane_elems);
    L.off_sm_mats = take(sizeof(NsSmall) * L.sm_mats.size());
    for (int k = 0; k < kNsSmallClasses; ++k) L.off_sm_items[k] = take(sizeof(NsSmallItem) * L.sm_items[k].size());
    L.off_sm_part = take(sizeof(float) * (size_t)L.sm_part_floats);
    L.off_sm_sums = take(sizeof(double) * (size_t)L.sm_sums);
    L.off_sm_sync = take(sizeof(int) * (size_t)L.sm_sync);
    L.off_slice_mats = take(sizeof(SliceMat) * L.slice_mats.size());
    for (int k = 0; k < kSliceLaneSets; ++k) L.off_slice_items_l[k] = take(sizeof(Item) * L.slice_items_l[k].size());
    L.off_slice_items_w = take(sizeof(Item) * L.slice_items_w.size());
    L.off_slice_items_b = take(sizeof(Item) * L.slice_items_b.size());
  }
  L.total = off;
  return 0;
}

constexpr int kStageSlots = PYLO_ARG_TABLES;
constexpr int kVeloHiddenMax = 1024;  // workspace is sized for LSTM widths up to this

}  // namespace

struct PyloPlan {
  int kind = 0, T = 0;
  Layout L;
  char* ws = nullptr;
  PyloTensorArgs* stage[kStageSlots] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t ev[kStageSlots] = {nullptr, nullptr, nullptr, nullptr};
  bool ev_used[kStageSlots] = {false, false, false, false};
  bool handed[kStageSlots] = {false, false, false, false};  // given to the caller by plan_arg_table
  int slot = 0;
  PyloDeviceSteps dsteps = {nullptr, 0.0, 0.0, 1.0};
  std::vector<PyloTensorArgs> last;
  size_t last_dst = 0;   // where `last` was copied to
  bool have_last = false;
  bool mlp_on_matrix_pipe = true;  // env_matrix_pipe() when the plan was created
  bool adafac_hf = true;           // AdafacLO's element MLP on the fp16 matrix instructions (PYLO_MI355_ADAFAC_F32=1: fp32 ones)
  // optional per-launch timing (pylo_mi355_plan_timing_begin/end)
  std::vector<hipEvent_t> tev;
  int t_steps_max = 0, t_steps = 0, t_per_step = 0;
  bool timing = false;
  // VeLO: the LSTM's input sums were left by the previous step's apply items (see k_velo_elem); false
  // until a step has run and after pylo_mi355_plan_invalidate_statistics
  bool stats_carried = false;
  // the guard of those sums: 1 + tensor in pinned host memory that the kernel writes straight into when it catches a
  // mismatch (nothing is copied on the steps that find none; pylo_mi355_plan_invalidate_statistics clears it), and
  // its address as the device sees it
  int* stale_host = nullptr;
  int* stale_dev = nullptr;
  hipStream_t side = nullptr;            // the LSTM runs next to the gradient sums on a stream of the plan's own
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  // ELO-CELO2: the Newton-Schulz chains of several groups of matrices run on streams of the plan's own (env_ns_groups)
  hipStream_t ns_side[4] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t ns_fork = nullptr, ns_join[4] = {nullptr, nullptr, nullptr, nullptr};
  // the per-slice finishing launches next to the matrices' products, where the groups leave a hardware queue free
  hipStream_t slice_side = nullptr;
  hipStream_t small_side = nullptr;   // two of the small matrices' classes (enqueue_small)
  hipEvent_t small_fork = nullptr, small_join = nullptr;
  float thin_c[3] = {};               // what thin_run (thin_runs) was worked out for
  int thin_iters = 0;
  std::vector<int> thin_run;
  hipEvent_t slice_fork = nullptr, slice_join = nullptr;

  template <class Tp>
  Tp* at(size_t off) const { return reinterpret_cast<Tp*>(ws + off); }
};

extern "C" {

int pylo_mi355_abi_version(void) { return PYLO_MI355_ABI_VERSION; }

const char* pylo_mi355_last_error(void) { return g_err.c_str(); }

int pylo_mi355_plan_workspace_bytes(int kind, const PyloTensorShape* shapes, int n_tensors, size_t* bytes_out) {
  if (!bytes_out) return fail("workspace_bytes: null output");
  Layout L;
  if (int rc = build_layout(kind, shapes, n_tensors, L, kVeloHiddenMax)) return rc;
  *bytes_out = L.total;
  return 0;
}

int pylo_mi355_plan_create(int kind, const PyloTensorShape* shapes, int n_tensors, void* workspace,
                           size_t workspace_bytes, void* stream, PyloPlan** plan_out) {
  if (!plan_out) return fail("plan_create: null output");
  *plan_out = nullptr;
  PyloPlan* P = new PyloPlan();
  P->kind = kind;
  P->T = n_tensors;
  P->mlp_on_matrix_pipe = env_matrix_pipe();
  P->adafac_hf = env_adafac_hf();
  if (int rc = build_layout(kind, shapes, n_tensors, P->L, kVeloHiddenMax)) { delete P; return rc; }
  if (workspace == nullptr || workspace_bytes < P->L.total) { delete P; return fail("plan_create: workspace too small"); }
  if (reinterpret_cast<uintptr_t>(workspace) % 256 != 0) { delete P; return fail("plan_create: workspace must be 256-byte aligned"); }
  P->ws = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const Layout& L = P->L;
  auto up = [&](size_t off, const void* src, size_t bytes) -> hipError_t {
    if (bytes == 0) return hipSuccess;
    return hipMemcpyAsync(P->ws + off, src, bytes, hipMemcpyHostToDevice, s);
  };
  hipError_t e = hipSuccess;
  if (e == hipSuccess) e = up(L.off_descs, L.descs.data(), sizeof(TDesc) * L.descs.size());
  if (e == hipSuccess) e = up(L.off_p0_items, L.p0_items.data(), sizeof(Item) * L.p0_items.size());
  if (e == hipSuccess && L.typed) e = up(L.off_stage_ofs, L.stage_ofs.data(), sizeof(StageOfs) * L.stage_ofs.size());
  if (e == hipSuccess) e = up(L.off_cast_items, L.cast_items.data(), sizeof(Item) * L.cast_items.size());
  if (e == hipSuccess) e = up(L.off_nd_items, L.nd_items.data(), sizeof(Item) * L.nd_items.size());
  if (e == hipSuccess) e = up(L.off_sl_items, L.sl_items.data(), sizeof(Item) * L.sl_items.size());
  if (e == hipSuccess) e = up(L.off_sl_wave_items, L.sl_wave_items.data(), sizeof(Item) * L.sl_wave_items.size());
  if (e == hipSuccess) e = up(L.off_seg_items, L.seg_items.data(), sizeof(Item) * L.seg_items.size());
  if (e == hipSuccess) e = up(L.off_el_items, L.el_items.data(), sizeof(Item) * L.el_items.size());
  if (e == hipSuccess) e = up(L.off_ap_items, L.ap_items.data(), sizeof(Item) * L.ap_items.size());
  if (e == hipSuccess) e = up(L.off_pp_items, L.pp_items.data(), sizeof(Item) * L.pp_items.size());
  if (e == hipSuccess) e = up(L.off_ga_items, L.ga_items.data(), sizeof(Item) * L.ga_items.size());
  if (e == hipSuccess) e = up(L.off_fin_items, L.fin_items.data(), sizeof(Item) * L.fin_items.size());
  if (e == hipSuccess) e = up(L.off_fin_units, L.fin_units.data(), sizeof(FinUnit) * L.fin_units.size());
  if (e == hipSuccess) e = up(L.off_fac_list, L.fac_list.data(), sizeof(int) * L.fac_list.size());
  if (e == hipSuccess) e = up(L.off_v0a_items, L.v0a_items.data(), sizeof(Item) * L.v0a_items.size());
  if (e == hipSuccess) e = up(L.off_v0b_items, L.v0b_items.data(), sizeof(Item) * L.v0b_items.size());
  if (e == hipSuccess) e = up(L.off_mx_items, L.mx_items.data(), sizeof(Item) * L.mx_items.size());
  if (e == hipSuccess) e = up(L.off_big_items, L.big_items.data(), sizeof(Item) * L.big_items.size());
  if (e == hipSuccess) e = up(L.off_big_apply, L.big_apply.data(), sizeof(Item) * L.big_apply.size());
  if (e == hipSuccess) e = up(L.off_big_seg, L.big_seg.data(), sizeof(Item) * L.big_seg.size());
  if (e == hipSuccess) e = up(L.off_big_list, L.big_list.data(), sizeof(int) * L.big_list.size());
  if (e == hipSuccess) e = up(L.off_ns_mats, L.ns_mats.data(), sizeof(NsMat) * L.ns_mats.size());
  if (e == hipSuccess) e = up(L.off_ns_gram, L.ns_gram.data(), sizeof(NsItem) * L.ns_gram.size());
  if (e == hipSuccess) e = up(L.off_ns_poly, L.ns_poly.data(), sizeof(NsItem) * L.ns_poly.size());
  if (e == hipSuccess) e = up(L.off_ns_upd, L.ns_upd.data(), sizeof(NsItem) * L.ns_upd.size());
  if (e == hipSuccess) e = up(L.off_ns_upd4, L.ns_upd4.data(), sizeof(NsItem) * L.ns_upd4.size());
  if (e == hipSuccess) e = up(L.off_ns_split, L.ns_split.data(), sizeof(int) * L.ns_split.size());
  if (e == hipSuccess && kind == PYLO_KIND_CELO2) e = up(L.off_ns_xalt, L.ns_xalt.data(), sizeof(long long) * L.ns_xalt.size());
  if (e == hipSuccess) e = up(L.off_nsb_mats, L.nsb_mats.data(), sizeof(NsHfMat) * L.nsb_mats.size());
  if (e == hipSuccess) e = up(L.off_nsb_split_items, L.nsb_split_items.data(), sizeof(NsTileItem) * L.nsb_split_items.size());
  if (e == hipSuccess) e = up(L.off_ns_list, L.ns_list.data(), sizeof(int) * L.ns_list.size());
  if (e == hipSuccess) e = up(L.off_ns_flag_items, L.ns_flag_items.data(), sizeof(Item) * L.ns_flag_items.size());
  if (e == hipSuccess) e = up(L.off_slice_mats, L.slice_mats.data(), sizeof(SliceMat) * L.slice_mats.size());
  for (int k = 0; k < kSliceLaneSets; ++k)
    if (e == hipSuccess) e = up(L.off_slice_items_l[k], L.slice_items_l[k].data(), sizeof(Item) * L.slice_items_l[k].size());
  if (e == hipSuccess) e = up(L.off_slice_items_w, L.slice_items_w.data(), sizeof(Item) * L.slice_items_w.size());
  if (e == hipSuccess) e = up(L.off_slice_items_b, L.slice_items_b.data(), sizeof(Item) * L.slice_items_b.size());
  if (e == hipSuccess) e = up(L.off_sm_mats, L.sm_mats.data(), sizeof(NsSmall) * L.sm_mats.size());
  for (int k = 0; k < kNsSmallClasses; ++k)
    if (e == hipSuccess) e = up(L.off_sm_items[k], L.sm_items[k].data(), sizeof(NsSmallItem) * L.sm_items[k].size());
  // the meeting counters start at zero; every launch leaves them there
  if (e == hipSuccess && L.sm_sync > 0) e = hipMemsetAsync(P->ws + L.off_sm_sync, 0, sizeof(int) * (size_t)L.sm_sync, s);
  // the padding of the operand planes is read by the products and written by nobody: zero, once
  if (e == hipSuccess && L.nsb_plane_elems > 0)
    e = hipMemsetAsync(P->ws + L.off_ns_pw, 0, sizeof(hbits) * (size_t)L.nsb_plane_elems, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  for (int i = 0; i < kStageSlots && e == hipSuccess; ++i) {
    e = hipHostMalloc(reinterpret_cast<void**>(&P->stage[i]), (sizeof(PyloTensorArgs) * n_tensors + 15) / 16 * 16,
                      hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->ev[i], hipEventDisableTiming);
  }
  if (e == hipSuccess && kind == PYLO_KIND_VELO) {
    e = hipHostMalloc(reinterpret_cast<void**>(&P->stale_host), 64, hipHostMallocMapped);
    if (e == hipSuccess) P->stale_host[0] = P->stale_host[1] = 0;
    if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&P->stale_dev), P->stale_host, 0);
    if (e == hipSuccess) {   // its address, where the kernels look for it (behind the counters of `sync`)
      const long long addr = reinterpret_cast<long long>(P->stale_dev);
      e = hipMemcpyAsync(P->ws + L.off_sync + sizeof(int) * (size_t)((2 * n_tensors + 3) & ~3), &addr, sizeof(addr),
                         hipMemcpyHostToDevice, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
    }
  }
  if (e == hipSuccess && kind == PYLO_KIND_VELO && P->L.fused) {
    e = hipStreamCreateWithFlags(&P->side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->ev_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->ev_join, hipEventDisableTiming);
  }
  size_t ns_streams = 0;
  for (const NsBatch& bt : L.ns_batches) ns_streams = std::max<size_t>(ns_streams, bt.n_groups);
  for (size_t g = 0; ns_streams > 1 && g < std::max<size_t>(ns_streams, 3) && e == hipSuccess; ++g) {
    if (g == 0) e = hipEventCreateWithFlags(&P->ns_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&P->ns_side[g], hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->ns_join[g], hipEventDisableTiming);
  }
  bool plan_has_slices = !L.slice_items_w.empty() || !L.slice_items_b.empty();
  for (const auto& v : L.slice_items_l) plan_has_slices = plan_has_slices || !v.empty();
  plan_has_slices = plan_has_slices || !L.sm_mats.empty();   // the small matrices' launches ride on the same stream
  if (e == hipSuccess && plan_has_slices && ns_streams >= 1 && ns_streams <= 3) {   // groups + this one <= 4 queues
    e = hipStreamCreateWithFlags(&P->slice_side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->slice_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->slice_join, hipEventDisableTiming);
  }
  // the small matrices' classes on two streams (enqueue_small), with the caller's and slice_side three
  const bool small_a = !L.sm_items[0].empty() || !L.sm_items[3].empty(), small_b = !L.sm_items[1].empty() || !L.sm_items[2].empty();
  if (e == hipSuccess && small_a && small_b && ns_streams <= 1) {
    e = hipStreamCreateWithFlags(&P->small_side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->small_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&P->small_join, hipEventDisableTiming);
  }
  if (e != hipSuccess) {
    pylo_mi355_plan_destroy(P);
    return fail(std::string("plan_create: ") + hipGetErrorString(e));
  }
  *plan_out = P;
  return 0;
}

int pylo_mi355_plan_destroy(PyloPlan* P) {
  if (!P) return 0;
  for (hipEvent_t e : P->tev) (void)hipEventDestroy(e);
  if (P->ev_fork) (void)hipEventDestroy(P->ev_fork);
  if (P->ev_join) (void)hipEventDestroy(P->ev_join);
  if (P->side) (void)hipStreamDestroy(P->side);
  if (P->stale_host) (void)hipHostFree(P->stale_host);
  if (P->ns_fork) (void)hipEventDestroy(P->ns_fork);
  if (P->slice_fork) (void)hipEventDestroy(P->slice_fork);
  if (P->slice_join) (void)hipEventDestroy(P->slice_join);
  if (P->slice_side) (void)hipStreamDestroy(P->slice_side);
  if (P->small_side) (void)hipStreamDestroy(P->small_side);
  if (P->small_fork) (void)hipEventDestroy(P->small_fork);
  if (P->small_join) (void)hipEventDestroy(P->small_join);
  for (int g = 0; g < 4; ++g) {
    if (P->ns_join[g]) (void)hipEventDestroy(P->ns_join[g]);
    if (P->ns_side[g]) (void)hipStreamDestroy(P->ns_side[g]);
  }
  for (int i = 0; i < kStageSlots; ++i) {
    if (P->ev[i]) (void)hipEventDestroy(P->ev[i]);
    if (P->stage[i]) (void)hipHostFree(P->stage[i]);
  }
  delete P;
  return 0;
}

static const char* kCelo2Launches[] = {"k_p0(sums)", "k_gnorm", "k_p0(exact)", "k_v0a", "k_v0b",
                                       "k_celo2_stats", "k_celo2_fold", "k_celo2_apply"};
static const char* kCelo2FusedLaunches[] = {"k_p0(sums)", "k_gnorm", "k_p0(exact)", "k_v0a", "k_v0b",
                                            "k_celo2_elem", "k_celo2_slices"};
static const char* kVeloLaunches[] = {"k_p0(sums)", "k_p0_nd", "k_v0a", "k_v0b", "k_velo_stats",
                                      "k_lo_reduce", "k_velo_mix", "k_velo_gates", "k_velo_heads", "k_terms",
                                      "k_velo_apply"};

static const char* kVeloFusedLaunches[] = {"k_p0(sums) | LSTM", "k_v0a", "k_v0b", "k_terms", "k_velo_elem"};
static const char* kAdafacLaunches[] = {"k_p0(sums)", "k_p0_nd", "k_adafac_v0a", "k_v0b", "k_adafac_stats",
                                        "k_adafac_fold", "k_adafac_apply"};

int pylo_mi355_plan_num_launches(const PyloPlan* P) {
  if (!P) return -1;
  const int n_celo2 = !P->L.fused ? (int)(sizeof(kCelo2Launches) / sizeof(kCelo2Launches[0]))
                                            : (int)(sizeof(kCelo2FusedLaunches) / sizeof(kCelo2FusedLaunches[0]));
  const int n_velo = !P->L.fused ? (int)(sizeof(kVeloLaunches) / sizeof(kVeloLaunches[0]))
                                           : (int)(sizeof(kVeloFusedLaunches) / sizeof(kVeloFusedLaunches[0]));
  constexpr int n_adafac = sizeof(kAdafacLaunches) / sizeof(kAdafacLaunches[0]);
  return P->kind == PYLO_KIND_CELO2 ? n_celo2 : P->kind == PYLO_KIND_VELO ? n_velo : P->kind == PYLO_KIND_ADAFAC ? n_adafac : -1;
}

const char* pylo_mi355_plan_launch_name(const PyloPlan* P, int launch) {
  if (!P || launch < 0 || launch >= pylo_mi355_plan_num_launches(P)) return "";
  return P->kind == PYLO_KIND_CELO2 ? (!P->L.fused ? kCelo2Launches[launch] : kCelo2FusedLaunches[launch])
         : P->kind == PYLO_KIND_VELO ? (!P->L.fused ? kVeloLaunches[launch] : kVeloFusedLaunches[launch])
                                     : kAdafacLaunches[launch];
}

int pylo_mi355_plan_timing_begin(PyloPlan* P, int max_steps) {
  if (!P || max_steps <= 0) return fail("timing_begin: bad argument");
  const int per = pylo_mi355_plan_num_launches(P) + 1;
  for (hipEvent_t e : P->tev) (void)hipEventDestroy(e);
  P->tev.assign((size_t)per * max_steps, nullptr);
  for (auto& e : P->tev) HIP_TRY(hipEventCreate(&e));
  P->t_steps_max = max_steps;
  P->t_steps = 0;
  P->t_per_step = per;
  P->timing = true;
  return 0;
}

int pylo_mi355_plan_timing_end(PyloPlan* P, float* ms_out, int capacity, int* steps_out) {
  if (!P || !ms_out || !steps_out) return fail("timing_end: bad argument");
  P->timing = false;
  const int nl = P->t_per_step - 1;
  const int steps = P->t_steps;
  if (capacity < steps * nl) return fail("timing_end: output too small");
  if (steps > 0) HIP_TRY(hipEventSynchronize(P->tev[(size_t)steps * P->t_per_step - 1]));
  for (int s = 0; s < steps; ++s)
    for (int k = 0; k < nl; ++k) {
      float ms = 0.0f;
      HIP_TRY(hipEventElapsedTime(&ms, P->tev[(size_t)s * P->t_per_step + k], P->tev[(size_t)s * P->t_per_step + k + 1]));
      ms_out[s * nl + k] = ms;
    }
  *steps_out = steps;
  return 0;
}

int pylo_mi355_plan_arg_table(PyloPlan* P, int slot, PyloTensorArgs** table_out) {
  if (!P || !table_out || slot < 0 || slot >= kStageSlots) return fail("plan_arg_table: bad argument");
  // a staged copy out of this slot may still be pending on the device
  if (P->ev_used[slot]) HIP_TRY(hipEventSynchronize(P->ev[slot]));
  P->handed[slot] = true;
  *table_out = P->stage[slot];
  return 0;
}

int pylo_mi355_plan_device_steps(PyloPlan* P, const PyloDeviceSteps* steps) {
  if (!P) return fail("plan_device_steps: null plan");
  if (!steps || !steps->counters) {
    P->dsteps = PyloDeviceSteps{nullptr, 0.0, 0.0, 1.0};
    return 0;
  }
  if (reinterpret_cast<uintptr_t>(steps->counters) % 4 != 0) return fail("plan_device_steps: misaligned counters");
  if (P->kind == PYLO_KIND_VELO && !(steps->num_steps > 0.0)) return fail("plan_device_steps: num_steps must be positive");
  P->dsteps = *steps;
  return 0;
}

int pylo_mi355_plan_factored_dims(const PyloPlan* P, int tensor, int* dc, int* dr) {
  if (!P || tensor < 0 || tensor >= P->T || !dc || !dr) return fail("factored_dims: bad argument");
  *dc = P->L.dc[tensor];
  *dr = P->L.dr[tensor];
  return 0;
}

}  // extern "C"

namespace {

// Copies the per-step argument table to the device through a ring of pinned slots; skipped when
// the table is byte-identical to the one already resident.
// The per-step argument table goes from pinned host memory to the workspace with a small kernel on
// the launch stream: an async memcpy on the same stream costs a hand-over to the copy engine and back
// (about 0.1 ms of idle GPU between two steps), a kernel reading 10 KB over the host link does not.
__global__ __launch_bounds__(256) void k_copy_args(const uint4* __restrict__ src, uint4* __restrict__ dst, int n16) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n16; i += gridDim.x * 256) dst[i] = src[i];
}

// `dst_off`: where the table goes, the records the kernels read (off_dyn) or, for a step of a plan with
// tensors of other storage types, the caller's records that k_stage_args copies from (off_dyn_user).
int upload_args(PyloPlan* P, const PyloTensorArgs* args, hipStream_t s, size_t dst_off) {
  const size_t bytes = sizeof(PyloTensorArgs) * P->T;
  static_assert(sizeof(PyloTensorArgs) % 8 == 0, "argument records are copied in 16-byte pieces");
  const int n16 = (int)((bytes + 15) / 16);
  const dim3 grid(std::min(64, (n16 + 255) / 256));
  for (int j = 0; j < kStageSlots; ++j) {
    if (args != P->stage[j]) continue;
    // one of the plan's own pinned tables: read in place when the kernel runs (a graph replay sees the
    // table as it is then); nothing on the host side depends on earlier calls
    void* src_dev = nullptr;
    HIP_TRY(hipHostGetDevicePointer(&src_dev, P->stage[j], 0));
    hipLaunchKernelGGL(k_copy_args, grid, dim3(256), 0, s, static_cast<const uint4*>(src_dev),
                       reinterpret_cast<uint4*>(P->ws + dst_off), n16);
    P->have_last = false;
    return 0;
  }
  if (P->have_last && P->last_dst == dst_off && std::memcmp(P->last.data(), args, bytes) == 0) return 0;
  int i = -1;
  for (int k = 0; k < kStageSlots && i < 0; ++k) {
    const int c = (P->slot + k) % kStageSlots;
    if (!P->handed[c]) i = c;
  }
  if (i < 0) return fail("step: every argument table of the plan has been handed out; call with one of them");
  P->slot = (i + 1) % kStageSlots;
  if (P->ev_used[i]) HIP_TRY(hipEventSynchronize(P->ev[i]));
  std::memcpy(P->stage[i], args, bytes);
  void* src_dev = nullptr;
  HIP_TRY(hipHostGetDevicePointer(&src_dev, P->stage[i], 0));
  hipLaunchKernelGGL(k_copy_args, grid, dim3(256), 0, s,
                     static_cast<const uint4*>(src_dev), reinterpret_cast<uint4*>(P->ws + dst_off), n16);
  HIP_TRY(hipEventRecord(P->ev[i], s));
  P->ev_used[i] = true;
  P->last.assign(args, args + P->T);
  P->last_dst = dst_off;
  P->have_last = true;
  return 0;
}

// Step of a plan with tagged tensors: the records the kernels read are the caller's with grad / param of the
// tagged tensors redirected into the staging, which is filled here.  `what`: 1 gradient, 2 parameter, 3 both.
void stage_in(PyloPlan* P, hipStream_t s, int what) {
  const Layout& L = P->L;
  if (!L.typed) return;
  hipLaunchKernelGGL(k_stage_args, dim3((P->T + 255) / 256), dim3(256), 0, s, P->T, P->at<TDesc>(L.off_descs),
                     P->at<PyloTensorArgs>(L.off_dyn_user), P->at<PyloTensorArgs>(L.off_dyn),
                     P->at<StageOfs>(L.off_stage_ofs), P->at<float>(L.off_stage));
  if (L.cast_items.empty()) return;   // every tensor is read in place
  hipLaunchKernelGGL(k_cast_in, dim3((unsigned)L.cast_items.size()), dim3(kThreads), 0, s, P->at<TDesc>(L.off_descs),
                     P->at<PyloTensorArgs>(L.off_dyn_user), P->at<Item>(L.off_cast_items),
                     P->at<StageOfs>(L.off_stage_ofs), P->at<float>(L.off_stage), what);
}

void stage_out(PyloPlan* P, hipStream_t s, int flat_only) {
  const Layout& L = P->L;
  if (L.cast_items.empty()) return;
  hipLaunchKernelGGL(k_cast_out, dim3((unsigned)L.cast_items.size()), dim3(kThreads), 0, s, P->at<TDesc>(L.off_descs),
                     P->at<PyloTensorArgs>(L.off_dyn_user), P->at<Item>(L.off_cast_items),
                     P->at<StageOfs>(L.off_stage_ofs), P->at<float>(L.off_stage), flat_only);
}

// Step counters kept on the device: advances them and writes what the host otherwise supplies per
// step into the device copy of the argument table (bias corrections, AdafacLO's counter) or into
// the VeLO time-feature buffer.  One thread per tensor (VeLO: per group).
__global__ __launch_bounds__(256) void k_advance_steps(int kind, int T, const TDesc* __restrict__ descs,
                                                       PyloTensorArgs* __restrict__ dyn, PyloDeviceSteps ds,
                                                       float* __restrict__ frac_out) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (kind == PYLO_KIND_VELO) {
    if (t >= PYLO_MAX_GROUPS) return;
    const float ts[9] = {0.03f, 0.1f, 0.2f, 0.4f, 0.6f, 0.8f, 0.9f, 1.0f, 1.1f};
    const int c = ds.counters[t];
    const float x = (float)((double)c / ds.num_steps);
#pragma unroll
    for (int q = 0; q < 9; ++q) frac_out[t * 9 + q] = tanhf((x - ts[q]) * 10.0f);
    ds.counters[t] = c + 1;
    return;
  }
  if (t >= T) return;
  const bool has_grad = dyn[t].grad != nullptr;
  if (kind == PYLO_KIND_ADAFAC) {
    if (!has_grad) return;
    const int c = ds.counters[t];
    dyn[t].bc1 = (float)c;
    ds.counters[t] = c + 1;
    return;
  }
  // CELO2 kind: a per-parameter counter (independent AdamW moments) sits a step out with its tensor,
  // the others count the calls like the reference's per-group counter
  if (descs[t].adam_indep && !has_grad) return;
  const int c = ds.counters[t] + 1;
  ds.counters[t] = c;
  if (descs[t].mode != kModeFlat) return;
  dyn[t].bc1 = (float)(1.0 - pow(ds.beta1, (double)c));
  dyn[t].bc2 = (float)(1.0 - pow(ds.beta2, (double)c));
}

void advance_steps(PyloPlan* P, hipStream_t s) {
  if (!P->dsteps.counters) return;
  const int n = P->kind == PYLO_KIND_VELO ? PYLO_MAX_GROUPS : P->T;
  hipLaunchKernelGGL(k_advance_steps, dim3((n + 255) / 256), dim3(256), 0, s, P->kind, P->T,
                     P->at<TDesc>(P->L.off_descs), P->at<PyloTensorArgs>(P->L.off_dyn), P->dsteps,
                     P->kind == PYLO_KIND_VELO ? P->at<float>(P->L.off_frac) : nullptr);
}

int check_args(const PyloPlan* P, const PyloTensorArgs* args, bool need_all_grads) {
  for (int t = 0; t < P->T; ++t) {
    const TDesc& d = P->L.descs[t];
    const PyloTensorArgs& a = args[t];
    const std::string at = " at tensor " + std::to_string(t);
    if (a.grad == nullptr) {
      // an empty tensor has no gradient buffer to point to; its LSTM row sees zero statistics
      if (need_all_grads && d.n > 0) return fail("step: every tensor needs a gradient" + at);
      continue;
    }
    if (d.n == 0) continue;
    if (!a.param || !a.mom || !a.rms) return fail("step: null param/mom/rms pointer" + at);
    const bool factored = d.mode == kModeFac2D || d.mode == kModeFacND;
    if (factored && (!a.fac_r || !a.fac_c)) return fail("step: null fac_r/fac_c pointer" + at);
    if ((factored || d.mode == kModeVec) && P->kind == PYLO_KIND_CELO2 && !a.step_out)
      return fail("step: null step_out pointer" + at);
    if (d.mode == kModeVec && !a.fac_v) return fail("step: null fac_v pointer" + at);
    if (a.group < 0 || a.group >= PYLO_MAX_GROUPS) return fail("step: group index out of range" + at);
    const uintptr_t m = reinterpret_cast<uintptr_t>(a.grad) | reinterpret_cast<uintptr_t>(a.param) |
                        reinterpret_cast<uintptr_t>(a.mom) | reinterpret_cast<uintptr_t>(a.rms) |
                        reinterpret_cast<uintptr_t>(a.fac_r) | reinterpret_cast<uintptr_t>(a.fac_c) |
                        reinterpret_cast<uintptr_t>(a.fac_v) | reinterpret_cast<uintptr_t>(a.step_out);
    if (m % (d.vec == 4 ? 16 : 4) != 0) return fail("step: misaligned pointer (16 bytes needed)" + at);
    const uintptr_t gp = reinterpret_cast<uintptr_t>(a.grad) | reinterpret_cast<uintptr_t>(a.param);
    if (d.store != kStoreF32 && gp % 16 != 0)
      return fail("step: grad / param of a tensor with a storage type tag must be 16-byte aligned" + at);
  }
  return 0;
}

// The sums of g^2 of a globally clipped 2-D tensor are taken on the raw gradient and scaled afterwards;
// that is exact unless some scaled element lies beyond the tensor's clamp, in which case a second
// pass redoes them (k_p0, pass 1).  The scaled gradient is bounded by the global norm times the scale,
// i.e. by clip_norm, so with clip_norm below clip_val (1.0 against 1000 by default) the second pass can
// never be needed and is not launched.  Tensors whose NaNs are replaced always keep it.
bool exact_pass_possible(const PyloPlan* P, const PyloTensorArgs* args) {
  for (int t = 0; t < P->T; ++t) {
    const PyloTensorArgs& a = args[t];
    if (a.grad == nullptr || !(a.clip_norm > 0.0f)) continue;
    if (P->L.descs[t].nan0) return true;
    if (a.clip_val > 0.0f && !(a.clip_norm <= 0.99f * a.clip_val)) return true;
  }
  return false;
}

struct Marks {  // per-launch HIP events when timing is on
  PyloPlan* P;
  hipStream_t s;
  hipEvent_t* ev;
  int mark = 0;
  Marks(PyloPlan* P_, hipStream_t s_) : P(P_), s(s_) {
    const bool timed = P->timing && P->t_steps < P->t_steps_max;
    ev = timed ? &P->tev[(size_t)P->t_steps * P->t_per_step] : nullptr;
  }
  hipError_t operator()(bool skip = false) { return ev && !skip ? hipEventRecord(ev[mark++], s) : hipSuccess; }
  void done() { if (ev) P->t_steps++; }
};

}  // namespace

// The instantiation <TYPED, SPLIT> of a kernel, from all four of them.
template <class F>
F variant(bool typed, bool split, F plain, F split_only, F typed_only, F both) {
  return typed ? (split ? both : typed_only) : (split ? split_only : plain);
}
inline auto p0_kernel(bool typed, bool split) {
  return variant(typed, split, k_p0<false, false>, k_p0<false, true>, k_p0<true, false>, k_p0<true, true>);
}
inline auto norm_p0_kernel(bool typed, bool split) {
  return variant(typed, split, k_gnorm_p0<false, false>, k_gnorm_p0<false, true>, k_gnorm_p0<true, false>, k_gnorm_p0<true, true>);
}

extern "C" int pylo_mi355_celo2_step(PyloPlan* P, const PyloTensorArgs* args, const PyloDecays* decays,
                                     const float* mlp, void* stream) {
  if (!P || !args || !decays || !mlp) return fail("celo2_step: null argument");
  if (P->kind != PYLO_KIND_CELO2) return fail("celo2_step: plan is not a CELO2 plan");
  if (int rc = check_args(P, args, false)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (int rc = upload_args(P, args, s, P->L.off_dyn_user)) return rc;
  stage_in(P, s, 3);
  advance_steps(P, s);
  const Layout& L = P->L;
  const TDesc* descs = P->at<TDesc>(L.off_descs);
  const PyloTensorArgs* dyn = P->at<PyloTensorArgs>(L.off_dyn);
  const Item* p0_items = P->at<Item>(L.off_p0_items);
  const Item* el_items = P->at<Item>(L.off_el_items);
  const Item* v0a_items = P->at<Item>(L.off_v0a_items);
  const Item* v0b_items = P->at<Item>(L.off_v0b_items);
  const Item* nd_items = P->at<Item>(L.off_nd_items);
  const Item* sl_items = P->at<Item>(L.off_sl_items);
  const int n_nd = (int)L.nd_items.size(), n_sl = (int)L.sl_items.size();
  const int* fac_list = P->at<int>(L.off_fac_list);
  float* part = P->at<float>(L.off_part);
  double* gsq = P->at<double>(L.off_gsq);
  int* flag = P->at<int>(L.off_flag);
  Globals* gl = P->at<Globals>(L.off_globals);
  float* fac_tab = P->at<float>(L.off_fac);
  float* term_tab = P->at<float>(L.off_term);
  double* v0part = P->at<double>(L.off_v0part);
  BScale* bscale = P->at<BScale>(L.off_bscale);
  double* stats = P->at<double>(L.off_stats);
  float* wfold = P->at<float>(L.off_wfold);
  float* chan_ms = P->at<float>(L.off_chan_ms);
  const int n_p0 = (int)L.p0_items.size(), n_el = (int)L.el_items.size(), n_fac = (int)L.fac_list.size();
  const int n_v0a = (int)L.v0a_items.size(), n_v0b = (int)L.v0b_items.size();
  const PyloDecays dec = *decays;
  const bool in_place = L.in_place;   // tensors of 16-bit storage without staging (the matrix pipe's walks only)
  Marks mark(P, s);

  const bool exact_pass = exact_pass_possible(P, args);
  // Where no tensor is clipped by the global norm nobody reads it: only the matrices' sums are taken, and those of tensors with
  // more dims, which wait for its scale otherwise, in the same launch.  (Records that are read when the kernels run, as
  // under capture, may ask for it later.)  CELO2 on ResNet-50, both launches: 124 us, now 54 in one.
  const bool clips = std::any_of(args, args + P->T, [](const PyloTensorArgs& a) { return a.grad != nullptr && a.clip_norm > 0.0f; }) ||
                     std::find(P->stage, P->stage + kStageSlots, args) != P->stage + kStageSlots;
  const int n_tail = clips ? 0 : n_nd;
  HIP_TRY(mark());
  if (n_p0 + n_tail > 0)
    hipLaunchKernelGGL(p0_kernel(in_place, L.split), dim3(n_p0 + n_tail), dim3(kThreads), 0, s, descs, dyn, p0_items, part, gsq, flag,
                       gl, clips ? 0 : 2, nd_items, n_p0);
  HIP_TRY(mark());
  const NormArgs na{gsq, flag, n_p0, exact_pass ? 1 : 0, P->at<int>(L.off_sync), 2 * P->T};
  const bool few = n_p0 > 0 && n_p0 <= kNormBlocks, norm_p0 = few && exact_pass;
  const bool norm_v0a = few && !exact_pass && n_v0a > 0 && !(n_nd > 0 && clips);
  if (!norm_p0 && !norm_v0a) hipLaunchKernelGGL(k_gnorm, dim3(1), dim3(kThreads), 0, s, na, gl);
  HIP_TRY(mark());
  if (norm_p0)
    hipLaunchKernelGGL(norm_p0_kernel(in_place, L.split), dim3(n_p0), dim3(kThreads), 0, s, descs, dyn, p0_items, part, na, gl);
  else if (n_p0 > 0 && exact_pass)
    hipLaunchKernelGGL(p0_kernel(in_place, L.split), dim3(n_p0), dim3(kThreads), 0, s, descs, dyn, p0_items, part, gsq, flag, gl, 1,
                       (const Item*)nullptr, n_p0);
  if (n_nd > 0 && clips) hipLaunchKernelGGL(k_p0_nd, dim3(n_nd), dim3(kThreads), 0, s, descs, dyn, nd_items, part, gl);
  HIP_TRY(mark());
  if (norm_v0a)
    hipLaunchKernelGGL(k_gnorm_v0a, dim3(n_v0a), dim3(kThreads), 0, s, descs, dyn, v0a_items, part, na, gl, dec, v0part);
  else if (n_v0a > 0)
    hipLaunchKernelGGL(k_v0a, dim3(n_v0a), dim3(kV0aThreads), 0, s, descs, dyn, v0a_items, part, gl, dec, v0part);
  HIP_TRY(mark());
  const auto v0b = L.slice_runs ? k_v0b<8, true> : k_v0b<8>;
  if (n_v0b > 0)
    hipLaunchKernelGGL(v0b, dim3(n_v0b), dim3(kThreads), 0, s, descs, dyn, v0b_items, v0part, 1e-9f, mlp,
                       mlp + 240, 0, fac_tab, term_tab, bscale);
  HIP_TRY(mark());
  auto apply_items = [&](const Item* items, int n) {   // the apply pass as a launch of its own
    const auto apply = in_place                ? (L.split ? k_celo2_apply<true, true, true> : k_celo2_apply<true, true, false>)
                       : P->mlp_on_matrix_pipe ? (L.split ? k_celo2_apply<true, false, true> : k_celo2_apply<true, false, false>)
                                               : (L.split ? k_celo2_apply<false, false, true> : k_celo2_apply<false, false, false>);
    hipLaunchKernelGGL(apply, dim3(n), dim3(kThreads), 0, s, descs, dyn, items, fac_tab, term_tab, gl, dec, wfold);
  };
  const auto stats_pass = variant(in_place, L.split, k_celo2_stats<false, false>, k_celo2_stats<false, true>,
                                  k_celo2_stats<true, false>, k_celo2_stats<true, true>);
  // statistics and folded weights of n_fac tensors as launches of their own
  auto stats_items = [&](const Item* items, int n, const Item* seg, int n_seg, const int* list, int n_fac) {
    double* seg_tot = P->at<double>(L.off_segtot);
    if (n > 0) hipLaunchKernelGGL(stats_pass, dim3(n), dim3(kThreads), 0, s, descs, dyn, items, fac_tab, gl, dec, stats);
    HIP_TRY(mark(L.fused));
    if (n_seg > 0) hipLaunchKernelGGL(k_stat_segsum<kStatW>, dim3(n_seg), dim3(kThreads), 0, s, descs, seg, stats, seg_tot);
    if (n_fac > 0)
      hipLaunchKernelGGL(k_celo2_fold, dim3(n_fac), dim3(kFoldThreads), 0, s, descs, dyn, list, stats, seg_tot, mlp, wfold, chan_ms);
    HIP_TRY(mark(L.fused));
    return 0;
  };
  const int n_mx = (int)L.mx_items.size(), n_big = (int)L.big_items.size();
  if (L.fused) {
    if (n_big > 0)
      if (int rc = stats_items(P->at<Item>(L.off_big_items), n_big, P->at<Item>(L.off_big_seg), (int)L.big_seg.size(),
                               P->at<int>(L.off_big_list), (int)L.big_list.size())) return rc;
    const Item* mx_items = P->at<Item>(L.off_mx_items);
    int* sync = P->at<int>(L.off_sync);
    const auto elem = in_place              ? (L.split ? k_celo2_elem<true, true, true> : k_celo2_elem<true, false, true>)
                      : P->mlp_on_matrix_pipe ? (L.split ? k_celo2_elem<true, true> : k_celo2_elem<true, false>)
                                              : (L.split ? k_celo2_elem<false, true> : k_celo2_elem<false, false>);
    if (n_mx > 0)
      hipLaunchKernelGGL(elem, dim3(n_mx), dim3(kThreads), 0, s, descs, dyn, mx_items, fac_tab, term_tab, gl, dec, mlp,
                         wfold, chan_ms, stats, sync, P->T);
    if (n_big > 0) apply_items(P->at<Item>(L.off_big_apply), n_big);
    HIP_TRY(mark());
  } else {
    if (int rc = stats_items(el_items, n_el, P->at<Item>(L.off_seg_items), (int)L.seg_items.size(), fac_list, n_fac)) return rc;
    if (n_el > 0) apply_items(el_items, n_el);
  }
  if (n_sl > 0)
    hipLaunchKernelGGL(k_celo2_slices, dim3(n_sl), dim3(kThreads), 0, s, descs, dyn, sl_items, fac_tab, gl, dec, mlp);
  for (int c = 0, at = 0; c < kSliceWaveClasses; at += L.sl_wave_n[c], ++c) {
    if (L.sl_wave_n[c] == 0) continue;
    const auto wave = c == kSliceOne    ? k_celo2_slices_wave<1, true>
                      : c == kSliceNine ? k_celo2_slices_wave<9, true>
                      : c == kSliceAny  ? k_celo2_slices_wave<0, true>
                                        : k_celo2_slices_wave<0, false>;
    hipLaunchKernelGGL(wave, dim3((unsigned)L.sl_wave_n[c]), dim3(kThreads), 0, s, descs, dyn, P->at<Item>(L.off_sl_wave_items) + at,
                       fac_tab, term_tab, gl, dec, mlp);
  }
  HIP_TRY(mark());
  mark.done();
  stage_out(P, s, 1);   // only the AdamW tensors were updated
  HIP_TRY(hipGetLastError());
  return 0;
}

namespace {

// The split-fp16 product kernels take their LDS as dynamic shared memory; tiles of 256 columns need more than
// the 64 KB a kernel may have without asking.
int ns_hf_lds_once() {
  static std::mutex mu;
  static std::vector<int> done;   // devices on which the attribute has been set
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  for (int d : done)
    if (d == dev) return 0;
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsGram, 2, 2, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 2, 1)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsGram, 1, 1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(1, 1, 4)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsPoly, 2, 2, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 2, 1)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsPoly, 1, 1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(1, 1, 4)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsProd, 2, 2, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 2, 1)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsProd, 1, 1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(1, 1, 4)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsProdA, 2, 2, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 2, 1)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsProdA, 1, 1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(1, 1, 4)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsUpdate, 2, 2, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 2, 1)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsUpdate, 1, 1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(1, 1, 4)));
  HIP_TRY(hipFuncSetAttribute((const void*)k_ns_hf_gemm<kNsUpdate, 2, 4, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 4, 1)));
  done.push_back(dev);
  return 0;
}

int slice_lds_once() {
  static std::mutex mu;
  static std::vector<int> done;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  for (int d : done)
    if (d == dev) return 0;
  HIP_TRY(hipFuncSetAttribute((const void*)k_celo2_slice_finish<true>, hipFuncAttributeMaxDynamicSharedMemorySize, kSliceLdsBlock));
  done.push_back(dev);
  return 0;
}

__global__ __launch_bounds__(256) void k_ns_zero(u32x4* __restrict__ p, size_t n16) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256) p[i] = u32x4{0u, 0u, 0u, 0u};
}

// The iterations as runs that k_ns_thin takes from one Gram matrix each.  An entry of A (of the largest eigenvalue `top`) is off by 2^-52
// of that; an iteration multiplies what is off between two eigenvectors of eigenvalues a, b by at most `grow`, in the kernel's own
// order of operands (B = p(A A^T), T = A B^T, A <- T B^T), and B is off by B' times it.  A run ends before that is 2^-27 of B.
// With the usual coefficients grow is 23: runs of six.  (Errors at six and seven, eight, nine iterations of a run, 32 x 500 of ones: the last
// rounding, 4e-8, 2e-6, 5e-5.)
std::vector<int> thin_runs(double c0, double c1, double c2, int iters) {
  constexpr int N = 32;
  std::vector<int> runs{0};
  double top = 1.0, err = 0x1p-52;
  for (int i = 0; i < iters; ++i) {
    double b_max = 0.0, db_max = 0.0, next = 0.0, grow = 0.0;
    for (int k = 0; k <= N; ++k) {
      const double a = top * k / N, B = c0 + a * (c1 + a * c2);
      b_max = std::max(b_max, std::fabs(B));
      db_max = std::max(db_max, std::fabs(c1 + 2.0 * a * c2));
      next = std::max(next, a * B * B);
      for (int l = 0; l <= N; ++l) {
        const double b = top * l / N, Bb = c0 + b * (c1 + b * c2);
        double row = 0.0;   // what A'_ab takes from A_ab and A_ba
        for (int q = 0; q < 2; ++q) {
          const double x = 1 - q, y = q, p21 = c2 * (a * y + b * x) + c1 * y;
          row += std::fabs(a * B * p21 + (a * p21 + x * Bb) * Bb);
        }
        grow = std::max(grow, row);
      }
    }
    if (runs.back() > 0 && !(err * db_max <= 0x1p-27 * b_max)) {
      runs.push_back(0);
      err = 0x1p-52 * std::max(top, 1.0);
    }
    ++runs.back();
    top = next;
    err = err * grow + 0x1p-52 * std::max(top, 1.0);
  }
  return runs;
}

int small_lds_once() {
  static std::mutex mu;
  static std::vector<int> done;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  for (int d : done)
    if (d == dev) return 0;
  HIP_TRY(hipFuncSetAttribute((const void*)(k_ns_small<4, 2, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, SmLarge::kLds));
  HIP_TRY(hipFuncSetAttribute((const void*)(k_ns_small<2, 1, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, SmMid::kLds));
  done.push_back(dev);
  return 0;
}

// The launches of the small matrices (k_ns_small.h): one per class, largest first.  A class is a launch of chains that leaves
// most of the chip idle (three thousand matrices: 102, 120, 50 and 71 us one after the other, 345 us next to 235 of tiled products): where
// the groups of tiled products have left a queue, the middle two run on a stream of their own, which the caller joins.
int enqueue_small(PyloPlan* P, hipStream_t s, const TDesc* descs, const PyloTensorArgs* dyn, const float* coeffs, int ns_iters,
                  float ns_eps) {
  const Layout& L = P->L;
  if (int rc = small_lds_once()) return rc;
  const int orth = coeffs != nullptr && ns_iters > 0;
  NsSmallStep st{};
  if (orth) {
    const NsExps ex = ns_plane_exps(coeffs[0], coeffs[1], coeffs[2], ns_iters);
    const int q2 = ex.q[std::min<size_t>(2, ex.q.size() - 1)];
    st.x_s = pow2(ex.x); st.a_s = pow2(ex.a); st.b_s = pow2(ex.b); st.t_s = pow2(ex.t); st.q_s = pow2(q2);
    st.gram = pow2(-2 * ex.x); st.poly = pow2(-2 * ex.a);
    st.prod_t = pow2(-(ex.a + ex.b)); st.prod_a = pow2(-(ex.b + ex.t)); st.prod_q = pow2(-2 * ex.b);
    st.upd_b = pow2(-(ex.x + ex.b)); st.upd_q = pow2(-(ex.x + q2));
    st.c0 = coeffs[0]; st.c1 = coeffs[1]; st.c2 = coeffs[2]; st.eps = ns_eps;
    // pairs, or single iterations where the environment asks for those (plans made while it asks for other chains have no
    // small matrices)
    st.n_pairs = ns_iters / 2;
    const std::vector<int> chains = ns_chains(ns_iters);
    if (*std::max_element(chains.begin(), chains.end()) == 1) st.n_pairs = 0;
    st.n_chains = ns_iters - st.n_pairs;
  }
  if (P->small_side != nullptr) {
    HIP_TRY(hipEventRecord(P->small_fork, s));
    HIP_TRY(hipStreamWaitEvent(P->small_side, P->small_fork, 0));
  }
  auto launch = [&](auto kern, int cls, int threads, int lds, hipStream_t s) {
    if (!L.sm_items[cls].empty())
      hipLaunchKernelGGL(kern, dim3((unsigned)L.sm_items[cls].size()), dim3(threads), lds, s, P->at<NsSmall>(L.off_sm_mats),
                         P->at<NsSmallItem>(L.off_sm_items[cls]), descs, dyn, P->at<float>(L.off_sm_part),
                         P->at<double>(L.off_sm_sums), P->at<int>(L.off_sm_sync), st, orth,
                         L.sm_meets[cls] ? P->at<int>(L.off_sm_sync) + L.sm_ticket0 + cls : (int*)nullptr);
  };
  if (orth && (P->thin_c[0] != coeffs[0] || P->thin_c[1] != coeffs[1] || P->thin_c[2] != coeffs[2] || P->thin_iters != ns_iters)) {
    std::copy(coeffs, coeffs + 3, P->thin_c);
    P->thin_iters = ns_iters;
    P->thin_run = thin_runs(coeffs[0], coeffs[1], coeffs[2], ns_iters);
  }
  auto launch_thin = [&](auto kern, int cls, int lds, hipStream_t s) {
    if (L.sm_items[cls].empty()) return;
    const size_t n_runs = orth ? P->thin_run.size() : 1;
    for (size_t r = 0; r < n_runs; ++r) {
      const ThinStep thin{st.c0, st.c1, st.c2, ns_eps, orth ? P->thin_run[r] : 0, r == 0, r + 1 == n_runs};
      hipLaunchKernelGGL(kern, dim3((unsigned)L.sm_items[cls].size()), dim3(kThreads), lds, s, P->at<NsSmall>(L.off_sm_mats),
                         P->at<NsSmallItem>(L.off_sm_items[cls]), descs, dyn, P->at<float>(L.off_sm_part), P->at<int>(L.off_sm_sync),
                         thin, orth, L.sm_meets[cls] ? P->at<int>(L.off_sm_sync) + L.sm_ticket0 + cls : (int*)nullptr);
    }
  };
  const hipStream_t mid = P->small_side != nullptr ? P->small_side : s;
  launch(k_ns_small<4, 2, 1>, 3, SmLarge::kThr, SmLarge::kLds, s);
  launch(k_ns_small<2, 1, 2>, 2, SmMid::kThr, SmMid::kLds, mid);
  const bool runs = orth && P->thin_run.size() > 1;
  launch_thin(runs ? k_ns_thin<2, true> : k_ns_thin<2, false>, 1, ThinDims<2>::kLds, mid);
  launch_thin(runs ? k_ns_thin<1, true> : k_ns_thin<1, false>, 0, ThinDims<1>::kLds, s);
  if (P->small_side != nullptr) HIP_TRY(hipEventRecord(P->small_join, P->small_side));
  return 0;
}

// Newton-Schulz (ns_iters > 0, on the tensors flagged PYLO_ARG_ORTHOGONALIZE) and the finishing pass.
int finish_impl(PyloPlan* P, const PyloTensorArgs* args, const float* coeffs, int ns_iters, float ns_eps, void* stream,
                const char* who) {
  const std::string w(who);
  if (!P || P->kind != PYLO_KIND_CELO2) return fail(w + ": not an ELO-CELO2 plan");
  if (!args) return fail(w + ": null argument");
  const Layout& L = P->L;
  bool any_ns = false, any_slices = false, any_small = false;
  for (int t = 0; t < P->T; ++t) {
    const TDesc& d = L.descs[t];
    const PyloTensorArgs& a = args[t];
    if (a.grad == nullptr || d.mode == kModeFlat || d.n == 0) continue;
    const std::string at = " (tensor " + std::to_string(t) + ")";
    if (!a.param || !a.step_out) return fail(w + ": null param/step_out pointer" + at);
    const uintptr_t m = reinterpret_cast<uintptr_t>(a.param) | reinterpret_cast<uintptr_t>(a.step_out);
    if (d.mode == kModeFacND && L.slice_of_tensor[t] >= 0) {
      if (reinterpret_cast<uintptr_t>(a.step_out) % 4 != 0 || reinterpret_cast<uintptr_t>(a.param) % (d.store != 0 ? 2 : 4) != 0)
        return fail(w + ": misaligned pointer" + at);
      if (coeffs && (a.flags & PYLO_ARG_ORTHOGONALIZE) && L.slice_mats[L.slice_of_tensor[t]].no_orth)
        return fail(w + ": PYLO_ARG_ORTHOGONALIZE on a tensor whose shape carries PYLO_F_NO_ORTHOGONALIZE" + at);
      any_slices = true;
      continue;
    }
    const bool small = L.small_of_tensor[t] != 0;
    const bool vec = small ? L.small_of_tensor[t] == 2 : d.fin_units > 0 && L.fin_units[d.fin_unit0].vec;
    if (m % (vec ? 16 : 4) != 0) return fail(w + ": misaligned pointer" + at);   // the same whatever launch takes the tensor
    any_small = any_small || small;
    if (coeffs && ns_iters == 0 && (a.flags & PYLO_ARG_ORTHOGONALIZE))
      return fail(w + ": PYLO_ARG_ORTHOGONALIZE with ns_iters = 0 on a tensor that the tiled products orthogonalise "
                  "(the division by the norm alone is the caller's)" + at);
    if (ns_iters > 0 && (a.flags & PYLO_ARG_ORTHOGONALIZE)) {
      if (small) continue;
      if (L.ns_of_tensor[t] < 0) return fail(w + ": PYLO_ARG_ORTHOGONALIZE on a tensor the library cannot orthogonalise" + at);
      any_ns = true;
    }
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  // the caller's records as they are: the update kernel reads and writes the parameter in its storage type
  if (int rc = upload_args(P, args, s, L.off_dyn)) return rc;
  const TDesc* descs = P->at<TDesc>(L.off_descs);
  const PyloTensorArgs* dyn = P->at<PyloTensorArgs>(L.off_dyn);
  const Item* fin_items = P->at<Item>(L.off_fin_items);
  const FinUnit* units = P->at<FinUnit>(L.off_fin_units);
  double* fin_part = P->at<double>(L.off_finpart);
  float* fin_scale = P->at<float>(L.off_finscale);
  const int n_fin = (int)L.fin_items.size();
  // The per-slice launches touch only their own tensors: next to the matrices' chains of products they run on a stream
  // of their own (forked from and joined into the caller's like the groups').
  const bool slices_aside = (any_slices || any_small) && any_ns && L.ns_hf && P->slice_side != nullptr;
  if (slices_aside) {
    HIP_TRY(hipEventRecord(P->slice_fork, s));
    HIP_TRY(hipStreamWaitEvent(P->slice_side, P->slice_fork, 0));
  }
  if (any_small)
    if (int rc = enqueue_small(P, slices_aside ? P->slice_side : s, descs, dyn, coeffs, ns_iters, ns_eps)) return rc;
  if (any_slices) {
    // tensors with more than two dims: everything per slice, in LDS (k_slice_finish.h)
    if (int rc = slice_lds_once()) return rc;
    hipStream_t caller = s;
    hipStream_t s = slices_aside ? P->slice_side : caller;
    const SliceMat* smats = P->at<SliceMat>(L.off_slice_mats);
    const float c0 = coeffs ? coeffs[0] : 0.0f, c1 = coeffs ? coeffs[1] : 0.0f, c2 = coeffs ? coeffs[2] : 0.0f;
    const int orth_call = coeffs != nullptr;
    auto lanes = [&](auto kern, int set) {
      if (!L.slice_items_l[set].empty())
        hipLaunchKernelGGL(kern, dim3((unsigned)L.slice_items_l[set].size()), dim3(64), L.slice_lds_l[set], s, smats,
                           P->at<Item>(L.off_slice_items_l[set]), descs, dyn, orth_call, ns_iters, ns_eps, c0, c1, c2);
    };
    lanes(k_celo2_slice_finish_lane<1>, 0);
    lanes(k_celo2_slice_finish_lane<3>, 1);
    lanes(k_celo2_slice_finish_lane<5>, 2);
    lanes(k_celo2_slice_finish_lane<7>, 3);
    for (int set = 4; set < kSliceLaneSets; ++set) lanes(k_celo2_slice_finish_lane<0>, set);
    if (!L.slice_items_w.empty())
      hipLaunchKernelGGL(k_celo2_slice_finish<false>, dim3((unsigned)L.slice_items_w.size()), dim3(256), L.slice_lds_w, s,
                         smats, P->at<Item>(L.off_slice_items_w), descs, dyn, orth_call, ns_iters, ns_eps, c0, c1, c2);
    if (!L.slice_items_b.empty())
      hipLaunchKernelGGL(k_celo2_slice_finish<true>, dim3((unsigned)L.slice_items_b.size()), dim3(256), L.slice_lds_b, s,
                         smats, P->at<Item>(L.off_slice_items_b), descs, dyn, orth_call, ns_iters, ns_eps, c0, c1, c2);
  }
  if (any_small && P->small_side != nullptr) HIP_TRY(hipStreamWaitEvent(slices_aside ? P->slice_side : s, P->small_join, 0));
  if (slices_aside) HIP_TRY(hipEventRecord(P->slice_join, P->slice_side));
  if (n_fin == 0) {
    HIP_TRY(hipGetLastError());
    return 0;
  }
  // sum of squares, per-unit scale and update over a range of the finishing pass's blocks and units
  auto finish_range = [&](hipStream_t st, int fin0, int nf, int unit0, int nu, const long long* x_alt, const float* ws) {
    if (nf == 0) return;
    hipLaunchKernelGGL(k_celo2_sumsq, dim3(nf), dim3(kThreads), 0, st, units, dyn, fin_items + fin0, fin_part + fin0, x_alt, ws);
    hipLaunchKernelGGL(k_celo2_finscale, dim3(nu), dim3(kThreads), 0, st, units + unit0, dyn, fin_part, fin_scale + unit0);
    hipLaunchKernelGGL(k_celo2_update, dim3(nf), dim3(kThreads), 0, st, units, descs, dyn, fin_items + fin0, fin_scale, x_alt, ws);
  };
  if (!any_ns) {
    finish_range(s, 0, n_fin, 0, (int)L.fin_units.size(), nullptr, nullptr);
  } else if (L.ns_hf) {
    // The split-fp16 kernels.  Every group of matrices is a chain of its own from the norms of its raw steps to the
    // update of its parameters, on a stream of its own where there are several: the memory-bound ends of one chain run
    // under the matrix products of the others.
    const NsMat* mats = P->at<NsMat>(L.off_ns_mats);
    const NsItem* gram = P->at<NsItem>(L.off_ns_gram);
    const NsItem* poly = P->at<NsItem>(L.off_ns_poly);
    const NsItem* upd = P->at<NsItem>(L.off_ns_upd);
    const NsItem* upd4 = P->at<NsItem>(L.off_ns_upd4);
    const int* split = P->at<int>(L.off_ns_split);
    const int* list = P->at<int>(L.off_ns_list);
    float* scale = P->at<float>(L.off_ns_scale);
    float* ns_ws = P->at<float>(L.off_ns_ws);
    const NsHfMat* bmats = P->at<NsHfMat>(L.off_nsb_mats);
    const NsTileItem* sitems = P->at<NsTileItem>(L.off_nsb_split_items);
    hbits* pw = P->at<hbits>(L.off_ns_pw);
    if (int rc = ns_hf_lds_once()) return rc;
    finish_range(s, L.fin_rest0, L.n_fin_rest, L.unit_rest0, L.n_unit_rest, nullptr, nullptr);   // tensors of no group
    const bool several = L.ns_batches.size() > 1;
    const float c0 = coeffs[0], c1 = coeffs[1], c2 = coeffs[2];
    const std::vector<int> chains = ns_chains(ns_iters);
    const NsExps ex = ns_plane_exps(c0, c1, c2, ns_iters);
    // chain lengths chosen per matrix on the device: an odd iteration count of three or more, nothing given in the environment
    const bool adaptive = ns_adaptive() && ns_iters >= 3 && (ns_iters & 1);
    int* chain_flags = P->at<int>(L.off_ns_flags);
    float* chain_part = P->at<float>(L.off_ns_fpart);
    const Item* flag_items = P->at<Item>(L.off_ns_flag_items);
    const float chain_tau2 = (16.0f / 196.0f) * (16.0f / 196.0f);
    for (const NsBatch& bt : L.ns_batches) {
      // the planes' padding: zero from plan creation on when one batch has the memory to itself
      if (several) {
        const size_t n16 = (size_t)bt.plane_elems * sizeof(hbits) / 16;
        hipLaunchKernelGGL(k_ns_zero, dim3((unsigned)std::min<size_t>((n16 + 255) / 256, 1u << 16)), dim3(256), 0, s,
                           reinterpret_cast<u32x4*>(pw), n16);
      }
      const int n_groups = bt.n_groups;
      auto stream_of = [&](int g) { return n_groups == 1 ? s : P->ns_side[g]; };
      if (n_groups > 1) {
        HIP_TRY(hipEventRecord(P->ns_fork, s));
        for (int g = 0; g < n_groups; ++g) HIP_TRY(hipStreamWaitEvent(P->ns_side[g], P->ns_fork, 0));
      }
      for (int g = 0; g < n_groups; ++g) {
        // ||raw|| per matrix (the finishing pass's sums of squares, taken on the raw steps), then the planes
        const NsGroup& G = L.ns_groups[bt.group0 + g];
        hipStream_t sg = stream_of(g);
        if (G.n_fin > 0)
          hipLaunchKernelGGL(k_celo2_sumsq, dim3(G.n_fin), dim3(kThreads), 0, sg, units, dyn, fin_items + G.fin0,
                             fin_part + G.fin0, (const long long*)nullptr, (const float*)nullptr);
        if (G.n_list > 0)
          hipLaunchKernelGGL(k_ns_scale, dim3(G.n_list), dim3(256), 0, sg, mats, list + G.list0, G.n_list, units, fin_part,
                             ns_eps, scale);
        if (G.n_sitems > 0)
          hipLaunchKernelGGL(k_ns_hf_split, dim3((unsigned)G.n_sitems), dim3(256), 0, sg, bmats, sitems + G.sitem0, dyn,
                             (const float*)scale, pw, pow2(ex.x));
      }
      // The launch sequence of one group (every group runs the same one on its own tables), then its launches,
      // interleaved over the groups so that every stream is fed in turn.
      enum OpKind { kOpGram, kOpFlag, kOpPoly, kOpProd, kOpProdA, kOpUpdate };
      struct Op { OpKind kind; NsBufs b; int par, last; NsPick pick; };
      std::vector<Op> ops;
      const NsPick all{nullptr, kNsAll, 0, 0, 0.0f};
      int par = 0;   // which Xl buffer the next update reads
      // A is buffer A throughout; B' of the latest iteration in `bprev`, the product of all B' so far in `q`
      // (`nq` of them); eb[]: the exponent of the scale of the planes in each buffer
      int bprev = kNsBufB, q = kNsBufB, nq = 1;
      int eb[kNsBufs] = {};
      // the accumulators of a product of planes with exponents e1 and e2, and planes out with exponent ed
      auto bufs = [&](int s1, int s2, int d, int e1, int e2, int ed) {
        if (d >= 0) eb[d] = ed;
        return NsBufs{s1, s2, d < 0 ? 0 : d, pow2(-(e1 + e2)), pow2(ed)};
      };
      auto extend = [&](NsPick pk) {   // one more iteration into the chain: A <- B' A B', the next B', Q <- B' Q
        int free_buf[2], nf = 0;
        for (int b : {kNsBufB, kNsBufT, kNsBufC})
          if (b != bprev && b != q && nf < 2) free_buf[nf++] = b;
        const int t = free_buf[0];
        ops.push_back(Op{kOpProd, bufs(kNsBufA, bprev, t, ex.a, eb[bprev], ex.t), par, 0, pk});
        ops.push_back(Op{kOpProdA, bufs(bprev, t, kNsBufA, eb[bprev], ex.t, ex.a), par, 0, pk});
        ops.push_back(Op{kOpPoly, bufs(kNsBufA, kNsBufA, t, ex.a, ex.a, ex.b), par, 0, pk});
        const int qn = q == bprev ? free_buf[1] : bprev;   // (the old B' is done with)
        ++nq;
        ops.push_back(Op{kOpProd, bufs(t, q, qn, ex.b, eb[q], ex.q[std::min<size_t>(nq, ex.q.size() - 1)]), par, 0, pk});
        bprev = t;
        q = qn;
      };
      auto open_chain = [&](NsPick pk) {   // Gram product and the first B'
        ops.push_back(Op{kOpGram, bufs(0, 0, kNsBufA, ex.x, ex.x, ex.a), par, 0, pk});
        ops.push_back(Op{kOpPoly, bufs(kNsBufA, kNsBufA, kNsBufB, ex.a, ex.a, ex.b), par, 0, pk});
        bprev = q = kNsBufB;
        nq = 1;
      };
      auto update = [&](int last, NsPick pk) {   // X <- Q X
        ops.push_back(Op{kOpUpdate, bufs(q, 0, -1, ex.x, eb[q], ex.x), par, last, pk});
        par ^= 1;
      };
      if (adaptive) {
        // First chain: two iterations for every matrix, a third for those whose flag says so (k_ns_hf_chain_flag),
        // then pairs for all -- the last of them is the end for the flagged ones -- and one iteration more for the others.
        const NsPick longer{chain_flags, kNsLongOnly, 0, 0, 0.0f}, shorter{chain_flags, kNsShortOnly, 0, 0, 0.0f};
        const int n_pairs = (ns_iters - 3) / 2;
        open_chain(all);
        ops.push_back(Op{kOpFlag, NsBufs{0, 0, 0, 0.0f, 0.0f}, par, 0, all});
        extend(all);
        const int q_short = q, e_short = eb[q];
        extend(longer);
        update(n_pairs == 0, NsPick{chain_flags, kNsBoth, q_short, 0, pow2(-(ex.x + e_short))});
        for (int p = 0; p < n_pairs; ++p) {
          open_chain(all);
          extend(all);
          update(p == n_pairs - 1, NsPick{chain_flags, kNsBoth, q, 0, pow2(-(ex.x + eb[q]))});
        }
        open_chain(shorter);
        update(1, shorter);
      } else {
        int done = 0;
        for (size_t ch = 0; ch < chains.size(); ++ch) {
          // a chain of iterations: one Gram product, 4 len - 3 products of m x m matrices and one update (k_ns_hf.h)
          done += chains[ch];
          open_chain(all);
          for (int j = 1; j < chains[ch]; ++j) extend(all);
          update(done == ns_iters, all);
        }
      }
      for (const Op& op : ops)
        for (int g = 0; g < n_groups; ++g) {
          const NsGroup& G = L.ns_groups[bt.group0 + g];
          hipStream_t sg = stream_of(g);
          auto launch = [&](auto kern, int lds, const NsItem* items, int n) {
            if (n > 0)
              hipLaunchKernelGGL(kern, dim3(n), dim3(256), lds, sg, bmats, items, dyn, ns_ws, pw, op.par, op.last, op.b, c0, c1,
                                 c2, op.pick);
          };
          auto by_edge = [&](int edge, auto k128, auto k64, const NsItem* items, int n) {
            if (edge == 64) launch(k64, hf_gemm_lds(1, 1, 4), items, n);
            else launch(k128, hf_gemm_lds(2, 2, 1), items, n);
          };
          switch (op.kind) {
            case kOpGram:
              by_edge(G.gram_edge, k_ns_hf_gemm<kNsGram, 2, 2, 1>, k_ns_hf_gemm<kNsGram, 1, 1, 4>, gram + G.gram0, G.n_gram);
              if (G.n_split > 0)
                hipLaunchKernelGGL(k_ns_hf_gram_reduce, dim3(16 * hf_tiles_upper(G.split_max_m), G.n_split), dim3(64), 0, sg, bmats, split + G.split0, dyn, ns_ws, pw, op.pick, op.b.out_scale);
              break;
            case kOpFlag:
              if (G.n_list > 0) {
                hipLaunchKernelGGL(k_ns_hf_chain_sumsq, dim3(G.n_fitems), dim3(256), 0, sg, bmats, flag_items + G.fitem0, dyn,
                                   (const float*)ns_ws, chain_part);
                hipLaunchKernelGGL(k_ns_hf_chain_flag, dim3(G.n_list), dim3(64), 0, sg, bmats, list + G.list0, dyn,
                                   (const float*)chain_part, chain_tau2, chain_flags);
              }
              break;
            case kOpPoly:
              by_edge(G.poly_edge, k_ns_hf_gemm<kNsPoly, 2, 2, 1>, k_ns_hf_gemm<kNsPoly, 1, 1, 4>, poly + G.poly0, G.n_poly);
              break;
            case kOpProd:
              by_edge(G.poly_edge, k_ns_hf_gemm<kNsProd, 2, 2, 1>, k_ns_hf_gemm<kNsProd, 1, 1, 4>, poly + G.poly0, G.n_poly);
              break;
            case kOpProdA:
              by_edge(G.poly_edge, k_ns_hf_gemm<kNsProdA, 2, 2, 1>, k_ns_hf_gemm<kNsProdA, 1, 1, 4>, poly + G.poly0, G.n_poly);
              break;
            case kOpUpdate:
              launch(k_ns_hf_gemm<kNsUpdate, 2, 4, 1>, hf_gemm_lds(2, 4, 1), upd4 + G.upd40, G.n_upd4);
              by_edge(G.upd_edge, k_ns_hf_gemm<kNsUpdate, 2, 2, 1>, k_ns_hf_gemm<kNsUpdate, 1, 1, 4>, upd + G.upd0, G.n_upd);
              break;
          }
        }
      for (int g = 0; g < n_groups; ++g) {
        const NsGroup& G = L.ns_groups[bt.group0 + g];
        finish_range(stream_of(g), G.fin0, G.n_fin, G.unit0, G.n_units, nullptr, nullptr);
      }
      for (int g = 0; n_groups > 1 && g < n_groups; ++g) {
        HIP_TRY(hipEventRecord(P->ns_join[g], P->ns_side[g]));
        HIP_TRY(hipStreamWaitEvent(s, P->ns_join[g], 0));
      }
    }
  } else {
    // The fp32 matrix instructions: one chain for all matrices.
    const NsMat* mats = P->at<NsMat>(L.off_ns_mats);
    const NsItem* gram = P->at<NsItem>(L.off_ns_gram);
    const NsItem* poly = P->at<NsItem>(L.off_ns_poly);
    const NsItem* upd = P->at<NsItem>(L.off_ns_upd);
    const int* split = P->at<int>(L.off_ns_split);
    float* scale = P->at<float>(L.off_ns_scale);
    float* ns_ws = P->at<float>(L.off_ns_ws);
    const int n_mats = (int)L.ns_mats.size(), n_gram = (int)L.ns_gram.size(), n_poly = (int)L.ns_poly.size(),
              n_upd = (int)L.ns_upd.size(), n_split = (int)L.ns_split.size();
    // ||raw||: the finishing pass's sums of squares, taken on the raw steps
    hipLaunchKernelGGL(k_celo2_sumsq, dim3(n_fin), dim3(kThreads), 0, s, units, dyn, fin_items, fin_part,
                       (const long long*)nullptr, (const float*)nullptr);
    hipLaunchKernelGGL(k_ns_scale, dim3(n_mats), dim3(256), 0, s, mats, (const int*)nullptr, n_mats, units, fin_part, ns_eps,
                       scale);
    for (int it = 0; it < ns_iters; ++it) {
      const int first = it == 0, par = it & 1;
      hipLaunchKernelGGL(k_ns_gemm<kNsGram>, dim3(n_gram), dim3(256), 0, s, mats, gram, dyn, ns_ws, scale, first, par,
                         coeffs[0], coeffs[1], coeffs[2]);
      if (n_split > 0)
        hipLaunchKernelGGL(k_ns_gram_reduce, dim3(((size_t)L.ns_max_m * L.ns_max_m + 255) / 256, n_split), dim3(256), 0, s,
                           mats, split, dyn, ns_ws);
      hipLaunchKernelGGL(k_ns_gemm<kNsPoly>, dim3(n_poly), dim3(256), 0, s, mats, poly, dyn, ns_ws, scale, first, par,
                         coeffs[0], coeffs[1], coeffs[2]);
      hipLaunchKernelGGL(k_ns_gemm<kNsUpdate>, dim3(n_upd), dim3(256), 0, s, mats, upd, dyn, ns_ws, scale, first, par,
                         coeffs[0], coeffs[1], coeffs[2]);
    }
    // an odd number of iterations leaves the result in the second buffer
    const long long* x_alt = (ns_iters & 1) ? P->at<long long>(L.off_ns_xalt) : nullptr;
    finish_range(s, 0, n_fin, 0, (int)L.fin_units.size(), x_alt, ns_ws);
  }
  if (slices_aside) HIP_TRY(hipStreamWaitEvent(s, P->slice_join, 0));
  HIP_TRY(hipGetLastError());
  return 0;
}

}  // namespace

extern "C" int pylo_mi355_celo2_finish(PyloPlan* P, const PyloTensorArgs* args, void* stream) {
  return finish_impl(P, args, nullptr, 0, 0.0f, stream, "celo2_finish");
}

extern "C" int pylo_mi355_celo2_orthogonalize_finish(PyloPlan* P, const PyloTensorArgs* args, const float* ns_coeffs,
                                                     int ns_iters, float ns_eps, void* stream) {
  if (ns_iters < 0 || (ns_iters > 0 && !ns_coeffs)) return fail("celo2_orthogonalize_finish: bad Newton-Schulz arguments");
  return finish_impl(P, args, ns_coeffs, ns_iters, ns_eps, stream, "celo2_orthogonalize_finish");
}

extern "C" int pylo_mi355_plan_finish_supported(const PyloPlan* P, int tensor) {
  if (!P || tensor < 0 || tensor >= P->T || P->kind != PYLO_KIND_CELO2) return 0;
  return P->L.descs[tensor].mode == kModeFlat ? 0 : 1;
}

extern "C" int pylo_mi355_plan_orthogonalize_supported(const PyloPlan* P, int tensor) {
  if (!P || tensor < 0 || tensor >= P->T || P->kind != PYLO_KIND_CELO2) return 0;
  if (P->L.slice_of_tensor[tensor] >= 0) return P->L.slice_mats[P->L.slice_of_tensor[tensor]].no_orth ? 0 : 2;
  return P->L.ns_of_tensor[tensor] >= 0 || P->L.small_of_tensor[tensor] ? 1 : 0;
}

extern "C" int pylo_mi355_velo_step(PyloPlan* P, const PyloTensorArgs* args, const PyloDecays* decays,
                                    const PyloVeloNets* nets, const PyloVeloStep* step, void* stream) {
  if (!P || !args || !decays || !nets || !step) return fail("velo_step: null argument");
  if (P->kind != PYLO_KIND_VELO) return fail("velo_step: plan is not a VeLO plan");
  const int H = nets->hidden, K = nets->n_bank, T = P->T;
  if (H <= 0 || H % 64 != 0 || H > kVeloHiddenMax) return fail("velo_step: LSTM width must be a multiple of 64, at most 1024");
  if (K <= 0 || K > 4096) return fail("velo_step: bank size out of range");
  if (!nets->mix2_wt || !nets->mix2_b || !nets->fmix_wt || !nets->fmix_b || !nets->lstm_wt || !nets->lstm_b ||
      !nets->ctrl_wt || !nets->ctrl_b || !nets->lr_w || !nets->lr_b || !nets->bank)
    return fail("velo_step: null weight pointer");
  if (!step->lstm_h || !step->lstm_c || !step->loss_means || !step->loss_running_min || !step->loss_decays ||
      !step->loss_iteration || !step->loss)
    return fail("velo_step: null state pointer");
  if (int rc = check_args(P, args, true)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (int rc = upload_args(P, args, s, P->L.off_dyn_user)) return rc;
  stage_in(P, s, 3);
  advance_steps(P, s);
  // the sums the apply items carry over are taken on the fp32 parameter they write; the next step starts
  // from that value rounded to the tensor's storage type
  if (P->L.typed) P->stats_carried = false;
  const Layout& L = P->L;
  const TDesc* descs = P->at<TDesc>(L.off_descs);
  const PyloTensorArgs* dyn = P->at<PyloTensorArgs>(L.off_dyn);
  const Item* p0_items = P->at<Item>(L.off_p0_items);
  const Item* nd_items = P->at<Item>(L.off_nd_items);
  const Item* el_items = P->at<Item>(L.off_el_items);
  const Item* v0a_items = P->at<Item>(L.off_v0a_items);
  const Item* v0b_items = P->at<Item>(L.off_v0b_items);
  float* part = P->at<float>(L.off_part);
  double* gsq = P->at<double>(L.off_gsq);
  int* flag = P->at<int>(L.off_flag);
  Globals* gl = P->at<Globals>(L.off_globals);
  float* fac_tab = P->at<float>(L.off_fac);
  float* term_tab = P->at<float>(L.off_term);
  double* v0part = P->at<double>(L.off_v0part);
  BScale* bscale = P->at<BScale>(L.off_bscale);
  double* stats = P->at<double>(L.off_stats);
  float* wfold = P->at<float>(L.off_wfold);
  double* totals = P->at<double>(L.off_totals);
  float* xfeat = P->at<float>(L.off_xfeat);
  float* xT = P->at<float>(L.off_xT);
  float* canon = P->at<float>(L.off_canon);
  float* mixbuf = P->at<float>(L.off_mixbuf);
  const int n_p0 = (int)L.p0_items.size(), n_nd = (int)L.nd_items.size(), n_el = (int)L.el_items.size();
  const int n_v0a = (int)L.v0a_items.size(), n_v0b = (int)L.v0b_items.size();
  const PyloDecays dec = *decays;
  VeloStep vs;
  std::memcpy(vs.frac, step->frac, sizeof(vs.frac));
  vs.frac_dev = P->dsteps.counters ? P->at<float>(L.off_frac) : nullptr;
  Marks mark(P, s);
  float* piv = P->at<float>(L.off_piv);
  double* newsum = P->at<double>(L.off_newsum);
  float* wmix = P->at<float>(L.off_wmix);
  const LossState ls{step->loss_means, step->loss_running_min, step->loss_decays, step->loss_iteration, step->loss};
  const int n_chunks = (T + kMixRows - 1) / kMixRows;
  float* pmax = n_chunks > 1 ? P->at<float>(L.off_pmax) : nullptr;
  const size_t heads_lds = sizeof(float) * (H + K + 160 + 32 + 16 + 4 * (size_t)std::max(K, 160));
  auto heads = [&](hipStream_t q, const double* tot, bool many) {
    const bool rows4 = many && 4 * heads_lds <= 64 * 1024;
    hipLaunchKernelGGL((rows4 ? k_velo_heads<4, kThreads> : k_velo_heads<1, kFoldThreads>), dim3(rows4 ? (T + 3) / 4 : T),
                       dim3(rows4 ? kThreads : kFoldThreads),
                       rows4 ? 4 * heads_lds : heads_lds, q, descs, T, H, K, step->lstm_h,
                       nets->ctrl_wt, nets->ctrl_b, nets->lr_w, nets->lr_b, nets->bank, tot, canon, wfold,
                       step->controls_out, step->lr_mult_out, wmix);
  };
  // The LSTM from the tensors' 30 input features on: input mixing across tensors, cell, heads.
  auto lstm = [&](hipStream_t q, const double* tot, bool timed) {
    if (pmax != nullptr)
      hipLaunchKernelGGL(k_velo_colmax, dim3(H / 64, n_chunks), dim3(kThreads), 0, q, (const float*)mixbuf, T, H, pmax);
    hipLaunchKernelGGL(k_velo_mix, dim3(H / 64, L.Tpad / kGateBT), dim3(kThreads), 0, q, (const float*)mixbuf, T, L.Tpad, H,
                       (const float*)pmax, n_chunks, step->lstm_h, xT, ls);
    if (timed) (void)mark();
    const bool many = T >= kManyRows;
    if (many)
      hipLaunchKernelGGL(k_velo_gates_many, dim3((T + kGateM - 1) / kGateM * (H / kGateMU)), dim3(kThreads), 0, q, xT, T, L.Tpad, H,
                         nets->lstm_wt, nets->lstm_b, step->lstm_h, step->lstm_c);
    else
      hipLaunchKernelGGL(k_velo_gates, dim3((L.Tpad / kGateBT) * (H / kGateU)), dim3(kThreads), 0, q, xT, T, L.Tpad, H,
                         nets->lstm_wt, nets->lstm_b, step->lstm_h, step->lstm_c);
    if (timed) (void)mark();
    heads(q, tot, many);
    if (timed) (void)mark();
  };
  // clip_norm is 0 for VeLO tensors: k_p0 clamps directly; its norm / flag outputs are not used
  // no global norm to wait for: the N-D tensors' sums ride in the tail blocks of the same launch
  const bool typed = L.in_place;
  auto gradient_sums = [&]() {
    if (n_p0 + n_nd > 0)
      hipLaunchKernelGGL(p0_kernel(typed, L.split), dim3(n_p0 + n_nd), dim3(kThreads), 0, s, descs, dyn, p0_items, part, gsq, flag, gl, 0,
                         nd_items, n_p0);
  };
  auto factor_tables = [&]() {
    if (n_v0a > 0)
      hipLaunchKernelGGL(k_v0a, dim3(n_v0a), dim3(kV0aThreads), 0, s, descs, dyn, v0a_items, part, gl, dec, v0part);
    HIP_TRY(mark());
    if (n_v0b > 0)
      hipLaunchKernelGGL(k_v0b<4>, dim3(n_v0b), dim3(kThreads), 0, s, descs, dyn, v0b_items, v0part, 1e-5f,
                         (const float*)nullptr, (const float*)nullptr, 0, fac_tab, term_tab, bscale);
    HIP_TRY(mark());
    return 0;
  };
  const int n_mx = (int)L.mx_items.size();
  HIP_TRY(mark());
  if (L.fused && P->stats_carried) {
    // The LSTM's inputs are sums over the parameters and accumulators as they stand before the step: the
    // previous step's apply items left them.  It runs next to the gradient sums, on the plan's own stream or, where there are
    // few blocks, in the launches of the caller's.
    const unsigned n_big = (unsigned)L.big_items.size();
    const bool paired = n_p0 + n_nd + T <= kVeloPaired && T <= kMixRows && n_big == 0;
    const hipStream_t q = paired ? s : P->side;
    if (!paired) {
      HIP_TRY(hipEventRecord(P->ev_fork, s));
      HIP_TRY(hipStreamWaitEvent(q, P->ev_fork, 0));
    }
    if (!L.seg_items.empty())
      hipLaunchKernelGGL(k_stat_segsum<kNewSumW>, dim3((unsigned)L.seg_items.size()), dim3(kThreads), 0, q, descs,
                         P->at<Item>(L.off_seg_items), (const double*)newsum, P->at<double>(L.off_segtot));
    if (paired) {
      const int n_mix = (H / 64) * (L.Tpad / kGateBT), n_gates = (L.Tpad / kGateBT) * (H / kGateU);
      hipLaunchKernelGGL((L.split ? k_velo_p0_feat<true> : k_velo_p0_feat<false>), dim3(T + n_p0 + n_nd), dim3(kFoldThreads), 0, s, descs, dyn,
                         p0_items, part, gsq, flag, gl, nd_items, n_p0, T, (const double*)newsum, (const double*)P->at<double>(L.off_segtot),
                         piv, ls, vs, xfeat, H, nets->mix2_wt, nets->mix2_b, nets->fmix_wt, nets->fmix_b, mixbuf, P->at<int>(L.off_sync));
      HIP_TRY(mark());
      hipLaunchKernelGGL(k_velo_v0a_mix, dim3(n_mix + n_v0a), dim3(kThreads), 0, s, descs, dyn, v0a_items, part, gl, dec, v0part,
                         (const float*)mixbuf, T, L.Tpad, H, step->lstm_h, xT, ls);
      HIP_TRY(mark());
      hipLaunchKernelGGL(k_velo_v0b_gates, dim3(n_gates + n_v0b), dim3(kThreads), 0, s, descs, dyn, v0b_items, v0part, fac_tab, term_tab,
                         bscale, xT, T, L.Tpad, H, nets->lstm_wt, nets->lstm_b, step->lstm_h, step->lstm_c);
      heads(s, nullptr, false);
      HIP_TRY(mark());
    } else {
      hipLaunchKernelGGL(k_velo_feat, dim3(T), dim3(kThreads), 0, P->side, descs, dyn, T, (const double*)newsum,
                         (const double*)P->at<double>(L.off_segtot), piv, ls, vs,
                         xfeat, H, nets->mix2_wt, nets->mix2_b, nets->fmix_wt, nets->fmix_b, mixbuf, P->at<int>(L.off_sync));
      lstm(P->side, nullptr, false);
      HIP_TRY(hipEventRecord(P->ev_join, P->side));
      gradient_sums();
      HIP_TRY(mark());
      if (int rc = factor_tables()) return rc;
      // the streamed tensors' statistics need nothing from the LSTM either: its launches have this one to run under as well
      if (n_big > 0)
        hipLaunchKernelGGL((L.split ? k_velo_stats<false, true> : k_velo_stats<false, false>), dim3(n_big), dim3(kThreads), 0, s, descs, dyn,
                           P->at<Item>(L.off_big_items), fac_tab, dec, stats);
      HIP_TRY(hipStreamWaitEvent(s, P->ev_join, 0));
    }
    if (n_v0b > 0)
      hipLaunchKernelGGL(k_terms<4>, dim3(n_v0b), dim3(kThreads), 0, s, descs, dyn, v0b_items, bscale, canon, kVCanon, term_tab);
    HIP_TRY(mark());
    if (!L.big_seg.empty())
      hipLaunchKernelGGL(k_stat_segsum<kStatW>, dim3((unsigned)L.big_seg.size()), dim3(kThreads), 0, s, descs,
                         P->at<Item>(L.off_big_seg), (const double*)stats, P->at<double>(L.off_segtot));
    if (n_big > 0)
      hipLaunchKernelGGL(k_velo_fold, dim3((unsigned)L.big_list.size()), dim3(kThreads), 0, s, descs, dyn, P->at<int>(L.off_big_list),
                         (const double*)stats, (const double*)P->at<double>(L.off_segtot), (const float*)wmix, wfold,
                         P->at<int>(L.off_sync), T);
    const auto elem = L.split ? k_velo_elem<true> : k_velo_elem<false>;
    if (n_mx > 0)
      hipLaunchKernelGGL(elem, dim3(n_mx), dim3(kThreads), 0, s, descs, dyn, P->at<Item>(L.off_mx_items), fac_tab, term_tab,
                         dec, (const float*)wmix, wfold, stats, (const float*)piv, newsum, P->at<int>(L.off_sync), T);
    if (n_big > 0)
      hipLaunchKernelGGL((L.split ? k_velo_apply<false, true> : k_velo_apply<false, false>), dim3(n_big), dim3(kThreads), 0, s, descs, dyn, P->at<Item>(L.off_big_apply), fac_tab,
                         term_tab, dec, (const float*)wfold, (const float*)piv, newsum);
    HIP_TRY(mark());
    mark.done();
    stage_out(P, s, 0);
    HIP_TRY(hipGetLastError());
    return 0;
  }
  // Each pass as a launch of its own: the first step of a plan, a step after its carried sums were
  // invalidated, and every step with PYLO_MI355_SLAB_ELEMS=0.
  gradient_sums();
  HIP_TRY(mark());
  HIP_TRY(mark(L.fused));
  if (int rc = factor_tables()) return rc;
  const auto stats_pass = variant(typed, L.split, k_velo_stats<false, false>, k_velo_stats<false, true>, k_velo_stats<true, false>,
                                  k_velo_stats<true, true>);
  const auto apply_pass = variant(typed, L.split, k_velo_apply<false, false>, k_velo_apply<false, true>, k_velo_apply<true, false>,
                                  k_velo_apply<true, true>);
  if (n_el > 0) hipLaunchKernelGGL(stats_pass, dim3(n_el), dim3(kThreads), 0, s, descs, dyn, el_items, fac_tab, dec, stats);
  HIP_TRY(mark(L.fused));
  const Item* seg_items = P->at<Item>(L.off_seg_items);
  double* seg_tot = P->at<double>(L.off_segtot);
  const int n_seg = (int)L.seg_items.size();
  if (n_seg > 0) hipLaunchKernelGGL(k_stat_segsum<kStatW>, dim3(n_seg), dim3(kThreads), 0, s, descs, seg_items, stats, seg_tot);
  hipLaunchKernelGGL(k_lo_reduce, dim3(T), dim3(kFoldThreads), 0, s, descs, dyn, T, stats, seg_tot, totals, ls, vs, xfeat,
                     H, nets->mix2_wt, nets->mix2_b, nets->fmix_wt, nets->fmix_b, mixbuf, piv);
  HIP_TRY(mark(L.fused));
  lstm(s, totals, !L.fused);   // the LSTM's launches have intervals of their own only in the launch list without k_velo_elem
  if (n_v0b > 0)
    hipLaunchKernelGGL(k_terms<4>, dim3(n_v0b), dim3(kThreads), 0, s, descs, dyn, v0b_items, bscale, canon, kVCanon, term_tab);
  HIP_TRY(mark());
  if (n_el > 0)
    hipLaunchKernelGGL(apply_pass, dim3(n_el), dim3(kThreads), 0, s, descs, dyn, el_items, fac_tab, term_tab, dec, wfold,
                       (const float*)piv, newsum);
  HIP_TRY(mark());
  mark.done();
  stage_out(P, s, 0);
  HIP_TRY(hipGetLastError());
  P->stats_carried = L.fused;
  return 0;
}

extern "C" int pylo_mi355_plan_invalidate_statistics(PyloPlan* P) {
  if (!P) return fail("plan_invalidate_statistics: null plan");
  P->stats_carried = false;
  if (P->stale_host) *static_cast<volatile int*>(P->stale_host) = 0;   // what the guard found before this call no longer counts
  return 0;
}

extern "C" int pylo_mi355_plan_statistics_stale(const PyloPlan* P) {
  if (!P || !P->stale_host) return 0;
  return *static_cast<const volatile int*>(P->stale_host);
}

extern "C" int pylo_mi355_advance_counters(double* const* counters, int n, double* before) {
  if (n < 0 || (n > 0 && (!counters || !before))) return fail("advance_counters: null argument");
  for (int i = 0; i < n; ++i) {
    before[i] = *counters[i];
    *counters[i] = before[i] + 1.0;
  }
  return 0;
}

extern "C" int pylo_mi355_adafac_step(PyloPlan* P, const PyloTensorArgs* args, const PyloDecays* decays,
                                      const float* net, float step, void* stream) {
  if (!P || !args || !decays || !net) return fail("adafac_step: null argument");
  if (P->kind != PYLO_KIND_ADAFAC) return fail("adafac_step: plan is not an AdafacLO plan");
  if (int rc = check_args(P, args, false)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (int rc = upload_args(P, args, s, P->L.off_dyn_user)) return rc;
  stage_in(P, s, 3);
  advance_steps(P, s);
  const Layout& L = P->L;
  const TDesc* descs = P->at<TDesc>(L.off_descs);
  const PyloTensorArgs* dyn = P->at<PyloTensorArgs>(L.off_dyn);
  const Item* p0_items = P->at<Item>(L.off_p0_items);
  const Item* nd_items = P->at<Item>(L.off_nd_items);
  const Item* el_items = P->at<Item>(L.off_el_items);
  const Item* v0a_items = P->at<Item>(L.off_v0a_items);
  const Item* v0b_items = P->at<Item>(L.off_v0b_items);
  float* part = P->at<float>(L.off_part);
  double* gsq = P->at<double>(L.off_gsq);
  int* flag = P->at<int>(L.off_flag);
  Globals* gl = P->at<Globals>(L.off_globals);
  float* fac_tab = P->at<float>(L.off_fac);
  float* term_tab = P->at<float>(L.off_term);
  double* v0part = P->at<double>(L.off_v0part);
  BScale* bscale = P->at<BScale>(L.off_bscale);
  double* stats = P->at<double>(L.off_stats);
  float* wfold = P->at<float>(L.off_wfold);
  float* bias_eff = P->at<float>(L.off_xfeat);  // [T][32]; the LSTM feature buffer is unused by this kind
  const int n_p0 = (int)L.p0_items.size(), n_nd = (int)L.nd_items.size(), n_el = (int)L.el_items.size();
  const int n_v0a = (int)L.v0a_items.size(), n_v0b = (int)L.v0b_items.size();
  const int T = P->T;
  const PyloDecays dec = *decays;
  const bool in_place = L.in_place;   // tensors of 16-bit storage without staging (the fp16 matrix instructions' walk only)
  Marks mark(P, s);

  // ELO's global-norm clipping (ELO_cuda.py:153-161): the norm, then the exact sums where an element
  // is not a fixed point of the conditioning.  Plain AdafacLO steps skip both launches.
  bool clips = false;
  for (int t = 0; t < T; ++t) clips = clips || (args[t].grad != nullptr && args[t].clip_norm > 0.0f);
  if (clips && !L.global_norm)
    return fail("adafac_step: clip_norm > 0 needs a plan built with PYLO_F_GLOBAL_NORM or PYLO_F_TENSOR_NORM");
  if (clips && L.tensor_norm)
    for (int t = 0; t < T; ++t)
      if (args[t].grad != nullptr && args[t].clip_norm > 0.0f && args[t].clip_val != 0.0f)
        return fail("adafac_step: a tensor clipped by its own norm (PYLO_F_TENSOR_NORM) takes no clip_val");
  HIP_TRY(mark());
  // without global-norm clipping the N-D tensors' sums ride in the tail blocks of the first launch
  const int n_tail = clips ? 0 : n_nd;
  if (n_p0 + n_tail > 0)
    hipLaunchKernelGGL(p0_kernel(in_place, L.split), dim3(n_p0 + n_tail), dim3(kThreads), 0, s, descs, dyn, p0_items, part, gsq, flag, gl, 0,
                       nd_items, n_p0);
  if (clips && L.tensor_norm) {
    // every tensor against its own norm (AdafacLO_naive.py:199-200): no clamp on such tensors, no exact pass
    hipLaunchKernelGGL(k_tnorm, dim3(T), dim3(kThreads), 0, s, descs, dyn, gsq, gl, P->at<float>(L.off_tscale));
  }
  NormArgs na{gsq, flag, n_p0, 0, nullptr, 0};
  bool norm_v0a = false;
  if (clips && !L.tensor_norm) {
    const bool exact_pass = exact_pass_possible(P, args), few = n_p0 > 0 && n_p0 <= kNormBlocks;
    na.use_flags = exact_pass ? 1 : 0;
    norm_v0a = few && !exact_pass && n_nd == 0;
    if (few && exact_pass) {
      hipLaunchKernelGGL(norm_p0_kernel(in_place, L.split), dim3(n_p0), dim3(kThreads), 0, s, descs, dyn, p0_items, part, na, gl);
    } else if (!norm_v0a) {
      hipLaunchKernelGGL(k_gnorm, dim3(1), dim3(kThreads), 0, s, na, gl);
      if (n_p0 > 0 && exact_pass)
        hipLaunchKernelGGL(p0_kernel(in_place, L.split), dim3(n_p0), dim3(kThreads), 0, s, descs, dyn, p0_items, part, gsq, flag, gl, 1,
                           (const Item*)nullptr, n_p0);
    }
  }
  HIP_TRY(mark());
  if (n_nd > 0 && clips) hipLaunchKernelGGL(k_p0_nd, dim3(n_nd), dim3(kThreads), 0, s, descs, dyn, nd_items, part, gl);
  HIP_TRY(mark());
  hipLaunchKernelGGL((norm_v0a ? k_adafac_v0a<true> : k_adafac_v0a<false>), dim3(n_v0a + T), dim3(kThreads), 0, s, descs, dyn, v0a_items,
                     n_v0a, part, na, gl, dec, v0part, net, P->dsteps.counters ? -1.0f : step, bias_eff);
  HIP_TRY(mark());
  if (n_v0b > 0)
    hipLaunchKernelGGL(k_v0b<kAH>, dim3(n_v0b), dim3(kThreads), 0, s, descs, dyn, v0b_items, v0part, 1e-5f,
                       net + kAW1, (const float*)bias_eff, kAH, fac_tab, term_tab, bscale);
  HIP_TRY(mark());
  const auto stats_pass = variant(in_place, L.split, k_adafac_stats<false, false>, k_adafac_stats<false, true>,
                                  k_adafac_stats<true, false>, k_adafac_stats<true, true>);
  if (n_el > 0)
    hipLaunchKernelGGL(stats_pass, dim3(n_el), dim3(kThreads), 0, s, descs, dyn,
                       el_items, fac_tab, dec, stats, gl);
  HIP_TRY(mark());
  const Item* seg_items = P->at<Item>(L.off_seg_items);
  double* seg_tot = P->at<double>(L.off_segtot);
  const int n_seg = (int)L.seg_items.size();
  if (n_seg > 0) hipLaunchKernelGGL(k_stat_segsum<kStatW>, dim3(n_seg), dim3(kThreads), 0, s, descs, seg_items, stats, seg_tot);
  hipLaunchKernelGGL(k_adafac_fold, dim3(T), dim3(kFoldThreads), 0, s, descs, dyn, stats, seg_tot, net, wfold);
  HIP_TRY(mark());
  const Item* ap_items = P->at<Item>(L.off_ap_items);
  const Item* ga_items = P->at<Item>(L.off_ga_items);
  const Item* pp_items = P->at<Item>(L.off_pp_items);
  const int n_ap = (int)L.ap_items.size(), n_ga = (int)L.ga_items.size(), n_pp = (int)L.pp_items.size();
  const bool both = n_ga > 0 && n_ap > 0 && n_ga + n_ap <= kApplyTogether && L.lin_matrix && P->adafac_hf && !in_place;
  if (both)
    hipLaunchKernelGGL(k_adafac_apply_both, dim3(n_ap + n_ga), dim3(kThreads), 0, s, descs, dyn, ap_items, n_ap, ga_items, fac_tab, term_tab,
                       dec, wfold, net, (const float*)bias_eff, gl);
  else if (n_ga > 0 && L.lin_matrix)
    hipLaunchKernelGGL(k_adafac_apply_lin, dim3(n_ga), dim3(kThreads), 0, s, descs, dyn, ga_items, fac_tab, term_tab, dec,
                       wfold, net, (const float*)bias_eff, gl);
  else if (n_ga > 0)
    hipLaunchKernelGGL(k_adafac_apply, dim3(n_ga), dim3(kThreads), 0, s, descs, dyn, ga_items, fac_tab, term_tab, dec,
                       wfold, net, (const float*)bias_eff, gl);
  if (n_pp > 0)
    hipLaunchKernelGGL((k_adafac_apply_tile<true, true>), dim3(n_pp), dim3(kThreads), 0, s, descs, dyn, pp_items, fac_tab,
                       term_tab, dec, wfold, net, gl);
  if (n_ap > 0 && !both) {
    const auto apply = in_place       ? k_adafac_apply_tile<true, false, true>
                       : P->adafac_hf ? k_adafac_apply_tile<true, false, false>
                                      : k_adafac_apply_tile<false, false, false>;
    hipLaunchKernelGGL(apply, dim3(n_ap), dim3(kThreads), 0, s, descs, dyn, ap_items, fac_tab, term_tab, dec, wfold, net, gl);
  }
  HIP_TRY(mark());
  mark.done();
  stage_out(P, s, 0);
  HIP_TRY(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------------------------
// Single-tensor calls with the reference's argument lists
// ---------------------------------------------------------------------------------------------
namespace {

// Geometry as the reference launchers derive it from the parameter tensor (celo2_kernel.cu:306-312):
// sizes and strides of dims dr / dc of a contiguous tensor.
int single_geometry(const char* who, const int64_t* shape, int ndim, int dc, int dr, int vector_like, SingleArgs& a) {
  const std::string w(who);
  if (ndim < 0 || ndim > PYLO_MAX_DIMS || (ndim > 0 && !shape)) return fail(w + ": bad shape");
  long long n = 1;
  for (int i = 0; i < ndim; ++i) {
    if (shape[i] < 0) return fail(w + ": negative dim");
    n *= shape[i];
    if (n >= (1LL << 31)) return fail(w + ": tensors of 2^31 elements or more are not supported");
  }
  a.n = (int)n;
  a.vector_like = vector_like ? 1 : 0;
  if (vector_like) {
    a.num_rows = a.num_cols = a.n;
    a.row_stride = a.col_stride = 1;
    return 0;
  }
  if (dc < 0 || dr < 0 || dc >= ndim || dr >= ndim || dc == dr) return fail(w + ": dc / dr are not two dims of the tensor");
  auto stride = [&](int d) {
    long long st = 1;
    for (int i = d + 1; i < ndim; ++i) st *= shape[i];
    return (int)st;
  };
  a.num_rows = (int)shape[dr];
  a.num_cols = (int)shape[dc];
  a.row_stride = stride(dr);
  a.col_stride = stride(dc);
  if (a.n > 0) {   // then every dim is at least 1
    a.stride_r = a.n / a.num_rows;
    a.stride_c = a.n / a.num_cols;
    a.div_rblock = make_fastdiv((unsigned)a.num_rows * (unsigned)a.row_stride);
    a.div_rstride = make_fastdiv((unsigned)a.row_stride);
    a.div_cblock = make_fastdiv((unsigned)a.num_cols * (unsigned)a.col_stride);
    a.div_cstride = make_fastdiv((unsigned)a.col_stride);
  }
  return 0;
}

template <int F>
int single_check(const char* who, const SingleArgs& a) {
  if (a.n == 0) return 0;
  if (!a.g || !a.p || !a.m || !a.v || !a.fac_r || !a.fac_c || !a.row_factor || !a.second_moment || !a.w_in ||
      !a.b_in || !a.w_h || !a.b_h || !a.w_out || !a.b_out || (!a.vector_like && !a.col_factor) ||
      (F == kFamCelo2 && !a.step_out))
    return fail(std::string(who) + ": null pointer");
  return 0;
}

template <int F, int ST>
void single_enqueue(const SingleArgs& a, int blocks, hipStream_t s) {
  hipLaunchKernelGGL((k_single_moment<F, ST>), dim3(blocks), dim3(kSingleThreads), 0, s, a);
  hipLaunchKernelGGL((k_single_apply<F, ST>), dim3(blocks), dim3(kSingleThreads), 0, s, a);
}

// `dtype`: PYLO_F_STORE_* of every array but `second_moment` (the reference's scalar_t)
template <int F>
int single_launch(const char* who, const SingleArgs& a, void* stream, int dtype = PYLO_F_STORE_F32) {
  if (dtype & ~PYLO_F_STORE_MASK) return fail(std::string(who) + ": dtype must be one of PYLO_F_STORE_*");
  if (a.n == 0) return 0;
  if (int rc = single_check<F>(who, a)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int blocks = std::min((a.n + kSingleThreads - 1) / kSingleThreads, kSingleMaxBlocks);
  switch (dtype >> 8) {
    case kStoreF16: single_enqueue<F, kStoreF16>(a, blocks, s); break;
    case kStoreBF16: single_enqueue<F, kStoreBF16>(a, blocks, s); break;
    case kStoreF64: single_enqueue<F, kStoreF64>(a, blocks, s); break;
    default: single_enqueue<F, kStoreF32>(a, blocks, s);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

}  // namespace

extern "C" int pylo_mi355_celo2_kernel(const float* g, const float* p, const float* m, const float* v,
                                       const float* fac_r, const float* fac_c, const float* row_factor,
                                       const float* col_factor, float* second_moment, const float* w_in,
                                       const float* b_in, const float* w_h, const float* b_h, const float* w_out,
                                       const float* b_out, float* step_out, float exp_mult, const int64_t* shape,
                                       int ndim, int dc, int dr, int vector_like, void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("celo2_kernel", shape, ndim, dc, dr, vector_like, a)) return rc;
  a.g = g; a.p = const_cast<float*>(p); a.m = m; a.v = v; a.fac_r = fac_r; a.fac_c = fac_c;
  a.row_factor = row_factor; a.col_factor = col_factor; a.second_moment = second_moment;
  a.w_in = w_in; a.b_in = b_in; a.w_h = w_h; a.b_h = b_h; a.w_out = w_out; a.b_out = b_out;
  a.step_out = step_out; a.exp_mult = exp_mult;
  return single_launch<kFamCelo2>("celo2_kernel", a, stream);
}

extern "C" int pylo_mi355_learned_optimizer_kernel(const float* g, float* p, const float* m, const float* v,
                                                   const float* fac_r, const float* fac_c, const float* row_factor,
                                                   const float* col_factor, float* second_moment,
                                                   const float* input_weights, const float* input_bias,
                                                   const float* hidden_weights, const float* hidden_bias,
                                                   const float* output_weights, const float* output_bias, float lr,
                                                   float step_mult, float exp_mult, float epsilon, float step,
                                                   float weight_decay, const int64_t* shape, int ndim, int dc, int dr,
                                                   int vector_like, void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("learned_optimizer_kernel", shape, ndim, dc, dr, vector_like, a)) return rc;
  a.g = g; a.p = p; a.m = m; a.v = v; a.fac_r = fac_r; a.fac_c = fac_c;
  a.row_factor = row_factor; a.col_factor = col_factor; a.second_moment = second_moment;
  a.w_in = input_weights; a.b_in = input_bias; a.w_h = hidden_weights; a.b_h = hidden_bias;
  a.w_out = output_weights; a.b_out = output_bias;
  a.lr = lr; a.step_mult = step_mult; a.exp_mult = exp_mult; a.epsilon = epsilon; a.step = step;
  a.weight_decay = weight_decay;
  return single_launch<kFamLo>("learned_optimizer_kernel", a, stream);
}

extern "C" int pylo_mi355_velo_kernel_simple(const float* grad, float* param, const float* momentum, const float* rms,
                                             const float* row_factor, const float* col_factor,
                                             const float* fac_vec_row, const float* fac_vec_col, float* second_moment,
                                             const float* input_weights, const float* input_bias,
                                             const float* hidden_weights, const float* hidden_bias,
                                             const float* output_weights, const float* output_bias, float lr,
                                             float step_mult, float exp_mult, float epsilon, float weight_decay,
                                             const int64_t* shape, int ndim, int dc, int dr, int vector_like,
                                             void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("velo_kernel_simple", shape, ndim, dc, dr, vector_like, a)) return rc;
  a.g = grad; a.p = param; a.m = momentum; a.v = rms; a.fac_r = fac_vec_row; a.fac_c = fac_vec_col;
  a.row_factor = row_factor; a.col_factor = col_factor; a.second_moment = second_moment;
  a.w_in = input_weights; a.b_in = input_bias; a.w_h = hidden_weights; a.b_h = hidden_bias;
  a.w_out = output_weights; a.b_out = output_bias;
  a.lr = lr; a.step_mult = step_mult; a.exp_mult = exp_mult; a.epsilon = epsilon; a.weight_decay = weight_decay;
  return single_launch<kFamVelo>("velo_kernel_simple", a, stream);
}

// The same three calls for arrays of another element type (the reference's AT_DISPATCH_FLOATING_TYPES_AND_HALF
// over p.scalar_type(), celo2_kernel.cu:314,328, learned_optimizer.cu:338,364, velo_kernel.cu:405,427): every
// array but `second_moment` holds elements of `dtype`.
#define PYLO_AS_F(x) static_cast<const float*>(x)
extern "C" int pylo_mi355_celo2_kernel_typed(int dtype, const void* g, const void* p, const void* m, const void* v,
                                             const void* fac_r, const void* fac_c, const void* row_factor,
                                             const void* col_factor, float* second_moment, const void* w_in,
                                             const void* b_in, const void* w_h, const void* b_h, const void* w_out,
                                             const void* b_out, void* step_out, float exp_mult, const int64_t* shape,
                                             int ndim, int dc, int dr, int vector_like, void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("celo2_kernel", shape, ndim, dc, dr, vector_like, a)) return rc;
  a.g = PYLO_AS_F(g); a.p = const_cast<float*>(PYLO_AS_F(p)); a.m = PYLO_AS_F(m); a.v = PYLO_AS_F(v);
  a.fac_r = PYLO_AS_F(fac_r); a.fac_c = PYLO_AS_F(fac_c);
  a.row_factor = PYLO_AS_F(row_factor); a.col_factor = PYLO_AS_F(col_factor); a.second_moment = second_moment;
  a.w_in = PYLO_AS_F(w_in); a.b_in = PYLO_AS_F(b_in); a.w_h = PYLO_AS_F(w_h); a.b_h = PYLO_AS_F(b_h);
  a.w_out = PYLO_AS_F(w_out); a.b_out = PYLO_AS_F(b_out);
  a.step_out = static_cast<float*>(step_out); a.exp_mult = exp_mult;
  return single_launch<kFamCelo2>("celo2_kernel", a, stream, dtype);
}

extern "C" int pylo_mi355_learned_optimizer_kernel_typed(int dtype, const void* g, void* p, const void* m, const void* v,
                                                         const void* fac_r, const void* fac_c, const void* row_factor,
                                                         const void* col_factor, float* second_moment,
                                                         const void* input_weights, const void* input_bias,
                                                         const void* hidden_weights, const void* hidden_bias,
                                                         const void* output_weights, const void* output_bias, float lr,
                                                         float step_mult, float exp_mult, float epsilon, float step,
                                                         float weight_decay, const int64_t* shape, int ndim, int dc,
                                                         int dr, int vector_like, void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("learned_optimizer_kernel", shape, ndim, dc, dr, vector_like, a)) return rc;
  a.g = PYLO_AS_F(g); a.p = static_cast<float*>(p); a.m = PYLO_AS_F(m); a.v = PYLO_AS_F(v);
  a.fac_r = PYLO_AS_F(fac_r); a.fac_c = PYLO_AS_F(fac_c);
  a.row_factor = PYLO_AS_F(row_factor); a.col_factor = PYLO_AS_F(col_factor); a.second_moment = second_moment;
  a.w_in = PYLO_AS_F(input_weights); a.b_in = PYLO_AS_F(input_bias); a.w_h = PYLO_AS_F(hidden_weights);
  a.b_h = PYLO_AS_F(hidden_bias); a.w_out = PYLO_AS_F(output_weights); a.b_out = PYLO_AS_F(output_bias);
  a.lr = lr; a.step_mult = step_mult; a.exp_mult = exp_mult; a.epsilon = epsilon; a.step = step;
  a.weight_decay = weight_decay;
  return single_launch<kFamLo>("learned_optimizer_kernel", a, stream, dtype);
}

extern "C" int pylo_mi355_velo_kernel_simple_typed(int dtype, const void* grad, void* param, const void* momentum,
                                                   const void* rms, const void* row_factor, const void* col_factor,
                                                   const void* fac_vec_row, const void* fac_vec_col,
                                                   float* second_moment, const void* input_weights,
                                                   const void* input_bias, const void* hidden_weights,
                                                   const void* hidden_bias, const void* output_weights,
                                                   const void* output_bias, float lr, float step_mult, float exp_mult,
                                                   float epsilon, float weight_decay, const int64_t* shape, int ndim,
                                                   int dc, int dr, int vector_like, void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("velo_kernel_simple", shape, ndim, dc, dr, vector_like, a)) return rc;
  a.g = PYLO_AS_F(grad); a.p = static_cast<float*>(param); a.m = PYLO_AS_F(momentum); a.v = PYLO_AS_F(rms);
  a.fac_r = PYLO_AS_F(fac_vec_row); a.fac_c = PYLO_AS_F(fac_vec_col);
  a.row_factor = PYLO_AS_F(row_factor); a.col_factor = PYLO_AS_F(col_factor); a.second_moment = second_moment;
  a.w_in = PYLO_AS_F(input_weights); a.b_in = PYLO_AS_F(input_bias); a.w_h = PYLO_AS_F(hidden_weights);
  a.b_h = PYLO_AS_F(hidden_bias); a.w_out = PYLO_AS_F(output_weights); a.b_out = PYLO_AS_F(output_bias);
  a.lr = lr; a.step_mult = step_mult; a.exp_mult = exp_mult; a.epsilon = epsilon; a.weight_decay = weight_decay;
  return single_launch<kFamVelo>("velo_kernel_simple", a, stream, dtype);
}
#undef PYLO_AS_F

// ---------------------------------------------------------------------------------------------
// celo2_kernel for callers that cannot allocate: the per-channel sums live in the library's own
// device array instead of a caller-supplied `second_moment`
// ---------------------------------------------------------------------------------------------
namespace {

constexpr int kScratchFloats = 64;   // 30 channel sums, padded to one 256-byte line
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
float* g_scratch_ptr[kMaxDevices];   // device address of `scratch` per GPU, resolved on first use
std::mutex g_scratch_mu;

// The array's name is a host-side stand-in, not a device address: each GPU holds its own copy at its
// own address, looked up once per device with that device current.
int scratch_on_current_device(float** out) {
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail("celo2_kernel_noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (ptr == nullptr) return fail("celo2_kernel_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = static_cast<float*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

// a fill kernel rather than a memset node: callers may record the call into a HIP graph
__global__ __launch_bounds__(64) void k_scratch_clear(float* __restrict__ s) { s[threadIdx.x] = 0.0f; }

}  // namespace

extern "C" int pylo_mi355_celo2_kernel_noalloc(const float* g, const float* p, const float* m, const float* v,
                                               const float* fac_r, const float* fac_c, const float* row_factor,
                                               const float* col_factor, const float* w_in, const float* b_in,
                                               const float* w_h, const float* b_h, const float* w_out,
                                               const float* b_out, float* step_out, float exp_mult,
                                               const int64_t* shape, int ndim, int dc, int dr, int vector_like,
                                               void* stream) {
  SingleArgs a{};
  if (int rc = single_geometry("celo2_kernel_noalloc", shape, ndim, dc, dr, vector_like, a)) return rc;
  float* sums = nullptr;
  if (int rc = scratch_on_current_device(&sums)) return rc;
  a.g = g; a.p = const_cast<float*>(p); a.m = m; a.v = v; a.fac_r = fac_r; a.fac_c = fac_c;
  a.row_factor = row_factor; a.col_factor = col_factor; a.second_moment = sums;
  a.w_in = w_in; a.b_in = b_in; a.w_h = w_h; a.b_h = b_h; a.w_out = w_out; a.b_out = b_out;
  a.step_out = step_out; a.exp_mult = exp_mult;
  if (a.n == 0) return 0;
  if (int rc = single_check<kFamCelo2>("celo2_kernel_noalloc", a)) return rc;
  // the array keeps the previous call's sums: they start at zero on every call
  hipLaunchKernelGGL(k_scratch_clear, dim3(1), dim3(kScratchFloats), 0, static_cast<hipStream_t>(stream), sums);
  return single_launch<kFamCelo2>("celo2_kernel_noalloc", a, stream);
}

// ---------------------------------------------------------------------------------------------
// Bare streaming kernel (benchmark instrumentation): the rate the memory system gives an access mix
// ---------------------------------------------------------------------------------------------
namespace {

template <int R, int W, bool NT>
__global__ __launch_bounds__(kThreads) void k_stream_probe(const float* __restrict__ in, float* __restrict__ out,
                                                           size_t n) {
  constexpr int kIters = 8;
  const size_t base = (size_t)blockIdx.x * kThreads * 4 * kIters;
  for (int it = 0; it < kIters; ++it) {
    const size_t i = base + ((size_t)it * kThreads + threadIdx.x) * 4;
    if (i >= n) break;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const gv4f* p = (const gv4f*)(in + (size_t)r * n + i);
      acc += NT ? __builtin_nontemporal_load(p) : *p;
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
      gv4f* p = (gv4f*)(out + (size_t)w * n + i);
      const v4f v = acc * (float)(w + 1);
      if (NT) __builtin_nontemporal_store(v, p);
      else *p = v;
    }
    if (W == 0 && acc.x == 123.456f) out[0] = acc.y;   // keeps the loads of a read-only mix alive
  }
}

template <int R, int W>
void stream_launch(const float* in, float* out, size_t n, bool nt, hipStream_t s) {
  const unsigned grid = (unsigned)((n + (size_t)kThreads * 4 * 8 - 1) / ((size_t)kThreads * 4 * 8));
  if (nt) hipLaunchKernelGGL((k_stream_probe<R, W, true>), dim3(grid), dim3(kThreads), 0, s, in, out, n);
  else hipLaunchKernelGGL((k_stream_probe<R, W, false>), dim3(grid), dim3(kThreads), 0, s, in, out, n);
}

}  // namespace

extern "C" int pylo_mi355_stream_probe(const float* in, float* out, size_t n, int reads, int writes, int nontemporal,
                                       void* stream) {
  if (!in || !out || n == 0 || n % 4 != 0) return fail("stream_probe: null pointer or n not a multiple of 4");
  if ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) % 16 != 0)
    return fail("stream_probe: 16-byte alignment needed");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool nt = nontemporal != 0;
  if (reads == 6 && writes == 5) stream_launch<6, 5>(in, out, n, nt, s);
  else if (reads == 6 && writes == 0) stream_launch<6, 0>(in, out, n, nt, s);
  else if (reads == 6 && writes == 1) stream_launch<6, 1>(in, out, n, nt, s);
  else if (reads == 1 && writes == 1) stream_launch<1, 1>(in, out, n, nt, s);
  else if (reads == 1 && writes == 0) stream_launch<1, 0>(in, out, n, nt, s);
  else if (reads == 1 && writes == 5) stream_launch<1, 5>(in, out, n, nt, s);
  else return fail("stream_probe: reads must be 1 or 6, writes 0, 1 or 5");
  HIP_TRY(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------------------------
// Bare matrix-pipe kernel (benchmark instrumentation): what the fp16 matrix instructions deliver for the
// instruction mix of the Newton-Schulz update product, with parts of its data path taken away
// ---------------------------------------------------------------------------------------------
namespace {

// The main loop of k_ns_hf_gemm<kNsUpdate, 4> (128 x 256 outputs, three v_mfma_f32_32x32x16_f16 per pair of
// 32 x 32 blocks and 16 reduction steps) over synthetic planes.  MODE 0: as in the product (operands staged
// from memory into LDS every 16 steps); 1: the first stage is staged once and read from LDS in every step (no
// global loads, no barriers); 2: the first stage's fragments stay in registers (matrix instructions only).
template <int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_matrix_probe(
    const hbits* __restrict__ X, int rows_x, const hbits* __restrict__ B, int rows_b, int K, float* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) char lds_[];
  PYLO_LDS char* lds = (PYLO_LDS char*)lds_;
  constexpr int WN = 4, RB = 64 * WN, SA = 128 * kNsRowB;
  const int nj = rows_b / RB, i0 = (blockIdx.x / nj) * 128, j0 = (blockIdx.x % nj) * RB;
  v16f acc[2][WN];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  const HfPlanes PX{X, rows_x}, PB{B, rows_b};
  if (MODE == 0) {
    hf_tile_product<2, WN>(PX, i0, PB, j0, 0, K, lds, acc);
  } else if (MODE == 4) {
    hf_tile_product_direct<WN>(PX, i0, PB, j0, 0, K, lds, acc);
  } else {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = (wave >> 1) * 64, wj = (wave & 1) * 32 * WN;
    hf_stage_issue<128>((const char*)X + (size_t)i0 * kNsRowB + 16 * lane, lds, wave);
    hf_stage_issue<RB>((const char*)B + (size_t)j0 * kNsRowB + 16 * lane, lds + SA, wave);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int oa = hf_frag(wi, lane), ob = SA + hf_frag(wj, lane);
    f16x8 a[2][kNsPl], b[WN][kNsPl];
    for (int k = 0; k < K; k += kHfBK) {
      if (MODE == 1 || k == 0) {
#pragma unroll
        for (int q = 0; q < kNsPl; ++q) {
#pragma unroll
          for (int i = 0; i < 2; ++i) a[i][q] = __builtin_bit_cast(f16x8, *(const luint4*)(lds + oa + i * 32 * kNsRowB + q * 256));
#pragma unroll
          for (int j = 0; j < WN; ++j) b[j][q] = __builtin_bit_cast(f16x8, *(const luint4*)(lds + ob + j * 32 * kNsRowB + q * 256));
        }
      }
#pragma unroll
      for (int term = 0; term < 3; ++term) {
        constexpr int pa[3] = {1, 0, 0}, pb[3] = {0, 1, 0};
#pragma unroll
        for (int hi = 0; hi < 2; ++hi)
#pragma unroll
          for (int hj = 0; hj < WN; ++hj)
            acc[hi][hj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[hi][pa[term]], b[hj][pb[term]], acc[hi][hj], 0, 0, 0);
      }
      if (MODE == 1) asm volatile("" ::: "memory");   // the fragments are read again in the next step
    }
  }
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum += acc[i][j][r];
  out[(size_t)blockIdx.x * 256 + threadIdx.x] = sum;
}

// MODE 3: the same loop with tiles of 256 x 256 outputs by 512 threads (4 x 2 waves of 64 x 128): two thirds of the
// bytes staged per product.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_matrix_probe_wide(
    const hbits* __restrict__ X, int rows_x, const hbits* __restrict__ B, int rows_b, int K, float* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) char lds_[];
  PYLO_LDS char* lds = (PYLO_LDS char*)lds_;
  constexpr int WN = 4;
  const int nj = rows_b / 256, i0 = (blockIdx.x / nj) * 256, j0 = (blockIdx.x % nj) * 256;
  v16f acc[2][WN];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  const HfPlanes PX{X, rows_x}, PB{B, rows_b};
  hf_tile_product<2, WN, 1, 8>(PX, i0, PB, j0, 0, K, lds, acc);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum += acc[i][j][r];
  out[(size_t)blockIdx.x * 512 + threadIdx.x] = sum;
}

}  // namespace

extern "C" int pylo_mi355_matrix_probe(const void* x_planes, int rows_x, const void* b_planes, int rows_b, int k_steps,
                                       int mode, float* out, void* stream) {
  if (!x_planes || !b_planes || !out) return fail("matrix_probe: null pointer");
  if (rows_x <= 0 || rows_x % 128 != 0 || rows_b <= 0 || rows_b % 256 != 0 || k_steps <= 0 || k_steps % 16 != 0)
    return fail("matrix_probe: rows_x must be a multiple of 128, rows_b of 256, k_steps of 16");
  if (mode < 0 || mode > 4) return fail("matrix_probe: mode must be 0 .. 4");
  if (mode == 3 && rows_x % 256 != 0) return fail("matrix_probe: mode 3 takes rows_x in multiples of 256");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)(rows_x / 128) * (unsigned)(rows_b / 256);
  static std::mutex mu;
  {
    std::lock_guard<std::mutex> lock(mu);
    HIP_TRY(hipFuncSetAttribute((const void*)k_matrix_probe<0>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 4, 1)));
    HIP_TRY(hipFuncSetAttribute((const void*)k_matrix_probe<1>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 4, 1)));
    HIP_TRY(hipFuncSetAttribute((const void*)k_matrix_probe<2>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 4, 1)));
    HIP_TRY(hipFuncSetAttribute((const void*)k_matrix_probe_wide, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 512 * kNsRowB));
    HIP_TRY(hipFuncSetAttribute((const void*)k_matrix_probe<4>, hipFuncAttributeMaxDynamicSharedMemorySize, hf_gemm_lds(2, 4, 1)));
  }
  const hbits* X = static_cast<const hbits*>(x_planes);
  const hbits* B = static_cast<const hbits*>(b_planes);
  if (mode == 0) hipLaunchKernelGGL(k_matrix_probe<0>, dim3(grid), dim3(256), hf_gemm_lds(2, 4, 1), s, X, rows_x, B, rows_b, k_steps, out);
  else if (mode == 1) hipLaunchKernelGGL(k_matrix_probe<1>, dim3(grid), dim3(256), hf_gemm_lds(2, 4, 1), s, X, rows_x, B, rows_b, k_steps, out);
  else if (mode == 2) hipLaunchKernelGGL(k_matrix_probe<2>, dim3(grid), dim3(256), hf_gemm_lds(2, 4, 1), s, X, rows_x, B, rows_b, k_steps, out);
  else if (mode == 3) hipLaunchKernelGGL(k_matrix_probe_wide, dim3(grid / 2), dim3(512), 2 * 512 * kNsRowB, s, X, rows_x, B, rows_b, k_steps, out);
  else hipLaunchKernelGGL(k_matrix_probe<4>, dim3(grid), dim3(256), 2 * 256 * kNsRowB, s, X, rows_x, B, rows_b, k_steps, out);
  HIP_TRY(hipGetLastError());
  return 0;
}
