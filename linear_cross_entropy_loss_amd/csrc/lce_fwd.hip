// Forward of the fused linear + cross-entropy operator on gfx950.
//
// fwd_tiles_kernel computes one 256(v) x 256(token) tile of the scaled logits
// z = logit_scale * x W with MFMA and reduces it, in registers, to per-token
// partials over each 128-column slice: logsumexp, and when monitoring is on
// the slice max, sum softmax*z and sum z^2.  The logit of the target column is
// written by the one lane that holds it.  No logits reach memory.  (The
// reference kernel, linear_cross_entropy/ops.py:190-236, computes the same
// per-tile lse but also stores the fp32 logits, ops.py:216.)
//
// fwd_rows_kernel merges the slice partials of each token into its lse and
// forms the per-token loss terms (ops.py:753-761); fwd_final_kernel sums them
// in a fixed order into the five scalars of ops.py:802 and the valid-label
// count of ops.py:705.  All reductions are order-deterministic.
#include <type_traits>

#include "lce_gemm_small.h"
#include "lce_fwd_epilogue.h"
#include "lce_internal.h"

namespace lce {

namespace {

// Persistent workgroups, operand stream pipelined across output tiles.  The
// launch covers `tiles_p` tile columns of the vocabulary window [v0, v0 + vw)
// starting at its column tile `tp0` (all full columns, or the one straddling V
// for the VTAIL variant).  The token rows are those of x, or -- when the tokens with ignored
// labels were packed away -- the first `rows` rows of the packed copy (the count lives on the device).
// WVH: the weight is stored (V, H) row-major, so that the P operand runs along K in memory like x does.
template <class T, bool VTAIL, bool KMASK, bool WVH, bool MON> struct FwdProblem {
  typedef typename elem_of<T>::type E;
  static constexpr bool kKMask = KMASK;
  static constexpr bool kSwapAB = false;
  static constexpr bool kVarK = false;
  static constexpr bool kQBlocked = false;
  static constexpr bool kQScale = false;
  static constexpr bool kSplit = is_pair<T>::value;
  LCE_DEV int64_t p_lo() const { return a.H * a.ldw * 2; }
  LCE_DEV int64_t q_lo() const { return a.x_lo * 2; }
  static constexpr bool kColumnEpilogue = !VTAIL;
  const FwdArgs& a;
  int64_t rows, ldx;
  const E* x;
  int tp0, tiles_p, tiles_q;
  LCE_DEV FwdProblem(const FwdArgs& a_)
      : a(a_), tp0(VTAIL ? (int)(a_.vw / kTile) : 0), tiles_p(VTAIL ? 1 : (int)(a_.vw / kTile)) {
    rows = a.n_rows ? packed_rows(a.n_rows, a.N) : a.N;
    const bool packed = rows != a.N;
    x = reinterpret_cast<const E*>(packed ? a.xc : a.x);
    ldx = packed ? a.ldxc : a.ldx;
    // rows of this launch's chunk that exist
    int64_t here = rows - a.row0;
    here = here < 0 ? 0 : (here > a.nc ? a.nc : here);
    tiles_q = (int)((here + kTile - 1) / kTile);
  }
  LCE_DEV int num_tiles() const { return tiles_p * tiles_q; }
  LCE_DEV void coords(int tile, int& tp, int& tq) const {
    tile_coords(tile, num_tiles(), tiles_p, tiles_q, 8, a.live, tp, tq);
    tp += tp0;
  }
  LCE_DEV void origins(int tile, const void*& p, const void*& q) const {
    int tp, tq;
    coords(tile, tp, tq);
    const int64_t v = (a.v0 - a.wv0) + (int64_t)tp * kTile;  // first column of the tile inside the buffer `w`
    p = reinterpret_cast<const E*>(a.w) + (WVH ? v * a.ldw : v);
    q = x + (a.row0 + (int64_t)tq * kTile) * ldx;
  }
  LCE_DEV const void* p_end() const {
    return WVH ? matrix_end<E>(a.w, a.Vw, a.ldw, a.H) : matrix_end<E>(a.w, kSplit ? 2 * a.H : a.H, a.ldw, a.Vw);
  }
  LCE_DEV const void* q_end() const { return matrix_end<E>(x, rows, ldx, kSplit ? a.x_lo + a.H : a.H); }
  LCE_DEV int k_valid(int) const { return (int)a.H; }
  // Column epilogue: the labels of this lane's four tokens are fetched three K tiles ahead.
  int64_t pf_y[kNB];
  int etp, etq;
  LCE_DEV void prefetch(int tile) {
    if constexpr (kColumnEpilogue) {
      int tp, tq;
      coords(tile, tp, tq);
      const int lane = threadIdx.x & 63, wq = threadIdx.x >> 7;
#pragma unroll
      for (int qb = 0; qb < kNB; ++qb) {
        const int64_t tok = a.row0 + (int64_t)tq * kTile + wq * kWaveTile + qb * kBlk + (lane & 31);
        pf_y[qb] = tok < rows ? a.y[tok] : a.ignore_index;
      }
    }
  }
  LCE_DEV void epilogue_begin(int tile, char*) {
    coords(tile, etp, etq);
    etp += (int)(a.v0 / kTile);
  }
  FwdColumnState est;
  template <int J> LCE_DEV void epilogue_slot(int, f32x16_t (&acc)[kNB][kNB], int slot, char*) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    fwd_epilogue_slot<T, J, MON, kNB>(a, est, acc, (int64_t)etp * kTile + (wave & 1) * kWaveTile,
                                      (int64_t)etq * kTile + (wave >> 1) * kWaveTile, slot);
  }
  LCE_DEV void epilogue_end(int, f32x16_t (&acc)[kNB][kNB], char*) const {
    const int tid = opaque_tid();
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t slice_v0 = (int64_t)etp * kTile + (wave & 1) * kWaveTile;
#pragma unroll
    for (int qb = 0; qb < kNB; ++qb) {
      const int64_t tok = a.row0 + (int64_t)etq * kTile + (wave >> 1) * kWaveTile + qb * kBlk + (lane & 31);
      const int64_t yy = pf_y[qb], rel = yy - slice_v0;
      const bool here = yy != a.ignore_index && rel >= 0 && rel < kWaveTile && ((rel >> 2) & 1) == (lane >> 5);
      fwd_store_target(a, acc, tok, qb, here ? (int)rel : -1);
    }
  }
  LCE_DEV void epilogue(int tile, f32x16_t (&acc)[kNB][kNB], char*) const {
    int tp, tq;
    coords(tile, tp, tq);
    const int wave = opaque_tid() >> 6;
    fwd_epilogue<T, VTAIL, MON, kNB>(a, rows, acc, a.v0 + (int64_t)tp * kTile + (wave & 1) * kWaveTile,
                                     (int64_t)tq * kTile + (wave >> 1) * kWaveTile);
  }
};

// TAIL: which tile columns the launch covers: the full ones (kNoTail), the one that straddles V (kTailOnly), or both
// (kWithTail): the tail tiles are then dealt to the workgroups after those that take part in the last round of full
// tiles.  A launch of its own for them is one tile's time long whatever their number, on ceil(rows / 256) of the
// compute units (N=16384, H=1024, V=1000: 36 + 34 us in two launches).
template <class T, int TAIL, bool KMASK, bool WVH, bool MON>
__global__ __launch_bounds__(kThreads) void fwd_tiles_persistent_kernel(const FwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename elem_of<T>::type E;
  int first = (int)blockIdx.x;
  if constexpr (TAIL != kTailOnly) {
    typedef FwdProblem<T, false, KMASK, WVH, MON> Full;
    Full prob(a);
    Pipe3<T, E, WVH, E, true, Full> pipe(prob);
    pipe.run(a.ldw, prob.ldx, logit_ktiles<T>(a.H), lds, first);
    if (TAIL == kWithTail) first = first_tail_tile(first, (int)gridDim.x, prob.num_tiles());
  }
  if constexpr (TAIL != kNoTail) {
    typedef FwdProblem<T, true, true, WVH, MON> Tail;
    Tail prob(a);
    if (first >= prob.num_tiles()) return;
    __syncthreads();  // (every wave is done with the main loop's LDS stages)
    Pipe3<T, E, WVH, E, true, Tail> pipe(prob);
    pipe.run(a.ldw, prob.ldx, logit_ktiles<T>(a.H), lds, first);
  }
}

// The same on 128 x 128 tiles (lce_gemm_small.h): workgroup = one slice of 128 columns, 128 tokens.  tiles_p slices; those past
// the vocabulary's end get partials as well, which the row merge reads.
template <class T, bool WVH, bool MON, bool WF32>
__global__ __launch_bounds__(kThreads, 2) void fwd_small_kernel(const FwdArgs a, int tiles_p, int tiles_q) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename elem_of<T>::type E;
  const int64_t rows = a.n_rows ? packed_rows(a.n_rows, a.N) : a.N;
  const bool packed = rows != a.N;
  const E* x = reinterpret_cast<const E*>(packed ? a.xc : a.x);
  const int64_t ldx = packed ? a.ldxc : a.ldx;
  int tp, tq;
  tile_coords((int)blockIdx.x, (int)gridDim.x, tiles_p, tiles_q, 8, 8, tp, tq);
  const int64_t t0 = (int64_t)tq * kSmallTile;
  if (a.row0 + t0 >= rows) return;
  constexpr int kParts = is_pair<T>::value ? 2 : 1;
  const int64_t v = (a.v0 - a.wv0) + (int64_t)tp * kSmallTile;
  typedef typename std::conditional<WF32, float, E>::type W;
  constexpr int kRowsOf = WF32 ? 1 : kParts;  // (fp32: one part, which is both)
  const W* w = reinterpret_cast<const W*>(a.w);
  SmallPipe<T, WVH, true, false, 4, 1, false, WF32> pipe;
  f32x16_t acc[kNB][1];
  pipe.run(w + (WVH ? v * a.ldw : v), WVH ? matrix_end<W>(w, a.Vw, a.ldw, a.H) : matrix_end<W>(w, kRowsOf * a.H, a.ldw, a.Vw), a.ldw,
           x + (a.row0 + t0) * ldx, matrix_end<E>(x, rows, ldx, kParts == 2 ? a.x_lo + a.H : a.H), ldx, a.H,
           (int)small_logit_ktiles(a.H, kParts == 2 ? 3 : 1), WF32 ? 0 : a.H * a.ldw * 2, a.x_lo * 2, lds, acc);
  // (with the sums of the persistent kernel, bit for bit: by columns but in the tile of 256 columns that straddles the end)
  const int64_t slice_v0 = a.v0 + (int64_t)tp * kSmallTile;
  const int64_t tw = t0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * kBlk;
  if (slice_v0 / kTile * kTile + kTile <= a.V) {
    FwdColumnState st;
#pragma unroll
    for (int slot = 0; slot < 16; ++slot) fwd_epilogue_slot<T, 0, MON, 1>(a, st, acc, slice_v0, tw, slot);
    const int lane = threadIdx.x & 63;
    const int64_t tok = a.row0 + tw + (lane & 31), yy = tok < rows ? a.y[tok] : a.ignore_index, rel = yy - slice_v0;
    const bool here = yy != a.ignore_index && rel >= 0 && rel < kWaveTile && ((rel >> 2) & 1) == (lane >> 5);
    fwd_store_target<1>(a, acc, tok, 0, here ? (int)rel : -1);
  } else {
    fwd_epilogue<T, true, MON, 1>(a, rows, acc, slice_v0, tw);
  }
}

// The seven quantities that the row merge sums over tokens (the fifth is a maximum) are laid out [..][8] in doubles and summed
// with one quantity to a lane: lane l of a wave takes quantity l % 8 of every eighth row from l / 8 on, so that a thread
// holds one double and not seven.
constexpr int kMaxAt = 4, kSums = 7;
LCE_DEV double join_sums(int q, double v, double o) { return q == kMaxAt ? fmax(v, o) : v + o; }
LCE_DEV double no_sum(int q) { return q == kMaxAt ? -INFINITY : 0.0; }
// Over the eight lanes of a wave that hold the same quantity, in a fixed order; the same in all of them.
LCE_DEV double wave_join(int q, double v) {
#pragma unroll
  for (int d = 8; d < 64; d <<= 1) v = join_sums(q, v, __shfl_xor(v, d));
  return v;
}

// Row merge: one workgroup = 64 tokens (lanes) x 16 strided groups of slices (waves).  Bound by latency: a few
// workgroups (64 for a chunk of 4096 rows), each a chain of batches of 8 loads in flight, so a token's slices go to 16 waves.
// Against 4 waves, us a launch: 394 slices 9 / 13 (64 workgroups) and 6.7 / 10.4 (4), 512 slices 10 / 17 (64), 1002 slices
// with monitoring 46 / 80 (128), 32 slices 5.0 / 4.0 (4), 8 slices 5.1 / 4.7 (256): what 16 cost at few slices is less than a
// second variant would be worth.
//   No more than half of the registers that 16 waves leave a thread are used (52 of 128): loops over the groups' results in
// LDS are unrolled by four, and the seven sums go one to a lane.  (Unrolled whole, with seven doubles in every lane, the
// kernel spilled 16 of them to memory.)
//   The block sums are added up by a launch of its own (below).  Folded into the last workgroup to be done -- a fence, a count
// in memory, a second fence -- they cost 4.5 us on 4 workgroups, 6.5 on 64 and 10 on 256, against 2.3 to 5 for the launch.
//   FINAL: one workgroup has all the tokens there are and goes on to the final sums, with barriers alone in between: no second
// launch for the smallest calls, which wait for the host (a launch is 3 of the 35 us of a loss alone).  Up to 64 tokens it has
// their block (394 slices: 6.9 us against 6.4 + 2.3), up to 256 all four blocks of a tile, four waves each, which one compute
// unit reads at the rate of several up to 128 slices: 32 slices 4.4 against 4.8 + 2.4, 64 4.8 / 4.5 + 2.2, 128 6.3 / 4.9 + 2.3,
// but 256 9.8 / 5.4 + 2.2 and 394 13.2 / 6.8 + 3.7.
constexpr int kMergeWaves = 16;
constexpr int kOneTileBlocks = kTile / kMergeRows;

// From the totals of the seven quantities in lanes 0 .. 6 of a wave to the five scalars and the count.
LCE_DEV void store_results(const FwdArgs& a, double v) {
  const double ce_sum = __shfl(v, 0), zr_sum = __shfl(v, 1), ent_sum = __shfl(v, 2), nrm_sum = __shfl(v, 3);
  const double z_max = __shfl(v, kMaxAt), R = __shfl(v, 5);  // 0 valid labels -> 0/0 = NaN, as F.cross_entropy gives
  // Labels outside [0, V) that are not ignore_index have no column to match; the reference lets
  // them contribute lse alone, silently.  Here they turn the loss into NaN (F.cross_entropy
  // raises a device-side assert for them) -- visible to the caller, no synchronisation needed.
  const bool bad_labels = __shfl(v, 6) != 0.0;
  if ((threadIdx.x & 63) == 0) {
    const double ce = ce_sum / R, zr = zr_sum / R;
    a.out5[0] = bad_labels ? __builtin_nanf("") : (float)(ce + (double)a.z_reg * zr);
    a.out5[1] = (float)zr;
    a.out5[2] = a.monitoring ? (float)z_max : 0.f;
    a.out5[3] = a.monitoring ? (float)(ent_sum / R) : 0.f;
    a.out5[4] = a.monitoring ? (float)(nrm_sum / (double)a.N) : 0.f;
    a.n_valid[0] = (int64_t)R;
  }
}

// BLOCKS: blocks of 64 tokens in a workgroup, kMergeWaves / BLOCKS waves for each.
template <int BLOCKS, bool FINAL>
__global__ __launch_bounds__(64 * kMergeWaves) void fwd_rows_kernel(const FwdArgs a) {
  constexpr int G = kMergeWaves / BLOCKS;  // groups of slices
  __shared__ float sh_m[kMergeWaves][kMergeRows], sh_s[kMergeWaves][kMergeRows], sh_lse[BLOCKS][kMergeRows];
  __shared__ float sh_pz[kMergeWaves][kMergeRows], sh_sq[kMergeWaves][kMergeRows], sh_mx[kMergeWaves][kMergeRows];
  __shared__ double sh_q[BLOCKS * kMergeRows][kSums + 2];  // (rows of 9: those of 8 lanes that write together are in different banks)
  __shared__ double sh_fin[BLOCKS][8];
  const int r = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int block = wave / G, g = wave % G, w0 = block * G;  // block of the workgroup, group of slices, the block's first wave
  const int64_t tokl = ((int64_t)blockIdx.x * BLOCKS + block) * kMergeRows + r;  // row inside the chunk of this launch
  const int64_t tok = a.row0 + tokl;  // < Np; rows that do not exist only keep the block sums aligned
  const int64_t rows = a.n_rows ? packed_rows(a.n_rows, a.N) : a.N;
  const bool exists = tok < rows;
  // packed rows: lse goes back to the token's own place; tokens that were dropped get 0 (as every token with an
  // ignored label does, below)
  if (a.perm != nullptr && g == 1 && tok < a.N && a.y0[tok] == a.ignore_index) a.lse[tok] = 0.f;
  const int nslices = (int)(a.Vp / kChunkV);

  // Online (max, sum) merge of this group's slices, 8 at a time so that the loads of a
  // batch are in flight together (a slice without a single valid column holds -inf and
  // contributes exp2(-inf) = 0).
  float M = -INFINITY, S = 0.f;
  for (int c0 = g; c0 < nslices; c0 += 8 * G) {
    float l[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + G * u;
      l[u] = c < nslices ? a.part_lse[(int64_t)c * a.nc + tokl] : -INFINITY;
    }
    float mb = l[0];
#pragma unroll
    for (int u = 1; u < 8; ++u) mb = fmaxf(mb, l[u]);
    if (mb == -INFINITY) continue;
    float sb = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) sb += fast_exp2((l[u] - mb) * kLog2e);
    const float Mn = fmaxf(M, mb);
    S = S * fast_exp2((M - Mn) * kLog2e) + sb * fast_exp2((mb - Mn) * kLog2e);
    M = Mn;
  }
  sh_m[wave][r] = M;
  sh_s[wave][r] = S;
  __syncthreads();
  if (g == 0) {
    float Mt = sh_m[w0][r], St = 0.f;
#pragma unroll 4
    for (int i = 1; i < G; ++i) Mt = fmaxf(Mt, sh_m[w0 + i][r]);
#pragma unroll 4
    for (int i = 0; i < G; ++i)
      if (sh_s[w0 + i][r] != 0.f) St += sh_s[w0 + i][r] * fast_exp2((sh_m[w0 + i][r] - Mt) * kLog2e);
    const float lse = Mt + fast_log(St);
    sh_lse[block][r] = lse;
    if (a.lse_rows != nullptr) a.lse_rows[tok] = lse;
    // lse[i] of a token with an ignored label is 0, whether its row was computed (all rows are when they are not
    // packed) or not: a caller sees one thing.  (sh_lse keeps the value: logit_entropy is taken over valid rows only,
    // and the backward never looks at the lse of such a token.)
    if (exists) a.lse[a.perm != nullptr ? packed_token(a.perm, tok, a.N) : tok] = a.y[tok] != a.ignore_index ? lse : 0.f;
  }
  if (a.monitoring) {
    __syncthreads();
    const float lse = sh_lse[block][r];
    float pz = 0.f, sq = 0.f, mx = -INFINITY;
    for (int c0 = g; c0 < nslices; c0 += 8 * G) {
      float pl[8], pp[8], ps[8], pm[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int c = c0 + G * u;
        const bool in = c < nslices;
        const int64_t o = (int64_t)(in ? c : 0) * a.nc + tokl;
        pl[u] = in ? a.part_lse[o] : -INFINITY;
        pp[u] = in ? a.part_pz[o] : 0.f;
        ps[u] = in ? a.part_sq[o] : 0.f;
        pm[u] = in ? a.part_max[o] : -INFINITY;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        pz = fmaf(pp[u], fast_exp2((pl[u] - lse) * kLog2e), pz);
        sq += ps[u];
        mx = fmaxf(mx, pm[u]);
      }
    }
    sh_pz[wave][r] = pz;
    sh_sq[wave][r] = sq;
    sh_mx[wave][r] = mx;
    __syncthreads();
  }
  if (g == 0) {
    const bool valid = exists && a.y[tok] != a.ignore_index;
    const double l = (double)sh_lse[block][r];
    double ent = 0.0, nrm = 0.0, mx = -INFINITY;
    if (a.monitoring && exists) {
      float pz = 0.f, sq = 0.f, m = -INFINITY;
#pragma unroll 4
      for (int i = 0; i < G; ++i) {
        pz += sh_pz[w0 + i][r];
        sq += sh_sq[w0 + i][r];
        m = fmaxf(m, sh_mx[w0 + i][r]);
      }
      mx = (double)m;
      ent = valid ? (double)(sh_lse[block][r] - pz) : 0.0;
      nrm = (double)sqrtf(sq);
    }
    double* mine = sh_q[block * kMergeRows + r];
    // tgt[tok] is written by the one tile that holds the target column; it is only read for a valid
    // label (for a valid label outside [0, V) nothing wrote it -- and the loss is NaN anyway)
    mine[0] = valid ? l - (double)a.tgt[tok] : 0.0;
    mine[1] = valid ? l * l : 0.0;
    mine[2] = ent;
    mine[3] = nrm;
    mine[kMaxAt] = mx;
    mine[5] = valid ? 1.0 : 0.0;
    // a label that is neither ignore_index nor a column of W: poisons the loss (below)
    mine[6] = (valid && (a.y[tok] < 0 || a.y[tok] >= a.V)) ? 1.0 : 0.0;
    mine[kSums] = 0.0;
    __threadfence_block();  // (written and read by this wave alone)
    __builtin_amdgcn_wave_barrier();
    const int q = r & 7;
    double v = no_sum(q);
#pragma unroll
    for (int i = 0; i < kMergeRows / 8; ++i) v = join_sums(q, v, sh_q[block * kMergeRows + i * 8 + (r >> 3)][q]);
    v = wave_join(q, v);
    if (!FINAL) {
      if (r < kSums) reinterpret_cast<double*>(a.blk)[(a.row0 / kMergeRows + (int64_t)blockIdx.x) * 8 + r] = v;
    } else if (r < 8) {
      sh_fin[block][r] = v;
    }
  }
  if constexpr (FINAL) {  // the final sums, in the order of fwd_final_kernel
    __syncthreads();
    if (wave != 0) return;
    const int q = r & 7, b = r >> 3;
    store_results(a, wave_join(q, b < BLOCKS ? sh_fin[b][q] : no_sum(q)));
  }
}

// The block sums of all chunks into the five scalars, in a fixed order.  Bound by latency: one workgroup, a quantity to a lane
// as above, eight workgroups' sums in one 512-byte load of a wave.
__global__ __launch_bounds__(64 * kMergeWaves) void fwd_final_kernel(const FwdArgs a) {
  constexpr int G = kMergeWaves;
  const int r = threadIdx.x & 63, g = threadIdx.x >> 6;
  const double* blk = reinterpret_cast<const double*>(a.blk);
  const int64_t nblk = a.Np / kMergeRows;
  __shared__ double sh_fin[G][8];
  const int q = r & 7;
  double v = no_sum(q);
  if (q < kSums) {
#pragma unroll 4
    for (int64_t b = threadIdx.x >> 3; b < nblk; b += 8 * G) v = join_sums(q, v, blk[b * 8 + q]);
  }
  v = wave_join(q, v);
  if (r < 8) sh_fin[g][r] = v;
  __syncthreads();
  if (g != 0) return;
  v = no_sum(q);
#pragma unroll
  for (int i = 0; i < G / 8; ++i) v = join_sums(q, v, sh_fin[i * 8 + (r >> 3)][q]);
  v = wave_join(q, v);
  store_results(a, v);
}

template <class T, int TAIL, bool KMASK, bool WVH, bool MON>
hipError_t launch_one(const FwdArgs& a, int64_t tiles, hipStream_t s) {
  auto kern = fwd_tiles_persistent_kernel<T, TAIL, KMASK, WVH, MON>;
  static LdsOptIn optin;
  hipError_t e = optin.ensure(reinterpret_cast<const void*>(kern), kMainloopLds);
  if (e != hipSuccess) return e;
  const int grid = (int)(tiles < a.num_cus ? tiles : a.num_cus);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), kMainloopLds, s, a);
  return hipGetLastError();
}

// All tile columns of the vocabulary in one launch.
template <class T, bool WVH, bool MON> hipError_t launch_persistent(const FwdArgs& a, hipStream_t s) {
  const int64_t left = a.Np - a.row0;  // token tiles of this chunk at most
  const int64_t here = left < a.nc ? left : a.nc, there = a.N - a.row0, rows = here < there ? here : there;
  if constexpr (!is_pair<T>::value) {
    if (a.H <= kNarrowHidden && a.small_wgs > 0 && a.w_dtype != DT_F32) return launch_fwd_narrow(a, rows, s);
  }
  if (a.w_dtype == DT_F32) {  // read as it is (fwd_reads_f32)
    if constexpr (is_pair<T>::value && MON) {
      return hipErrorInvalidValue;
    } else {
      const int tiles_p = (int)(pad_to(a.vw, kTile) / kSmallTile), tiles_q = (int)((rows + kSmallTile - 1) / kSmallTile);
      hipLaunchKernelGGL((fwd_small_kernel<T, WVH, MON, true>), dim3((unsigned)(tiles_p * tiles_q)), dim3(kThreads), kSmallLds, s, a, tiles_p,
                         tiles_q);
      return hipGetLastError();
    }
  }
  if (few_logit_tiles(rows, a.vw, small_logit_ktiles(a.H, products_of(a.x_dtype)), a.small_wgs)) {
    const int tiles_p = (int)(pad_to(a.vw, kTile) / kSmallTile), tiles_q = (int)((rows + kSmallTile - 1) / kSmallTile);
    hipLaunchKernelGGL((fwd_small_kernel<T, WVH, MON, false>), dim3((unsigned)(tiles_p * tiles_q)), dim3(kThreads), kSmallLds, s, a, tiles_p,
                       tiles_q);
    return hipGetLastError();
  }
  const int64_t tq = (left < a.nc ? left : a.nc) / kTile, full = a.vw / kTile;
  const bool exact_k = (is_pair<T>::value ? padded_k_pair(a.H) : padded_k(a.H)) == a.H;  // the K tiles cover H exactly: no K mask needed
  const bool tail = a.vw % kTile != 0;        // a column that straddles V
  if (full == 0) return launch_one<T, kTailOnly, true, WVH, MON>(a, tq, s);
  if (tail)
    return exact_k ? launch_one<T, kWithTail, false, WVH, MON>(a, (full + 1) * tq, s)
                   : launch_one<T, kWithTail, true, WVH, MON>(a, (full + 1) * tq, s);
  return exact_k ? launch_one<T, kNoTail, false, WVH, MON>(a, full * tq, s) : launch_one<T, kNoTail, true, WVH, MON>(a, full * tq, s);
}

template <class T, bool WVH> hipError_t launch_layout(const FwdArgs& a, hipStream_t s) {
  return a.monitoring ? launch_persistent<T, WVH, true>(a, s) : launch_persistent<T, WVH, false>(a, s);
}

}  // namespace

hipError_t launch_fwd_tiles(const FwdArgs& a, hipStream_t s) {
  // (An fp32 weight arrives here as a copy in the compute type or, for few tokens, as it is; fp32 activations as the packed copy in
  // pairs.)
  const bool as_x = a.w_dtype == a.x_dtype || a.w_dtype == DT_F32;
  if (a.x_dtype == DT_BF16 && as_x) return a.w_vh ? launch_layout<BF16, true>(a, s) : launch_layout<BF16, false>(a, s);
  if (a.x_dtype == DT_F16 && as_x) return a.w_vh ? launch_layout<F16, true>(a, s) : launch_layout<F16, false>(a, s);
  if (a.x_dtype == DT_PAIR && as_x && !a.w_vh) return launch_layout<BF16P, false>(a, s);
  return hipErrorInvalidValue;
}

// Blocks of the row merge that forms the final sums as well (see fwd_rows_kernel), or 0.
static int final_merge_blocks(const FwdArgs& a) {
  if (a.Np != kTile) return 0;
  if (a.N <= kMergeRows && a.lse_rows == nullptr) return 1;  // (lse_rows is read for all rows of a tile)
  return a.Vp / kChunkV <= 128 ? kOneTileBlocks : 0;
}

hipError_t launch_fwd_rows(const FwdArgs& a, hipStream_t s) {
  const int64_t left = a.Np - a.row0;
  const int whole = final_merge_blocks(a);
  auto kern = whole == 0 ? fwd_rows_kernel<1, false> : whole == 1 ? fwd_rows_kernel<1, true> : fwd_rows_kernel<kOneTileBlocks, true>;
  const int64_t grid = whole != 0 ? 1 : (left < a.nc ? left : a.nc) / kMergeRows;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * kMergeWaves), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_fwd_final(const FwdArgs& a, hipStream_t s) {
  if (final_merge_blocks(a) != 0) return hipSuccess;
  hipLaunchKernelGGL(fwd_final_kernel, dim3(1), dim3(64 * kMergeWaves), 0, s, a);
  return hipGetLastError();
}

}  // namespace lce
