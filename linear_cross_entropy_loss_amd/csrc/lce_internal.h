// Internal launch interface between the C ABI (lce_api.hip) and the kernel
// translation units.  Not installed; the public surface is include/lce.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <atomic>

namespace lce {

enum { DT_BF16 = 0, DT_F16 = 1, DT_F32 = 2 };
// Compute type of fp32 tensors inside the library: bf16 pairs (lce_gemm.h).
enum { DT_PAIR = 3 };

// The tile kernels use more dynamic LDS than a kernel gets by default and have to opt in
// (hipFuncAttributeMaxDynamicSharedMemorySize): once per kernel and device, not before every launch.  One object
// per kernel (a function-local static of its launcher); thread-safe.
struct LdsOptIn {
  std::atomic<uint64_t> done{0};  // bit d: set on device d (devices from 64 on are set every time)
  hipError_t ensure(const void* kernel, int bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64 && ((done.load(std::memory_order_acquire) >> dev) & 1)) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && dev >= 0 && dev < 64) done.fetch_or((uint64_t)1 << dev, std::memory_order_release);
    return e;
  }
};

// Columns of logits covered by one forward partial (one wave's slice of a tile).
constexpr int kChunkV = 128;
// Rows handled by one workgroup of the row-merge kernel.
constexpr int kMergeRows = 64;

// Shapes need not be multiples of the tile sizes: the kernels work on the padded
// extents below, operand loads past the real extents return zero (buffer range
// checks and a K mask), and the epilogues neither use logits of columns >= V nor
// store anything for rows >= N, columns >= V or hidden indices >= H.
constexpr int64_t pad_to(int64_t v, int64_t m) { return (v + m - 1) / m * m; }
constexpr int64_t padded_tokens(int64_t N) { return pad_to(N, 256); }   // token tiles; K tiles of the dW contraction
constexpr int64_t padded_vocab(int64_t V) { return pad_to(V, 256); }    // vocabulary tiles
constexpr int64_t padded_hidden(int64_t H) { return pad_to(H, 256); }   // hidden tiles of dx and dW
// K extent of the logit contraction: an even number of 64-wide K tiles, at least four
constexpr int64_t padded_k(int64_t H) { return pad_to(H, 128) < 256 ? 256 : pad_to(H, 128); }

// Pairs: three K tiles for each of these 64-wide ones, so two of them are enough
constexpr int64_t padded_k_pair(int64_t H) { return pad_to(H, 128); }
// Matrix products per K tile of the compute type.
constexpr int products_of(int dtype) { return dtype == DT_PAIR ? 3 : 1; }
// K tiles of the logit contraction on 128 x 128 tiles, which need no four of them (N=8192, H=128, V=8192: 60 us with four, 47 with two).
__host__ __device__ constexpr int64_t small_logit_ktiles(int64_t H, int products) { return products * (pad_to(H, 128) / 64); }

// Modelled time of a logit kernel for `rows` token rows, `cols` columns and `kt` 64-deep K tiles (times the products of a pair), us:
// on 128 x 128 tiles, one workgroup each (lce_gemm_small.h), or on the 256 x 256 tiles of the persistent kernels.  The latter start
// with 14 us of fetching their code, the former with 5; a round of 512 workgroups, two to a compute unit, takes 0.9 us a K tile and
// 3.4 for prologue and epilogue, one of up to 256 little more than half of that a K tile, a round of 256 x 256 tiles 1.2 and 5,
// less where it leaves compute units, and with them power, to the others.  Loss alone, bf16, us measured, 128 x 128 / 256 x 256:
// N=256, V=4096, H=256 8.7 / 18.4, H=4096 46 / 74; N=1536, V=2560, H=2048 24 / 46; N=4096, V=2048, H=256 12.5 / 18.7, H=2048
// 42 / 49; N=5120, V=2048, H=256 20 / 20, H=1024 35 / 33, H=2048 61 / 50; N=1999, V=10007, H=500 32 / 45; N=16384, V=1000, H=1024
// 45 / 42; N=2048, V=16384, H=768 64 / 53; N=4096, V=16384, H=256 60 / 52.
inline double small_logits_us(int64_t rows, int64_t cols, int64_t kt) {
  const int64_t n = (rows + 127) / 128 * (pad_to(cols, 256) / 128), full = n / 512, rest = n % 512;
  return 5.0 + (double)full * (0.9 * (double)kt + 3.4) + (rest == 0 ? 0.0 : (rest > 256 ? 0.9 : 0.5) * (double)kt + 3.4);
}
inline double persistent_logits_us(int64_t rows, int64_t cols, int64_t kt) {
  const int64_t n = (rows + 255) / 256 * (pad_to(cols, 256) / 256), full = n / 256, rest = n % 256;
  const double round = 1.2 * (double)(kt < 4 ? 4 : kt) + 5.0;
  return 14.0 + (double)full * round + (rest == 0 ? 0.0 : round / (1.0 + 0.9 * (1.0 - (double)rest / 256.0)));
}
// Whether a logit kernel runs on 128 x 128 tiles: up to two workgroups to a compute unit, for up to 128 tokens (of which the other
// tiles are half empty: N=48, V=100000, H=256 19 / 33, H=2048 94 to 102 / 110), and where the model puts them 8 % ahead (what it is
// off by).  `most`: two workgroups for each compute unit (FwdArgs::small_wgs; 0: never).
inline bool few_logit_tiles(int64_t rows, int64_t cols, int64_t kt, int most) {
  const int64_t n = (rows + 127) / 128 * (pad_to(cols, 256) / 128);
  if (most <= 0) return false;
  return n <= most || rows <= 128 || (n < (int64_t)1 << 28 && small_logits_us(rows, cols, kt) < 0.92 * persistent_logits_us(rows, cols, kt));
}

// Which tile columns of the vocabulary a logit kernel covers: full ones, the one(s) from the column that straddles the end of
// the vocabulary on, or both.
enum { kNoTail = 0, kTailOnly = 1, kWithTail = 2 };

struct FwdArgs {
  const void* x;
  const void* w;
  const int64_t* y;
  int64_t N, H, V, ldx, ldw;
  int64_t Np, Vp;  // padded_tokens(N), padded_vocab(V)
  // Token rows [row0, row0 + nc) covered by this launch (both multiples of 256): the forward works through the
  // rows in chunks of nc, so that the per-slice partials below are nc rows wide however many tokens there are.
  int64_t row0, nc;
  // Vocabulary columns [v0, v0 + vw) covered by this launch (v0 a multiple of 256), and the
  // window of W that the buffer `w` holds: columns [wv0, wv0 + Vw) of the weight, row stride ldw.
  // (`w` is the caller's matrix, wv0 = 0, Vw = V -- or a 16-bit copy of one slab of an fp32 weight; an fp32 weight
  // itself for few tokens, w_dtype DT_F32.)
  int64_t v0, vw, wv0, Vw;
  // w_vh != 0: the weight is stored with the vocabulary as its row index, w[v * ldw + h] (the buffer `w` then
  // holds ROWS [wv0, wv0 + Vw)); otherwise w[h * ldw + v].
  int w_vh;
  int x_dtype, w_dtype;  // compute type = x_dtype (bf16 / f16 / pairs)
  // Pairs: x is rows of [hi | lo], the lo part x_lo elements behind the hi part, and w is H rows of hi, then H rows of lo.
  int64_t x_lo;
  int64_t ignore_index;
  float scale, z_reg;
  int monitoring;
  // Packed rows (tokens with an ignored label dropped; null / unused when the call works on all rows):
  // *n_rows (device) rows are worked on; when *n_rows != N they are the rows of xc (row stride ldxc) and
  // `y` holds their labels; perm[j] is the token that packed row j came from, y0 the labels of all tokens.
  const int64_t* n_rows;
  const void* xc;
  int64_t ldxc;
  const int* perm;
  const int64_t* y0;
  int num_cus;  // compute units of the device: grid size of the persistent kernels
  int small_wgs;  // few_logit_tiles: 0 where the caller has limited the workgroups of a launch
  int live;     // bands of W that the XCDs keep in flight together (lce_gemm.h, tile_coords)
  // outputs / scratch
  float* lse;        // [N]
  float* out5;       // [5]
  int64_t* n_valid;  // [1]
  float* part_lse;   // [Vp/128][nc]  per-slice logsumexp (-inf for a slice with no valid column), rows of the current chunk
  float* part_max;   // [Vp/128][nc]  per-slice max            (monitoring)
  float* part_pz;    // [Vp/128][nc]  per-slice sum softmax*z  (monitoring)
  float* part_sq;    // [Vp/128][nc]  per-slice sum z^2        (monitoring)
  float* tgt;        // [Np]          target logit (written for tokens whose label is a column of W)
  float* blk;        // [Np/64][8]    per-merge-block partial sums (doubles, seven of a block's eight)
  float* lse_rows;   // [Np] or null  lse of every row in the order the tile kernels see them (packed rows), whatever its label
};

struct BwdArgs {
  const void* x;
  const void* w;
  const int64_t* y;
  const float* lse;
  const int64_t* n_valid;
  const float* grad_out;
  int64_t N, H, V, ldx, ldw, lddx, lddw;
  int64_t Np, Hp;  // padded_tokens(N), padded_hidden(H)
  int x_dtype, w_dtype, dx_dtype, dw_dtype;  // compute type = x_dtype, as in FwdArgs
  int64_t x_lo;  // pairs, as in FwdArgs
  int64_t ignore_index;
  float scale, z_reg;
  void* dx;
  void* dw;
  // slab being processed
  int64_t v0, vs;   // first column and padded width (multiple of 256) of the vocabulary slab
  int64_t vw;       // columns of the slab that exist: min(vs, V - v0)
  int64_t wv0, Vw;  // `w` holds columns [wv0, wv0 + Vw) of the weight (the whole matrix, or a 16-bit copy of this slab)
  // w_vh != 0: weight and dW are stored with the vocabulary as their row index, w[v * ldw + h], dw[v * lddw + h]
  // (and the buffer `w` holds ROWS [wv0, wv0 + Vw)); otherwise w[h * ldw + v], dw[h * lddw + v].
  int w_vh;
  // Staged dz in the compute type (exact zeros outside N x vw), stored in blocks of 256 rows x 64 columns,
  // [rows / 256][vs / 64][256][64] (dz_block_offset below): the 64-deep K tiles of the dx contraction (K = v) are
  // consecutive 32 KiB blocks, the K tiles of the dW contraction (K = tokens) quarters of four neighbouring blocks,
  // and a token's 64 columns of a group are one 128-byte line.  dz_rows = Np rows.  Pairs: the block of the lo parts follows
  // each block of hi parts.
  void* dz;
  int64_t dz_rows;
  float* dx_acc;    // [Np][Hp] fp32 running dx (null when there is a single slab)
  // dx: tiles of a last, mostly idle round of workgroups are cut along K instead (planned on the device,
  // see lce_bwd_dx.hip); the segments' partial sums meet in dx_part, dx_tail_blocks() blocks of 256 x 256
  // floats, and a small kernel adds them in a fixed order.  dx_grid = workgroups of the tile kernel.
  int dx_grid;
  float* dx_part;
  // The same for dW (K = tokens): dw_part holds dw_tail_blocks() blocks, dw_grid = workgroups of the tile kernel.
  int dw_grid;
  float* dw_part;
  // The staged dz = softmax * gain - onehot is multiplied by 2^dz_shift before it is rounded to the 16-bit compute
  // type, and the dx / dW kernels fold 2^-dz_shift into their final factor.  bf16 has fp32's exponent range and
  // needs none (0); in fp16 the softmax probabilities of a large vocabulary (of order 1/V) would fall below the
  // normal range (6.1e-5) and lose precision bit by bit -- with 10 they stay normal down to 6e-8, while
  // |dz| * 2^10 stays below fp16's maximum for any gain = 1 + 2 * z_reg * lse below 63: bwd_dz clamps the gain to
  // +-63 when the factor is in place, and the host takes 0 instead when z_reg > 1/32, where logits of ordinary size
  // (|lse| < 992 at 1/32) would already reach that.
  int dz_shift;
  int first, last;  // slab position
  int num_cus;      // compute units of the device: grid size of the persistent kernels
  int small_wgs;    // as in FwdArgs
  int live;         // bwd_dz: bands of W that the XCDs keep in flight together (lce_gemm.h, tile_coords)
  // Packed rows (tokens with an ignored label dropped; n_rows == null: the call works on all rows).
  // *n_rows (device) rows are worked on.  When *n_rows != N they are the rows of xc (row stride ldxc) and
  // row j of dx belongs to token perm[j]: the dx kernels store it there themselves, or -- dxc != null, a dx
  // of 2 GiB or more -- into dxc (row stride lddxc), from where it is moved afterwards.  In either case `y`
  // and `lse` hold the labels / lse of the packed rows.
  const int64_t* n_rows;
  const int* perm;
  const void* xc;
  int64_t ldxc;
  void* dxc;
  int64_t lddxc;
  // One pass over the logits (lce_forward_backward): the problem is a chunk of token rows against the whole
  // vocabulary, and the logit kernel (launch_fwd_stage) leaves, instead of dz,
  //     e[token][v] = 2^dz_shift * exp(z[token][v] - m[token][v / 128])
  // in the stage, m = the largest logit of the token in that slice of 128 columns, together with the forward's
  // per-slice partials of the chunk: part_lse, part_max = m ([Vp/128][nc], as in FwdArgs) and the target logits
  // tgt (first row of the chunk).  Once the rows' lse are known, launch_stage_scale turns e into dz in
  // place, or the dx and dW kernels do on the way to LDS (dx_f, dw_f below).
  float* part_lse;
  float* part_max;
  float* part_pz;  // both null, or the monitoring partials of FwdArgs as well
  float* part_sq;
  float* tgt;
  int64_t nc;
  // Not null: the stage holds e, and the dx and dW kernels turn it into dz on its way to LDS, with one factor per token
  // and slice of 128 columns, [Vp/128][nc]: dx_f has the 256 tokens of a tile in the order (token % 32) * 8 + token / 32,
  // dw_f the 64 of a K tile in the order (token % 8) * 8 + token / 8, so that what one thread needs lies together.
  const float* dx_f;
  const float* dw_f;
  // rows of dx always go to the tokens perm[] names (the rows of a chunk can be all there and still not be the
  // tokens of the same numbers)
  int perm_always;
  // 16-bit dW summed over chunks of token rows: the fp32 sums are kept as 16-bit halves, the upper ones in dw
  // itself, the lower ones in dw_plane (one block of 256 x 256 halves per tile of dW); dw_plane_hi takes the upper
  // halves of the tiles that the edge of the matrix cuts (null if there is none) -- see lce_bwd_dw.hip.
  // dw_acc: 0 = no sums over chunks (dW is stored as it comes), 1 = the sums are stored (first chunk), 2 = added
  // to, 5 = added to, and the result scaled and stored as dW (last chunk); 6, 7, 8 = the same three with only the
  // upper byte of each lower half kept (dw_plane: 256 x 256 bytes per tile; the sums are rounded at 24 bits).
  // fp32 dW: 3 = the sums times the final factor are stored to dw itself (first chunk), 4 = added to it.
  void* dw_plane;
  void* dw_plane_hi;
  int dw_acc;
  int vtail_all;  // the logit kernel for the tile column that straddles the end of the vocabulary takes every column
};

// Element offset of block (row tile, column group) of a dz stage that is `vs` columns wide.
constexpr int kDzBlockElems = 256 * 64;
__host__ __device__ inline int64_t dz_block_offset(int64_t row_tile, int64_t group, int64_t vs) {
  return (row_tile * (vs / 64) + group) * kDzBlockElems;
}

// Factor applied to dx and dW after their fp32 accumulation: grad_out * logit_scale / n_valid
// (linear_cross_entropy/ops.py:332, 443-447, 810), times the power of two that undoes the scaling of the staged
// dz.  With no valid label at all every dz is zero and the factor is taken as 0, so both
// gradients are exact zeros (what F.cross_entropy's backward gives for such a batch; the loss itself is NaN).
__device__ __forceinline__ float final_factor_of(const BwdArgs& a) {
  const int64_t n = a.n_valid[0];
  const float unscale = __builtin_bit_cast(float, (127 - a.dz_shift) << 23);  // 2^-dz_shift
  return n > 0 ? a.grad_out[0] * a.scale / (float)n * unscale : 0.f;
}

hipError_t launch_fwd_tiles(const FwdArgs& a, hipStream_t s);
// Row merge of the current chunk (lse, per-block sums), and -- once, after the last chunk -- the final reduction (nothing to
// do there where the row merge was one workgroup's).
hipError_t launch_fwd_rows(const FwdArgs& a, hipStream_t s);
hipError_t launch_fwd_final(const FwdArgs& a, hipStream_t s);
hipError_t launch_bwd_dz(const BwdArgs& a, hipStream_t s);
// The logit kernel of lce_forward_backward and the pass that follows the row merge (see BwdArgs).
hipError_t launch_fwd_stage(const BwdArgs& a, hipStream_t s);
hipError_t launch_stage_scale(const BwdArgs& a, hipStream_t s);
// The same for pairs, of which the stage holds the logits themselves.
hipError_t launch_stage_pairs(const BwdArgs& a, hipStream_t s);
// The same with the factors only worked out (dx_f and dw_f of BwdArgs), and the slice of each token's target column
// rewritten.
hipError_t launch_stage_factors(const BwdArgs& a, hipStream_t s);
// t[r][c] *= g[0] (device scalar), in fp32; nothing is touched when g[0] == 1.  Rows on 16-byte boundaries.
hipError_t launch_scale_rows(void* t, int dtype, int64_t rows, int64_t cols, int64_t ld, const float* g, int num_cus,
                             hipStream_t s);
// The same for two matrices (either may be absent: t null) in one launch, by the factor g[0] / d[0] (d null: g[0]).
struct ScaleTask {
  void* t;
  int dtype;
  int64_t rows, cols, ld;
};
hipError_t launch_scale_two(const ScaleTask& t0, const ScaleTask& t1, const float* g, const float* d, int num_cus, hipStream_t s);
hipError_t launch_bwd_dx(const BwdArgs& a, hipStream_t s);
hipError_t launch_bwd_dw(const BwdArgs& a, hipStream_t s);
// dst[h][c] = 16-bit rounding of src[h * ld + v0 + c] for c < vw, 0 for vw <= c < dst_ld; h < H.
// compute_dtype: DT_BF16, DT_F16 or DT_PAIR: dst then has 2 H rows, [bf16 hi ; bf16 lo] of the fp32 values.
hipError_t launch_convert_w_slab(const float* src, int64_t ld, int64_t H, int64_t v0, int64_t vw, void* dst,
                                 int64_t dst_ld, int compute_dtype, hipStream_t s);
// The same for a weight stored (V, H) row-major (H a multiple of 8): rows [v0, v0 + vw) go to dst[vw][dst_ld].
hipError_t launch_convert_w_rows(const float* src, int64_t ld, int64_t H, int64_t v0, int64_t vw, void* dst,
                                 int64_t dst_ld, int compute_dtype, hipStream_t s);

// Row count / row -> token map of the packed rows as the kernels read them from device memory, forced
// into range: a call restricted to some phases on a workspace whose packing pre-pass did not run must
// give wrong numbers, not wild addresses.
__device__ __forceinline__ int64_t packed_rows(const int64_t* n_rows, int64_t N) {
  if (n_rows == nullptr) return N;  // this call works on all rows
  const int64_t r = n_rows[0];
  return r < 0 ? 0 : (r > N ? N : r);
}
__device__ __forceinline__ int64_t packed_token(const int* perm, int64_t j, int64_t N) {
  const int64_t t = perm[j];
  return t < 0 ? 0 : (t >= N ? N - 1 : t);
}

// dst row r = row_bytes bytes at src + r * src_ld (2-byte units, any 2-byte address), then zeros to dst_ld (lce_convert.hip).
hipError_t launch_pad_rows(const void* src, int64_t src_ld, int64_t rows, int64_t row_bytes, void* dst, int64_t dst_ld,
                           hipStream_t s);

// dst[r][c] = src[c * src_ld + r], c < cols, then zeros to dst_ld; es-byte elements, strides in elements (lce_convert.hip).
hipError_t launch_transpose_rows(const void* src, int64_t src_ld, int64_t rows, int64_t cols, int es, void* dst, int64_t dst_ld,
                                 hipStream_t s);

// *out = the largest power of two not above the number of labels that are not ignore_index (lce_compact.hip).
hipError_t launch_stand_in(const int64_t* y, int64_t N, int64_t ignore_index, float* out, hipStream_t s);

// Packing of the tokens whose label is not ignore_index (lce_compact.hip).  `cnt` holds one int per
// compact_segments(N); perm and yc hold N entries each: the kept tokens first (*n_rows of them), then the dropped ones.
// chunks > 0 (at most 1024), with `nc` rows each: chunk_rows[c] = rows of chunk c among the packed rows, min(max(*n_rows - c * nc, 0), nc);
// chunk_rows[1024 + c] = the same among all N rows.
int64_t compact_segments(int64_t N);
hipError_t launch_compact_labels(const int64_t* y, int64_t N, int64_t ignore_index, int* cnt, int64_t* n_rows,
                                 int* perm, int64_t* yc, hipStream_t s, int64_t nc = 0, int chunks = 0,
                                 int64_t* chunk_rows = nullptr);
// xc[j] = x[perm[j]] for j < *n_rows, in 16-byte pieces of rows ldxc_bytes long (skipped when *n_rows == N);
// row_bytes = bytes of a row that hold elements (nothing past them is read of the last row of x);
// lse_c[j] = lse[perm[j]] when lse is not null (always).  `always`: the rows are copied also when *n_rows == N.
hipError_t launch_gather_rows(const void* x, int64_t ldx_bytes, int64_t row_bytes, const int* perm,
                              const int64_t* n_rows, int64_t N, void* xc, int64_t ldxc_bytes, const float* lse,
                              float* lse_c, int num_cus, hipStream_t s, bool always = false);
// fp32 activations: xc[j] = [hi | lo] of x[perm[j]] as bf16 pairs, each part half of the row stride ldxc (a multiple of 16)
// and zero-padded to it.  Always made, also when no token is dropped; perm / n_rows may be null (all N rows in their
// order).  Strides in elements; rows of x on 16-byte boundaries.
hipError_t launch_gather_rows_split(const float* x, int64_t ldx, int64_t H, const int* perm, const int64_t* n_rows,
                                    int64_t N, void* xc, int64_t ldxc, const float* lse, float* lse_c, int num_cus,
                                    hipStream_t s);
// dx[perm[j]] = dxc[j] for j < *n_rows (skipped when dxc is null) and dx[i] = 0 for every token i with
// y[i] == ignore_index, in 8-byte pieces covering row_bytes; nothing when *n_rows == N.
hipError_t launch_scatter_rows(const void* dxc, int64_t lddxc_bytes, const int* perm, const int64_t* n_rows,
                               int64_t N, const int64_t* y, int64_t ignore_index, void* dx, int64_t lddx_bytes,
                               int64_t row_bytes, int num_cus, hipStream_t s);

// Bands to keep in flight (tile_coords in lce_gemm.h) for P bands of 8 tiles of 256 rows and `k_bytes` bytes per row:
// as many of 8, 4, 2, 1 as stay within a quarter of the Infinity Cache together (measured at H = 8192, where a band is
// 32 MiB: bwd_dz 27.5 / 26.4 / 25.0 / 25.2 ms with 8 / 4 / 2 / 1 bands in flight; no difference at H = 4096; 8 best at H = 2048).
inline int live_bands(int64_t k_bytes) {
  const int64_t band_bytes = 8 * 256 * k_bytes;
  int live = 8;
  while (live > 1 && live * band_bytes > ((int64_t)64 << 20)) live /= 2;
  return live;
}

// dx of one slab: at most (Np/256) x (Hp/256) tiles, K = vs columns.  Upper bound on the 256 x 256 fp32
// blocks of partial sums that the device-side plan of the dx kernel can ask for (0: it never splits).
constexpr int kTailBlocks = 256;
// most segments per tile: a power of two that leaves at least 16 K tiles per segment
__host__ __device__ inline int64_t max_k_segments(int64_t kt) {
  int64_t s = 1;
  while (kt / (s * 2) >= 16 && s * 2 <= kTailBlocks) s *= 2;
  return s;
}
// Segments that each of r tiles with kt K tiles is cut into on G workgroups: as many as keep every workgroup busy once.  (1: not
// cut.)
__host__ __device__ inline int k_segments(int r, int G, int kt) {
  const int cap = G < kTailBlocks ? G : kTailBlocks;
  if (r <= 0 || 2 * r > cap) return 1;
  const int s = cap / r, most = (int)max_k_segments(kt);
  return s < most ? s : most;
}
// A segment's K tiles, of kt (an even number) in s segments: even numbers of them, as equal as that goes.
__host__ __device__ inline int segment_start(int seg, int s, int kt) {
  const int base = kt / 2 / s, rest = kt / 2 - base * s;
  return 2 * (seg * base + (seg < rest ? seg : rest));
}
// (`products`: products_of the compute type)
inline int64_t dx_tail_blocks(int64_t Np, int64_t Hp, int64_t vs, int products) {
  const int64_t s = max_k_segments(products * vs / 64);
  if (s == 1) return 0;
  const int64_t most = (Np / 256) * (Hp / 256) * s;
  return most < kTailBlocks ? most : kTailBlocks;
}
// Whether T output tiles on G workgroups end in a last round that the kernels cut along K (at most half full).
inline bool has_split_tail(int64_t T, int64_t G) {
  const int64_t r = T % G, cap = G < kTailBlocks ? G : kTailBlocks;
  return r > 0 && r * 2 <= cap;
}
// Whether every one of T output tiles with `kt` K tiles each is a tail tile of the device-side plans (dx_plan,
// dw_plan): fewer tiles than workgroups, few enough to split, and a K extent long enough for two segments.
inline bool all_tiles_are_tails(int64_t T, int64_t G, int64_t kt) {
  return T < G && has_split_tail(T, G) && kt / 2 >= 16;
}
// dW of one slab: (vs/256) x (Hp/256) tiles, K = at most Np tokens.  The same bound for the dW kernel.
inline int64_t dw_tail_blocks(int64_t Np, int64_t Hp, int64_t vs, int products) {
  const int64_t s = max_k_segments(products * Np / 64);
  if (s == 1) return 0;
  const int64_t most = (vs / 256) * (Hp / 256) * s;
  return most < kTailBlocks ? most : kTailBlocks;
}

// dx and dW of a single slab on 128 x 128 tiles, in one launch (lce_bwd_small.hip): workgroups [0, first_span) are the tiles of
// one gradient times its stretches of K, the rest those of the other.  part: one block of 128 x 128 floats for each stretch, those
// of dx (where it has several) first.  The plan is one for both gradients, whichever the caller wants, and for rows that are not
// packed: sums of the same tokens are then cut the same way in every call.
struct SmallGrads {
  int dw_first, first_span, dx_nseg, dx_blocks, dw_nseg, dw_blocks;
  double us;  // modelled time
  float* part;
};
constexpr int64_t kSmallBlockBytes = 128 * 128 * 4;
constexpr int kSmallSlots = 512;  // workgroups that the chip holds at a time, two to a compute unit
// When the last of na items of la K tiles and then nb of lb (<= la) ends on the slots, each going to the first free one.
inline double small_span(int64_t na, double la, int64_t nb, double lb) {
  const int64_t S = kSmallSlots;
  if (na + nb <= S) return la;
  int64_t busy = na % S;                       // slots with one item more than the others
  double low = (double)(na / S) * la, high = busy > 0 ? low + la : low;
  if (busy == 0) busy = S;
  int64_t left = nb;
  double end = high;
  // (slots that are level with the busiest after k more items of the other kind)
  while (left > 0) {
    const int64_t free_slots = S - busy;
    if (free_slots > 0 && low + lb <= high) {
      const int64_t rounds = (int64_t)((high - low) / lb), can = rounds * free_slots;
      if (left <= can) return end;
      left -= can;
      low += (double)rounds * lb;
      continue;
    }
    if (free_slots > 0 && low < high) {
      end = low + lb > end ? low + lb : end;
      left -= free_slots;
      if (left <= 0) return end;
      low = high;  // (those run a little behind the others from here on)
    }
    const int64_t rounds = left / S, rest = left - rounds * S;
    return high + (double)(rounds + (rest > 0 ? 1 : 0)) * lb;
  }
  return end;
}
// The stretches of K: as many of each gradient as give the shortest launch, with what their sums cost on top, and fit `most_blocks`.
// tx tiles of dx with kx units of K each, tw of dW with kw; stretches of whole pairs of `pair` units, `least` at the shortest; `item`:
// what prologue and epilogue of a workgroup take, in units; block: what a stretch's sums cost.
struct CutRule {
  int64_t tx, kx, tw, kw, pair, least;
  double products, item, block;
};
inline double plan_cuts(const CutRule& c, int64_t most_blocks, SmallGrads* g) {
  auto most = [&](int64_t t, int64_t k) -> int64_t {
    const int64_t by_length = k / c.least, by_slots = 4 * kSmallSlots / t;
    const int64_t m = by_length < by_slots ? by_length : by_slots;
    return m < 1 ? 1 : m;
  };
  auto length = [&](int64_t k, int64_t n) { return (double)(((k + c.pair - 1) / c.pair + n - 1) / n * c.pair) * c.products + c.item; };
  auto next = [](int64_t n) { return n < 16 ? n + 1 : n + n / 8; };
  memset(g, 0, sizeof(*g));
  double best = -1;
  const int64_t mx = most(c.tx, c.kx), mw = most(c.tw, c.kw);
  for (int64_t nx = 1; nx <= mx; nx = next(nx))
    for (int64_t nw = 1; nw <= mw; nw = next(nw)) {
      const int64_t bx = nx > 1 ? c.tx * nx : 0, bw = nw > 1 ? c.tw * nw : 0;
      if (bx + bw > most_blocks) continue;
      const double lx = length(c.kx, nx), lw = length(c.kw, nw);
      const bool wf = lw > lx;
      double t = wf ? small_span(c.tw * nw, lw, c.tx * nx, lx) : small_span(c.tx * nx, lx, c.tw * nw, lw);
      if (c.tx * nx + c.tw * nw <= kSmallSlots / 2) t *= 0.55;  // (one to a compute unit)
      if (bx + bw > 0) t += 200.0 * c.block + (double)(bx + bw) * c.block;
      if (best >= 0 && t >= best) continue;
      best = t;
      g->dw_first = wf;
      g->dx_nseg = (int)nx;
      g->dw_nseg = (int)nw;
      g->dx_blocks = (int)bx;
      g->dw_blocks = (int)bw;
    }
  return best;
}
// A unit is a K tile of 64.
inline SmallGrads plan_small_grads(int64_t N, int64_t H, int64_t V, int products, int64_t most_blocks) {
  const int64_t th = (H + 127) / 128;
  const CutRule c = {th * ((N + 127) / 128), pad_to(V, 128) / 64, th * ((V + 127) / 128), pad_to(N, 128) / 64, 2, 8, (double)products, 4.0, 0.03};
  SmallGrads g;
  const double t = plan_cuts(c, most_blocks, &g);
  // (a long launch runs into the power limit: the K tile's time goes from 0.9 us to 1.2)
  g.us = 5.0 + 0.9 * t * (1.0 + 0.35 * (t < 40.0 ? 0.0 : t > 200.0 ? 1.0 : (t - 40.0) / 160.0));
  return g;
}
// Hidden sizes up to this: no stage (lce_narrow.hip).  A unit is a tile of 128 rows that streams past the 128 that stay; a block of
// sums has 128 rows of whole K tiles.
constexpr int64_t kNarrowHidden = 128;
inline int64_t narrow_block_bytes(int64_t H) { return 128 * (H <= 64 ? 64 : 128) * 4; }
inline SmallGrads plan_narrow_grads(int64_t N, int64_t H, int64_t V, int64_t most_blocks) {
  const int64_t tok = (N + 127) / 128, voc = (V + 127) / 128;
  const CutRule c = {tok, voc, voc, tok, 1, 1, 1.0, 1.5, 0.0075};
  SmallGrads g;
  const double t = plan_cuts(c, most_blocks, &g);
  g.us = 5.0 + (H <= 64 ? 3.2 : 4.6) * t;
  return g;
}
hipError_t launch_fwd_narrow(const FwdArgs& a, int64_t rows, hipStream_t s);
hipError_t launch_bwd_narrow(const BwdArgs& a, const SmallGrads& g, bool want_dx, bool want_dw, hipStream_t s);
hipError_t launch_bwd_grads_small(const BwdArgs& a, const SmallGrads& g, bool want_dx, bool want_dw, hipStream_t s);

}  // namespace lce
