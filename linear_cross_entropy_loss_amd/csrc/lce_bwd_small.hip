// Backward, steps 2 and 3 for problems with few output tiles: dx = dz W^T and dW = x^T dz (the contractions of
// linear_cross_entropy/ops.py:317 and 424) on 128 x 128 output tiles, both in one launch.
//
// What bounds such a problem is not the matrix pipe but launches that start from cold: a persistent kernel on 256 x 256 tiles
// spends 10 to 14 us on fetching its code before its first round is under way, its tiles leave compute units idle where there
// are fewer of them than those, and dx and dW come one after the other.  Here the code is a few KB (lce_gemm_small.h), a tile is a
// quarter of that, two workgroups share a compute unit, and a workgroup is one tile, or one stretch of K of a tile, of either
// gradient: both are spread over the chip together (SmallGrads, chosen on the host).  The stretches' fp32 sums meet in
// memory and are added, in order, by grads_tail_kernel.  A tile leaves through LDS, as rows: one short loop does for both gradients,
// every type and the stretches, where stores from the registers took 10 KB more of code.
//
// us, dx and dW with what adds their parts, 256 x 256 tiles / this: bf16 N=256, H=256, V=4096 45 / 16; N=1999, H=500, V=10007 92 / 56;
// N=1024, H=1024, V=8192 71 / 49; fp16 N=1536, H=192, V=6912 77 / 25; N=7552, H=512, V=512 141 / 55; fp32 N=655, H=128, V=4352 90 / 30.
// With the chip full of items of the same length a K tile takes 0.85 us (1.26 PFLOP/s); beyond that the persistent kernels are as
// fast or faster (N=2048, H=768, V=16384 115 / 120).
#include "lce_gemm_small.h"
#include "lce_internal.h"

namespace lce {

namespace {

// K tiles of the two contractions (even numbers).
LCE_DEV int small_kt(int64_t k) { return (int)((k + 2 * kBK - 1) / (2 * kBK) * 2); }

// Four consecutive columns of row r of either gradient, as stored; nothing goes past its limits (a quad that the last column cuts
// is written whole).  `sum`: the fp32 running sum of dx over slabs, or null.
template <class T, bool WVH>
LCE_DEV void small_put(const BwdArgs& a, bool is_dx, float* sum, float coef, int64_t r, int64_t c, f32x4_t v) {
  typedef typename elem_of<T>::type E;
  const int64_t rows = is_dx ? a.N : WVH ? a.V : a.H, cols = is_dx || WVH ? a.H : a.V;
  if (r >= rows || c >= cols) return;
  if (sum != nullptr) {
    f32x4_t* at = reinterpret_cast<f32x4_t*>(sum + r * a.Hp + c);
    if (!a.first) v += *at;
    if (!a.last) {
      *at = v;
      return;
    }
  }
  v *= coef;
  char* out = reinterpret_cast<char*>(is_dx ? a.dx : a.dw);
  const int64_t o = r * (is_dx ? a.lddx : a.lddw) + c;
  if ((is_dx ? a.dx_dtype : a.dw_dtype) == DT_F32) {
    f32x4_t* at = reinterpret_cast<f32x4_t*>(out + o * 4);
    if (!is_dx && a.dw_acc == 4) v += *at;  // (dW summed over chunks of token rows)
    *at = v;
  } else {
    u32x2_t b;
    b[0] = pack2<T>(v[0], v[1]);
    b[1] = pack2<T>(v[2], v[3]);
    *reinterpret_cast<u32x2_t*>(out + o * 2) = b;
  }
}

// A wave's 64 x 64 quarter of a tile to LDS, as the rows of the stored matrix: 128 rows of 128 floats, the 16-byte pieces of row r
// at the place XOR-ed by r % 8.  SWAP: the P index is the row (it runs along lanes), else the Q index.
static_assert(kSmallTile * kSmallTile * 4 <= kSmallLds, "a tile of sums fits where the stages were");
LCE_DEV float* small_piece(char* lds, int r, int c) {
  return reinterpret_cast<float*>(lds + r * (kSmallTile * 4) + (((c >> 2) ^ (r & 7)) << 4));
}
template <bool SWAP> LCE_DEV void small_to_lds(char* lds, const f32x16_t (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wp = wave & 1, wq = wave >> 1;
  const int wr = (SWAP ? wp : wq) * 64 + (lane & 31), wc = (SWAP ? wq : wp) * 64 + 4 * (lane >> 5);
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        f32x4_t v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (SWAP ? acc[rb][cb] : acc[cb][rb])[rq * 4 + j];
        *reinterpret_cast<f32x4_t*>(small_piece(lds, wr + rb * kBlk, wc + cb * kBlk + 8 * rq)) = v;
      }
}

template <class T, bool WVH>
__global__ __launch_bounds__(kThreads, 2) void grads_small_kernel(const BwdArgs a, const SmallGrads g) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename elem_of<T>::type E;
  constexpr int kParts = is_pair<T>::value ? 2 : 1, kProducts = is_pair<T>::value ? 3 : 1;
  const E* dz = reinterpret_cast<const E*>(a.dz);
  const void* dz_end = dz + kParts * a.dz_rows * a.vs;
  const bool in_first = (int)blockIdx.x < g.first_span, is_dx = in_first != (g.dw_first != 0);
  const int j = (int)blockIdx.x - (in_first ? 0 : g.first_span);
  const int tiles_p = (int)((a.H + kSmallTile - 1) / kSmallTile);
  const int nseg = is_dx ? g.dx_nseg : g.dw_nseg;
  const int tiles_q = (int)(((is_dx ? a.N : a.vw) + kSmallTile - 1) / kSmallTile);
  if (j >= tiles_p * tiles_q * nseg) return;  // (the first kind's share is a multiple of 8)
  int tile, tp, tq, seg;
  segment_coords(j, tiles_p * tiles_q, nseg, tile, seg);
  tile_coords(tile, 1, tiles_p, tiles_q, 8, 8, tp, tq);
  const int kt = small_kt(is_dx ? a.vw : a.N), s0 = segment_start(seg, nseg, kt), n = segment_start(seg + 1, nseg, kt) - s0;
  const int64_t k0 = (int64_t)s0 * kBK, h0 = (int64_t)tp * kSmallTile, q0 = (int64_t)tq * kSmallTile;
  f32x16_t acc[2][2];
  if (is_dx) {
    // P = W (rows h, K = v), Q = dz (rows token)
    const int64_t v0 = (a.v0 - a.wv0) + k0;
    const E* w = reinterpret_cast<const E*>(a.w);
    SmallPipe<T, !WVH, true, true, 2, 2, false> pipe;
    pipe.run(w + (WVH ? v0 * a.ldw + h0 : h0 * a.ldw + v0),
             WVH ? matrix_end<E>(w, a.Vw, a.ldw, a.H) : matrix_end<E>(w, kParts * a.H, a.ldw, a.Vw), a.ldw,
             dz + kParts * dz_block_offset(q0 / kTile, s0, a.vs) + q0 % kTile * kBK, dz_end, a.vs / kBK, a.vw - k0, kProducts * n,
             a.H * a.ldw * 2, kDzBlockElems * 2, lds, acc);
    small_to_lds<false>(lds, acc);
  } else {
    // P = x (K = token, columns h), Q = dz (columns v)
    const E* x = reinterpret_cast<const E*>(a.x);
    SmallPipe<T, false, false, true, 2, 2, !WVH> pipe;
    pipe.run(x + k0 * a.ldx + h0, matrix_end<E>(x, a.N, a.ldx, kParts == 2 ? a.x_lo + a.H : a.H), a.ldx,
             dz + kParts * dz_block_offset(k0 / kTile, q0 / kBK, a.vs) + k0 % kTile * kBK, dz_end, a.vs / kBK, 0, kProducts * n,
             a.x_lo * 2, kDzBlockElems * 2, lds, acc, s0 & 3);
    small_to_lds<!WVH>(lds, acc);
  }
  __syncthreads();
  float* part = nseg > 1 ? g.part + ((is_dx ? 0 : (int64_t)g.dx_blocks) + (int64_t)tile * nseg + seg) * (kSmallTile * kSmallTile) : nullptr;
  float* sum = !is_dx || (a.first && a.last) ? nullptr : a.dx_acc;
  const float coef = final_factor_of(a);
  const bool h_rows = !is_dx && !WVH;
  const int64_t qv = q0 + (is_dx ? 0 : a.v0), row0 = h_rows ? h0 : qv, col0 = h_rows ? qv : h0;
#pragma unroll 2
  for (int i = threadIdx.x; i < kSmallTile * kSmallTile / 4; i += kThreads) {
    const int r = i / (kSmallTile / 4), c = i % (kSmallTile / 4) * 4;
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(small_piece(lds, r, c));
    if (part != nullptr) *reinterpret_cast<f32x4_t*>(part + i * 4) = v;
    else small_put<T, WVH>(a, is_dx, sum, coef, row0 + r, col0 + c, v);
  }
}

// Adds the stretches of the tiles that are cut along K, in order; kTailParts workgroups to a tile.
constexpr int kTailParts = 8;
template <class T, bool WVH>
__global__ __launch_bounds__(256) void grads_tail_kernel(const BwdArgs a, const SmallGrads g, int dx_tiles) {
  int tile = (int)blockIdx.x / kTailParts, tp, tq, nseg;
  const int piece = (int)blockIdx.x % kTailParts;
  const bool is_dx = tile < dx_tiles;
  if (!is_dx) tile -= dx_tiles;
  const int tiles_p = (int)((a.H + kSmallTile - 1) / kSmallTile);
  const int tiles_q = (int)(((is_dx ? a.N : a.vw) + kSmallTile - 1) / kSmallTile);
  if (tile >= tiles_p * tiles_q) return;
  tile_coords(tile, 1, tiles_p, tiles_q, 8, 8, tp, tq);
  nseg = is_dx ? g.dx_nseg : g.dw_nseg;
  const float* part = g.part + ((is_dx ? 0 : (int64_t)g.dx_blocks) + (int64_t)tile * nseg) * (kSmallTile * kSmallTile);
  const int64_t h0 = (int64_t)tp * kSmallTile, q0 = (int64_t)tq * kSmallTile + (is_dx ? 0 : a.v0);
  float* sum = !is_dx || (a.first && a.last) ? nullptr : a.dx_acc;
  const float coef = final_factor_of(a);
  const bool h_rows = !is_dx && !WVH;
  const int64_t row0 = h_rows ? h0 : q0, col0 = h_rows ? q0 : h0;
  constexpr int kQuads = kSmallTile * kSmallTile / 4 / kTailParts;
#pragma unroll
  for (int u = 0; u < kQuads / 256; ++u) {
    const int i = piece * kQuads + u * 256 + (int)threadIdx.x, r = i / (kSmallTile / 4), c = i % (kSmallTile / 4) * 4;
    const float* at = part + r * kSmallTile + c;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nseg; s0 += 8) {  // (eight in flight; those that there are not are read again and dropped)
      f32x4_t t[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) t[k] = *reinterpret_cast<const f32x4_t*>(at + (int64_t)(s0 + k < nseg ? s0 + k : s0) * (kSmallTile * kSmallTile));
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (s0 + k < nseg) v += t[k];
    }
    small_put<T, WVH>(a, is_dx, sum, coef, row0 + r, col0 + c, v);
  }
}

template <class T, bool WVH> hipError_t launch_small(const BwdArgs& a, SmallGrads g, bool want_dx, bool want_dw, hipStream_t s) {
  const int64_t tp = (a.H + kSmallTile - 1) / kSmallTile;
  const int64_t dx_tiles = want_dx ? tp * ((a.N + kSmallTile - 1) / kSmallTile) : 0;
  const int64_t dw_tiles = want_dw ? tp * ((a.vw + kSmallTile - 1) / kSmallTile) : 0;
  const int64_t dx_items = dx_tiles * g.dx_nseg, dw_items = dw_tiles * g.dw_nseg;
  g.first_span = (int)pad_to(g.dw_first ? dw_items : dx_items, 8);  // (workgroup j of either gradient is on XCD j % 8)
  const int64_t grid = g.first_span + (g.dw_first ? dx_items : dw_items);
  if (grid <= 0) return hipSuccess;
  hipLaunchKernelGGL((grads_small_kernel<T, WVH>), dim3((unsigned)grid), dim3(kThreads), kSmallLds, s, a, g);
  hipError_t e = hipGetLastError();
  const int64_t dx_tails = g.dx_nseg > 1 ? dx_tiles : 0, tails = dx_tails + (g.dw_nseg > 1 ? dw_tiles : 0);
  if (e != hipSuccess || tails == 0) return e;
  hipLaunchKernelGGL((grads_tail_kernel<T, WVH>), dim3((unsigned)(tails * kTailParts)), dim3(256), 0, s, a, g, (int)dx_tails);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_bwd_grads_small(const BwdArgs& a, const SmallGrads& g, bool want_dx, bool want_dw, hipStream_t s) {
  if (a.n_rows != nullptr || a.dx_f != nullptr || a.dw_f != nullptr || (a.dw_acc != 0 && a.dw_acc != 3 && a.dw_acc != 4) || (a.dw_acc != 0 && a.dw_dtype != DT_F32) || ((g.dx_nseg > 1 || g.dw_nseg > 1) && g.part == nullptr))
    return hipErrorInvalidValue;
  if (a.w_vh) {
    if (a.x_dtype == DT_BF16 && a.w_dtype == DT_BF16) return launch_small<BF16, true>(a, g, want_dx, want_dw, s);
    if (a.x_dtype == DT_F16 && a.w_dtype == DT_F16) return launch_small<F16, true>(a, g, want_dx, want_dw, s);
    return hipErrorInvalidValue;
  }
  if (a.x_dtype == DT_BF16 && a.w_dtype == DT_BF16) return launch_small<BF16, false>(a, g, want_dx, want_dw, s);
  if (a.x_dtype == DT_F16 && a.w_dtype == DT_F16) return launch_small<F16, false>(a, g, want_dx, want_dw, s);
  if (a.x_dtype == DT_PAIR && a.w_dtype == DT_PAIR && a.dw_dtype == DT_F32) return launch_small<BF16P, false>(a, g, want_dx, want_dw, s);
  return hipErrorInvalidValue;
}

}  // namespace lce
