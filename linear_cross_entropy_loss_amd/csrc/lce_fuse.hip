// The pass between the logit kernel and the two gradient contractions when the logits are computed once
// (lce_forward_backward; the reference computes its gradients in the forward pass too,
// linear_cross_entropy/ops.py:721-799, from the logits chunk it keeps in memory).
//
// The logit kernel (launch_fwd_stage, lce_bwd_dz.hip) left e = 2^shift * exp(z - m) in the stage, m = the
// largest logit of the token within a slice of 128 columns, because a token's lse is only known once all its
// slices are done.  Here, with lse at hand,
//     dz[token][v] = e[token][v] * exp(m[token][v / 128] - lse[token]) * (1 + 2 * z_reg * lse[token])
//                  = 2^shift * softmax * gain                                       (ops.py:309-314, 415-422)
// in place, exact zeros for tokens with an ignored label and rows past the last one, and the target column
// gets the rounding of the fp32 value 2^shift * (softmax * gain - 1), formed from the target logit the logit
// kernel wrote, as in the kernel that recomputes the logits (lce_bwd_dz.hip).  The pass is bound by memory
// traffic: 2 bytes read and 2 written per logit.  For small hidden sizes, where that traffic is most of what the gradients
// cost beyond their matrix work, it is not made: the dx and dW kernels form dz on the way to LDS (stage_factors_kernel).
#include "lce_gemm3.h"
#include "lce_internal.h"

namespace lce {

namespace {

constexpr float kLog2e = 1.4426950408889634f;

// One workgroup per block of the stage (256 token rows x 64 columns, 32 KiB, BwdArgs::dz): blockIdx.x = column
// group, blockIdx.y = token tile.  Thread t first works out the factor of row t, then the block is
// rewritten in 16-byte pieces, consecutive lanes on consecutive pieces.
template <class T>
__global__ __launch_bounds__(256) void stage_scale_kernel(const BwdArgs a) {
  __shared__ float sh_f[kTile];
  __shared__ int sh_col[kTile];             // target column inside the block, or -1
  __shared__ unsigned short sh_tv[kTile];   // what goes there
  const int64_t rows = packed_rows(a.n_rows, a.N);
  const int64_t t0 = (int64_t)blockIdx.y * kTile;
  if (t0 >= rows) return;  // (token tiles without a row were not written and are not read)
  const int g = blockIdx.x;
  {
    const int64_t tok = t0 + threadIdx.x;
    const bool exists = tok < rows;
    const int64_t yy = exists ? a.y[tok] : a.ignore_index;
    const bool valid = yy != a.ignore_index;
    float f = 0.f;
    int col = -1;
    unsigned short tv = 0;
    if (valid) {
      const float lse = a.lse[tok];
      const float m = a.part_max[(a.v0 + (int64_t)g * 64) / kChunkV * a.nc + tok];
      float gain = 1.f + 2.f * a.z_reg * lse;
      if (a.dz_shift != 0) gain = fminf(fmaxf(gain, -63.f), 63.f);  // (as in lce_bwd_dz.hip)
      f = __builtin_amdgcn_exp2f((m - lse) * kLog2e) * gain;
      const int64_t rel = yy - (a.v0 + (int64_t)g * 64);
      if (rel >= 0 && rel < 64) {
        col = (int)rel;
        const float p = __builtin_amdgcn_exp2f(fmaf(a.tgt[tok] - lse, kLog2e, (float)a.dz_shift)) * gain;
        tv = to_bits<T>(p - __builtin_bit_cast(float, (127 + a.dz_shift) << 23));
      }
    }
    sh_f[threadIdx.x] = f;
    sh_col[threadIdx.x] = col;
    sh_tv[threadIdx.x] = tv;
  }
  __syncthreads();
  typedef typename elem_of<T>::type E;
  u32x4_t* blk = reinterpret_cast<u32x4_t*>(reinterpret_cast<E*>(a.dz) + dz_block_offset(blockIdx.y, g, a.vs));
  u32x4_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = blk[i * 256 + threadIdx.x];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int piece = i * 256 + threadIdx.x, r = piece >> 3, c0 = (piece & 7) * 8;
    const float f = sh_f[r];
    const int hit = sh_col[r] - c0;  // 0..7: the target is element `hit` of this piece
    u32x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = from_bits<T>((unsigned short)(v[i][j] & 0xffffu)) * f;
      const float hi = from_bits<T>((unsigned short)(v[i][j] >> 16)) * f;
      unsigned w = pack2<T>(lo, hi);
      if (hit == 2 * j) w = (w & 0xffff0000u) | sh_tv[r];
      if (hit == 2 * j + 1) w = (w & 0x0000ffffu) | ((unsigned)sh_tv[r] << 16);
      o[j] = w;
    }
    blk[piece] = o;
  }
}

// The same without the pass over the stage: only the factors are worked out, and the dx and dW kernels multiply e by them on
// its way to LDS (BwdArgs::dx_f, dw_f; the products and roundings are those of stage_scale_kernel).  The slice of 128 columns
// that holds a token's target is rewritten here, with a factor of 1 from then on.  One workgroup per token tile and
// kSlices slices.  (The two tables may be part_lse and part_max themselves: where there are several chunks, nothing reads
// those any more.)
// Bound by launch and latency: 12 bytes per 128 logits and 512 per token.  (4096 tokens, labels drawn uniformly, us a launch
// against the pass over the stage: V=32000 10 / 79, V=50264 12 / 122, V=65536 12 / 168; labels of a Zipf distribution, whose
// frequent ones give a workgroup many slices to rewrite: V=32000 17, V=50257 19.  Which problems take it: factors_in_gradients in
// lce_api.hip.)
constexpr int kSlices = 8;
template <class T>
__global__ __launch_bounds__(256) void stage_factors_kernel(const BwdArgs a) {
  __shared__ int sh_list[kTile];   // token rows whose target lies in one of this workgroup's slices
  __shared__ float sh_f[kTile];
  __shared__ unsigned short sh_tv[kTile];
  __shared__ int sh_rel[kTile];    // target column, from the first of these slices on
  __shared__ int sh_n;
  typedef typename elem_of<T>::type E;
  const int64_t rows = packed_rows(a.n_rows, a.N);
  const int64_t t0 = (int64_t)blockIdx.y * kTile;
  // (token tiles without a row were not written and are not read -- but for the first: dW's K extent is never empty, and zeros
  // stand there in the place of e)
  if (t0 >= rows && t0 > 0) return;
  const int slices = (int)(a.vs / kChunkV), s0 = blockIdx.x * kSlices;
  const int t = threadIdx.x;
  const int64_t tok = t0 + t;
  const bool exists = tok < rows;
  // (everything is asked for at once: a launch is a few latencies long)
  const int64_t yy = exists ? a.y[tok] : a.ignore_index;
  const float lse = exists ? a.lse[tok] : 0.f, zt = a.tgt[tok];  // (tgt: written where the label is a column of W)
  float f[kSlices];
#pragma unroll
  for (int i = 0; i < kSlices; ++i) f[i] = s0 + i < slices ? a.part_max[(int64_t)(s0 + i) * a.nc + tok] : 0.f;
  const bool valid = yy != a.ignore_index;
  float gain = 1.f + 2.f * a.z_reg * lse;
  if (a.dz_shift != 0) gain = fminf(fmaxf(gain, -63.f), 63.f);  // (as in lce_bwd_dz.hip)
  if (t == 0) sh_n = 0;
#pragma unroll
  for (int i = 0; i < kSlices; ++i) f[i] = valid ? __builtin_amdgcn_exp2f((f[i] - lse) * kLog2e) * gain : 0.f;
  __syncthreads();  // every partial has been read
  const int64_t rel = valid ? yy - (int64_t)s0 * kChunkV : -1;
  if (rel >= 0 && rel < kSlices * kChunkV && yy < a.vs) {
    const float p = __builtin_amdgcn_exp2f(fmaf(zt - lse, kLog2e, (float)a.dz_shift)) * gain;
    const int at = atomicAdd(&sh_n, 1);
    sh_list[at] = t;
    sh_rel[at] = (int)rel;
    sh_tv[at] = to_bits<T>(p - __builtin_bit_cast(float, (127 + a.dz_shift) << 23));
#pragma unroll
    for (int i = 0; i < kSlices; ++i)
      if ((int)(rel / kChunkV) == i) {
        sh_f[at] = f[i];
        f[i] = 1.f;
      }
  }
  // (the places of this tile's 256 tokens within a slice of either table)
  const int64_t px = t0 + (t & 31) * 8 + (t >> 5), pw = t0 + (t & ~63) + (t & 7) * 8 + ((t & 63) >> 3);
#pragma unroll
  for (int i = 0; i < kSlices; ++i)
    if (s0 + i < slices) {
      const_cast<float*>(a.dx_f)[(int64_t)(s0 + i) * a.nc + px] = f[i];
      const_cast<float*>(a.dw_f)[(int64_t)(s0 + i) * a.nc + pw] = f[i];
    }
  __syncthreads();
  // 16 threads rewrite the 128 columns of one token, four tokens of theirs in flight (frequent labels: up to all 256 tokens)
  const int n = sh_n, piece = t & 15;
  for (int e0 = t >> 4; e0 < n; e0 += 64) {
    u32x4_t* at[4];
    u32x4_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + 16 * u < n ? e0 + 16 * u : e0;
      at[u] = reinterpret_cast<u32x4_t*>(reinterpret_cast<E*>(a.dz) +
                                         dz_block_offset(blockIdx.y, 2 * (s0 + sh_rel[e] / kChunkV) + (piece >> 3), a.vs) +
                                         sh_list[e] * 64 + (piece & 7) * 8);
      v[u] = *at[u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + 16 * u;
      if (e >= n) break;
      const int hit = (sh_rel[e] & (kChunkV - 1)) - piece * 8;  // 0..7: the target is element `hit` of this piece
      u32x4_t o = scaled_piece<T>(v[u], sh_f[e]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (hit == 2 * j) o[j] = (o[j] & 0xffff0000u) | sh_tv[e];
        if (hit == 2 * j + 1) o[j] = (o[j] & 0x0000ffffu) | ((unsigned)sh_tv[e] << 16);
      }
      *at[u] = o;
    }
  }
}

// fp32 tensors: the stage holds the unscaled fp32 logits, halves apart (lce_bwd_dz.hip, KEEP), and dz as a bf16 pair takes their
// place, with the arithmetic of the kernel that recomputes the logits, so that dz has the same bits as there.  A workgroup per block,
// a thread on eight columns at a time.  Bound by memory traffic: 4 bytes read and 4 written per logit (1024 tokens, V=16384: 24 us, 5.6 TB/s).
__global__ __launch_bounds__(256) void stage_pairs_kernel(const BwdArgs a) {
  __shared__ float sh_nlse[kTile], sh_gain[kTile];
  __shared__ int sh_col[kTile];  // target column inside the block, -1 or, for a row without gradient, kNoRow
  constexpr int kNoRow = -0x7fffffff;
  const int64_t rows = packed_rows(a.n_rows, a.N);
  const int64_t t0 = (int64_t)blockIdx.y * kTile;
  if (t0 >= rows && t0 > 0) return;  // (token tiles without a row are not read, but for the first: dW's K extent is never empty)
  const int64_t v0 = (int64_t)blockIdx.x * 64;
  {
    const int64_t tok = t0 + threadIdx.x;
    const bool exists = tok < rows;
    const int64_t yy = exists ? a.y[tok] : a.ignore_index, rel = yy - v0;
    const float lse = exists ? a.lse[tok] : 0.f;
    sh_nlse[threadIdx.x] = fmaf(-lse, kLog2e, 0.f);
    sh_gain[threadIdx.x] = 1.f + 2.f * a.z_reg * lse;
    sh_col[threadIdx.x] = yy == a.ignore_index ? kNoRow : rel >= 0 && rel < 64 ? (int)rel : -1;
  }
  __syncthreads();
  const float c1 = a.scale * kLog2e;
  const int cols = a.vw - v0 < 64 ? (int)(a.vw - v0) : 64;  // (may be <= 0)
  u32x4_t* blk = reinterpret_cast<u32x4_t*>(reinterpret_cast<unsigned short*>(a.dz) + 2 * dz_block_offset(blockIdx.y, blockIdx.x, a.vs));
  constexpr int kLo = kDzBlockElems * 2 / 16;  // pieces to the block of the lo parts
  u32x4_t zh[8], zl[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    zh[i] = blk[i * 256 + threadIdx.x];
    zl[i] = blk[i * 256 + threadIdx.x + kLo];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int piece = i * 256 + threadIdx.x, r = piece >> 3, c0 = (piece & 7) * 8;
    const float nlse = sh_nlse[r], gain = sh_gain[r];
    const int col = sh_col[r];
    u32x4_t oh, ol;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float d[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const unsigned bits = __builtin_amdgcn_perm(zh[i][j], zl[i][j], e == 0 ? 0x05040100u : 0x07060302u);
        const float z = __builtin_bit_cast(float, bits);
        const int c = c0 + 2 * j + e;
        float p = __builtin_amdgcn_exp2f(fmaf(z, c1, nlse)) * gain;
        p = c == col ? p - 1.f : p;
        d[e] = c < cols && col != kNoRow ? p : 0.f;
      }
      oh[j] = pack2<BF16>(d[0], d[1]);
      ol[j] = pack2<BF16>(bf16_lo(d[0]), bf16_lo(d[1]));
    }
    blk[piece] = oh;
    blk[piece + kLo] = ol;
  }
}

// t[r][c] *= g[0] for r < rows, c < cols (row stride ld, rows on 16-byte boundaries), the product formed in fp32;
// nothing is read or written when g[0] is 1.  Pieces of 16 bytes, the last piece of a row element by element.
// v * f rounded to fp32 before anything else happens to it (the compiler may otherwise fold the product into
// a conversion that rounds the exact product once: another result on ties, and not the same in every code path).
LCE_DEV float scaled(float v, float f) {
  float p = v * f;
  asm volatile("" : "+v"(p));
  return p;
}

template <class E, int PER> LCE_DEV void scale_rows(E* t, int64_t rows, int64_t cols, int64_t ld, float f, int64_t first, int64_t step) {
  const int64_t pieces = (cols + PER - 1) / PER;
  for (int64_t i = first; i < rows * pieces; i += step) {
    const int64_t r = i / pieces, c0 = (i - r * pieces) * PER;
    E* at = t + r * ld + c0;
    if (c0 + PER <= cols) {
      u32x4_t v = *reinterpret_cast<const u32x4_t*>(at);
      E e[PER];
      __builtin_memcpy(e, &v, 16);
#pragma unroll
      for (int j = 0; j < PER; ++j) e[j] = (E)scaled((float)e[j], f);
      __builtin_memcpy(&v, e, 16);
      *reinterpret_cast<u32x4_t*>(at) = v;
    } else {
      for (int64_t c = c0; c < cols; ++c) t[r * ld + c] = (E)scaled((float)t[r * ld + c], f);
    }
  }
}
LCE_DEV void scale_task(const ScaleTask& t, float f, int64_t first, int64_t step) {
  if (t.t == nullptr) return;
  if (t.dtype == DT_BF16) scale_rows<__bf16, 8>((__bf16*)t.t, t.rows, t.cols, t.ld, f, first, step);
  else if (t.dtype == DT_F16) scale_rows<_Float16, 8>((_Float16*)t.t, t.rows, t.cols, t.ld, f, first, step);
  else scale_rows<float, 4>((float*)t.t, t.rows, t.cols, t.ld, f, first, step);
}
// Both gradients of a call in one launch: where the factor is 1, which is the rule, the launch is all there is to it.
__global__ __launch_bounds__(256) void scale_two_kernel(const ScaleTask t0, const ScaleTask t1, const float* g, const float* d) {
  const float f = d != nullptr ? g[0] / d[0] : g[0];
  if (f == 1.f) return;
  const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  scale_task(t0, f, first, step);
  scale_task(t1, f, first, step);
}

}  // namespace

hipError_t launch_scale_two(const ScaleTask& t0, const ScaleTask& t1, const float* g, const float* d, int num_cus, hipStream_t s) {
  int64_t work = 0;
  for (const ScaleTask* t : {&t0, &t1})
    if (t->t != nullptr) {
      if (t->dtype != DT_BF16 && t->dtype != DT_F16 && t->dtype != DT_F32) return hipErrorInvalidValue;
      const int per = t->dtype == DT_F32 ? 4 : 8;
      const int64_t w = t->rows * ((t->cols + per - 1) / per);
      work = w > work ? w : work;
    }
  if (work <= 0) return hipSuccess;
  int64_t grid = (work + 255) / 256;
  if (grid > (int64_t)num_cus * 16) grid = (int64_t)num_cus * 16;
  hipLaunchKernelGGL(scale_two_kernel, dim3((unsigned)grid), dim3(256), 0, s, t0, t1, g, d);
  return hipGetLastError();
}

hipError_t launch_scale_rows(void* t, int dtype, int64_t rows, int64_t cols, int64_t ld, const float* g, int num_cus,
                             hipStream_t s) {
  return launch_scale_two(ScaleTask{t, dtype, rows, cols, ld}, ScaleTask{}, g, nullptr, num_cus, s);
}

hipError_t launch_stage_scale(const BwdArgs& a, hipStream_t s) {
  if (a.part_max == nullptr || a.tgt == nullptr || a.lse == nullptr) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(a.vs / 64), (unsigned)(a.Np / kTile));
  if (a.x_dtype == DT_BF16) hipLaunchKernelGGL(stage_scale_kernel<BF16>, grid, dim3(256), 0, s, a);
  else if (a.x_dtype == DT_F16) hipLaunchKernelGGL(stage_scale_kernel<F16>, grid, dim3(256), 0, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_stage_pairs(const BwdArgs& a, hipStream_t s) {
  if (a.x_dtype != DT_PAIR || a.v0 != 0 || a.dz_shift != 0 || a.lse == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(stage_pairs_kernel, dim3((unsigned)(a.vs / 64), (unsigned)(a.Np / kTile)), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_stage_factors(const BwdArgs& a, hipStream_t s) {
  if (a.v0 != 0 || a.part_max == nullptr || a.tgt == nullptr || a.lse == nullptr || a.dx_f == nullptr || a.dw_f == nullptr)
    return hipErrorInvalidValue;
  const dim3 grid((unsigned)((a.vs / kChunkV + kSlices - 1) / kSlices), (unsigned)(a.Np / kTile));
  if (a.x_dtype == DT_BF16) hipLaunchKernelGGL(stage_factors_kernel<BF16>, grid, dim3(256), 0, s, a);
  else if (a.x_dtype == DT_F16) hipLaunchKernelGGL(stage_factors_kernel<F16>, grid, dim3(256), 0, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace lce
