// An fp32 (master) weight is rounded to the 16-bit compute type one vocabulary
// slab at a time, into a workspace buffer that the tile kernels of that slab
// then read like a 16-bit weight (the loss of few tokens reads the fp32 weight itself).  The reference converts the whole weight to
// fp16 on entry (custom_fwd(cast_inputs=torch.float16), linear_cross_entropy/ops.py:665-667);
// here the copy is one slab wide, is made in the compute type that the
// activations have, and costs one read of the slab.  The rounding (nearest
// even) is the same one the kernels apply to fp32 activations.
#include "lce_gemm.h"
#include "lce_internal.h"

namespace lce {

namespace {

// One thread converts 8 consecutive columns of one row (two 16-byte loads, one 16-byte store).
// Pairs (fp32 activations as well as weight): the copy has 2 H rows, bf16(w), then bf16(w - bf16(w)) (lce_gemm.h).
template <class T>
__global__ __launch_bounds__(256) void convert_w_slab_kernel(const float* src, int64_t ld, int64_t H, int64_t v0,
                                                               int64_t vw, unsigned short* dst, int64_t dst_ld) {
  const int64_t runs_per_row = dst_ld / 8;
  const int64_t total = H * runs_per_row;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t h = i / runs_per_row, c = (i - h * runs_per_row) * 8;
    const float* s = src + h * ld + v0 + c;
    float v[8];
    if (c + 8 <= vw) {
      const f32x4_t a = *reinterpret_cast<const f32x4_t*>(s), b = *reinterpret_cast<const f32x4_t*>(s + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = a[j];
        v[4 + j] = b[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = c + j < vw ? s[j] : 0.f;
    }
    u32x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = pack2<T>(v[2 * j], v[2 * j + 1]);
    *reinterpret_cast<u32x4_t*>(dst + h * dst_ld + c) = o;
    if constexpr (is_pair<T>::value) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = pack2<T>(bf16_lo(v[2 * j]), bf16_lo(v[2 * j + 1]));
      *reinterpret_cast<u32x4_t*>(dst + (H + h) * dst_ld + c) = o;
    }
  }
}

// The same for a weight stored (V, H) row-major: rows [v0, v0 + vw) of it, H columns (a multiple of 8).
template <class T>
__global__ __launch_bounds__(256) void convert_w_rows_kernel(const float* src, int64_t ld, int64_t H, int64_t v0,
                                                               int64_t vw, unsigned short* dst, int64_t dst_ld) {
  const int64_t runs_per_row = H / 8;
  const int64_t total = vw * runs_per_row;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / runs_per_row, c = (i - r * runs_per_row) * 8;
    const float* s = src + (v0 + r) * ld + c;
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(s), b = *reinterpret_cast<const f32x4_t*>(s + 4);
    u32x4_t o;
    o[0] = pack2<T>(a[0], a[1]);
    o[1] = pack2<T>(a[2], a[3]);
    o[2] = pack2<T>(b[0], b[1]);
    o[3] = pack2<T>(b[2], b[3]);
    *reinterpret_cast<u32x4_t*>(dst + r * dst_ld + c) = o;
  }
}

// Rows of 2-byte units at any 2-byte address, copied into rows that start on 16-byte boundaries, the rest of each of those
// cleared.  Bound by memory traffic, or by its launch where the matrix is small, which is why copying and clearing are one
// kernel.  A thread moves 16-byte pieces, four of a row in flight; the loads are of the source's alignment (the card takes
// them at any address), and the piece that the end of a row cuts goes unit by unit, so nothing past a row is read.
// 1 << shift threads share a row: few for a short one, so that a workgroup has work for all of its waves.
// (Against a copy and a fill of the padding columns, bf16 forward + backward: N=1999, H=500, V=10007 265 -> 256 us;
// N=4096, H=1023, V=32001 870 -> 858 us; N=8192, H=768, V=50257 2100 -> 2093 us.)
__global__ __launch_bounds__(256) void pad_rows_kernel(const char* src, int64_t src_ld, int64_t rows, int64_t row_bytes,
                                                       char* dst, int64_t dst_ld, int shift) {
  const int tpr = 1 << shift, rpb = 256 >> shift;
  const int c = threadIdx.x & (tpr - 1);
  const int64_t pieces = dst_ld / 16;
  for (int64_t r = (int64_t)blockIdx.x * rpb + (threadIdx.x >> shift); r < rows; r += (int64_t)gridDim.x * rpb) {
    const char* from = src + r * src_ld;
    u32x4_t* to = reinterpret_cast<u32x4_t*>(dst + r * dst_ld);
    for (int64_t p0 = (int64_t)blockIdx.y * 4 * tpr + c; p0 < pieces; p0 += (int64_t)gridDim.y * 4 * tpr) {
      u32x4_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t at = (p0 + u * tpr) * 16;
        v[u] = u32x4_t{0, 0, 0, 0};
        if (at + 16 <= row_bytes) __builtin_memcpy(&v[u], from + at, 16);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t at = (p0 + u * tpr) * 16;
        if (at < row_bytes && at + 16 > row_bytes) {
          const unsigned short* f = reinterpret_cast<const unsigned short*>(from + at);
          const int n = (int)(row_bytes - at) / 2;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (j < n) v[u][j / 2] |= (unsigned)f[j] << (16 * (j & 1));
        }
        if (p0 + u * tpr < pieces) to[p0 + u * tpr] = v[u];
      }
    }
  }
}

// dst[r][c] = src[c][r] for c < cols, zeros from there to the end of dst's rows: a matrix that lies transposed, with rows that may
// start anywhere.  Bound by memory traffic, read once and written once.  A workgroup turns 64 x 64 elements over in LDS: 16 bytes
// of a row of src to a thread, 8 rows apart by lane groups of 64 elements (loads of the source's alignment; the run that the end
// of a row cuts goes element by element), then 16 bytes of a row of dst.  Rows of the LDS tile are one 16-byte piece longer than
// 64 elements, so that the threads that gather a column meet different banks.
// (V=235136, H=481 in bf16: 128 us, 3.5 TB/s, against 1990 of an elementwise copy.)
template <class E>
__global__ __launch_bounds__(256) void transpose_rows_kernel(const E* src, int64_t src_ld, int64_t rows, int64_t cols, E* dst,
                                                             int64_t dst_ld) {
  constexpr int kPer = 16 / (int)sizeof(E), kPieces = 64 / kPer, kLine = 64 + kPer;
  __shared__ __attribute__((aligned(16))) E tile[64 * kLine];
  const int64_t tiles_c = (dst_ld + 63) / 64, tiles = (rows + 63) / 64 * tiles_c;
  for (int64_t b = blockIdx.x; b < tiles; b += gridDim.x) {
    const int64_t r0 = b / tiles_c * 64, c0 = b % tiles_c * 64;
#pragma unroll
    for (int i = 0; i < 64 * kPieces / 256; ++i) {
      const int p = i * 256 + threadIdx.x, c = p / kPieces, r = p % kPieces * kPer;
      E v[kPer] = {};
      const E* from = src + (c0 + c) * src_ld + r0 + r;
      if (c0 + c < cols) {
        if (r0 + r + kPer <= rows) {
          __builtin_memcpy(v, from, 16);
        } else {
#pragma unroll
          for (int j = 0; j < kPer; ++j)
            if (r0 + r + j < rows) v[j] = from[j];
        }
      }
      __builtin_memcpy(__builtin_assume_aligned(&tile[c * kLine + r], 16), v, 16);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * kPieces / 256; ++i) {
      const int p = i * 256 + threadIdx.x, r = p / kPieces, c = p % kPieces * kPer;
      E v[kPer];
#pragma unroll
      for (int j = 0; j < kPer; ++j) v[j] = tile[(c + j) * kLine + r];
      // (dst_ld is a multiple of kPer)
      if (r0 + r < rows && c0 + c < dst_ld)
        __builtin_memcpy(__builtin_assume_aligned(dst + (r0 + r) * dst_ld + c0 + c, 16), v, 16);
    }
    __syncthreads();
  }
}

}  // namespace

hipError_t launch_transpose_rows(const void* src, int64_t src_ld, int64_t rows, int64_t cols, int es, void* dst, int64_t dst_ld,
                                 hipStream_t s) {
  if (rows < 1 || cols < 1 || (es != 2 && es != 4) || dst_ld < cols || dst_ld * es % 16 != 0) return hipErrorInvalidValue;
  int64_t grid = (rows + 63) / 64 * ((dst_ld + 63) / 64);
  if (grid > 65536) grid = 65536;
  if (es == 2)
    hipLaunchKernelGGL(transpose_rows_kernel<unsigned short>, dim3((unsigned)grid), dim3(256), 0, s,
                       reinterpret_cast<const unsigned short*>(src), src_ld, rows, cols, reinterpret_cast<unsigned short*>(dst), dst_ld);
  else
    hipLaunchKernelGGL(transpose_rows_kernel<unsigned>, dim3((unsigned)grid), dim3(256), 0, s, reinterpret_cast<const unsigned*>(src),
                       src_ld, rows, cols, reinterpret_cast<unsigned*>(dst), dst_ld);
  return hipGetLastError();
}

hipError_t launch_convert_w_rows(const float* src, int64_t ld, int64_t H, int64_t v0, int64_t vw, void* dst,
                                 int64_t dst_ld, int compute_dtype, hipStream_t s) {
  if (H % 8 != 0 || dst_ld % 8 != 0) return hipErrorInvalidValue;
  const int64_t total = vw * (H / 8);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) return hipSuccess;
  unsigned short* d = reinterpret_cast<unsigned short*>(dst);
  if (compute_dtype == DT_F16) {
    hipLaunchKernelGGL((convert_w_rows_kernel<F16>), dim3((unsigned)blocks), dim3(256), 0, s, src, ld, H, v0, vw, d, dst_ld);
  } else {
    hipLaunchKernelGGL((convert_w_rows_kernel<BF16>), dim3((unsigned)blocks), dim3(256), 0, s, src, ld, H, v0, vw, d, dst_ld);
  }
  return hipGetLastError();
}

hipError_t launch_pad_rows(const void* src, int64_t src_ld, int64_t rows, int64_t row_bytes, void* dst, int64_t dst_ld,
                           hipStream_t s) {
  if (rows < 1 || row_bytes < 2 || row_bytes % 2 != 0 || dst_ld % 16 != 0 || dst_ld < row_bytes) return hipErrorInvalidValue;
  const int64_t pieces = dst_ld / 16;
  int shift = 3;
  while (shift < 8 && ((int64_t)4 << shift) < pieces) ++shift;
  int64_t gx = (rows + (256 >> shift) - 1) / (256 >> shift), gy = (pieces + (4 << shift) - 1) / (4 << shift);
  if (gx > 16384) gx = 16384;
  if (gy > 16384) gy = 16384;
  hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, reinterpret_cast<const char*>(src),
                     src_ld, rows, row_bytes, reinterpret_cast<char*>(dst), dst_ld, shift);
  return hipGetLastError();
}

hipError_t launch_convert_w_slab(const float* src, int64_t ld, int64_t H, int64_t v0, int64_t vw, void* dst,
                                 int64_t dst_ld, int compute_dtype, hipStream_t s) {
  const int64_t total = H * (dst_ld / 8);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) return hipSuccess;
  unsigned short* d = reinterpret_cast<unsigned short*>(dst);
  if (compute_dtype == DT_PAIR) {
    hipLaunchKernelGGL((convert_w_slab_kernel<BF16P>), dim3((unsigned)blocks), dim3(256), 0, s, src, ld, H, v0, vw, d, dst_ld);
  } else if (compute_dtype == DT_F16) {
    hipLaunchKernelGGL((convert_w_slab_kernel<F16>), dim3((unsigned)blocks), dim3(256), 0, s, src, ld, H, v0, vw, d, dst_ld);
  } else {
    hipLaunchKernelGGL((convert_w_slab_kernel<BF16>), dim3((unsigned)blocks), dim3(256), 0, s, src, ld, H, v0, vw, d, dst_ld);
  }
  return hipGetLastError();
}

}  // namespace lce
