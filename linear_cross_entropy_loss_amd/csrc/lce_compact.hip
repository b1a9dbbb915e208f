// Tokens whose label equals ignore_index contribute nothing to the loss or to
// either gradient (linear_cross_entropy/ops.py:213, 314, 422), so the tile
// kernels never look at them: the kept tokens are packed to the front, in
// their original order, and the kernels run on the packed rows only.  The
// number of kept tokens stays on the device (the kernels read it), so nothing
// here synchronises with the host.  (The reference computes the ignored rows
// and multiplies them away.)
//
//   compact_labels  perm[j] = original index of the j-th kept token, yc[j] its label, n_rows = how many; the dropped
//                   tokens follow in perm from n_rows on, in their order (yc = ignore_index), for a caller that
//                   wants all rows with the kept ones first
//   gather_rows     xc[j] = x[perm[j]], lse_c[j] = lse[perm[j]]  (fp32 activations: as bf16 pairs, see gather_rows_split_kernel)
//   scatter_rows    rows of dropped tokens of dx = 0 (and dx[perm[j]] = dxc[j] where dx was staged packed)
//
// When no token is dropped (n_rows == N) the row copies are skipped and the
// tile kernels read x and write dx in place.
#include "lce_gemm.h"
#include "lce_internal.h"

namespace lce {

namespace {

constexpr int kSegTokens = 2048;  // tokens per workgroup of the counting / packing kernels
constexpr int kPerThread = kSegTokens / 256;

// Sum of `v` over the 256 threads of the workgroup; exclusive prefix of this thread in `excl`.
LCE_DEV int block_scan(int v, int& excl, int* sh /* [4] */) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) sh[wave] = incl;
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += sh[w];
    total += sh[w];
  }
  __syncthreads();  // sh may be reused by the caller
  excl = before + incl - v;
  return total;
}

__global__ __launch_bounds__(256) void count_kept_kernel(const int64_t* y, int64_t N, int64_t ignore_index, int* cnt) {
  __shared__ int sh[4];
  const int64_t base = (int64_t)blockIdx.x * kSegTokens + (int64_t)threadIdx.x * kPerThread;
  int c = 0;
#pragma unroll
  for (int k = 0; k < kPerThread; ++k) c += (base + k < N && y[base + k] != ignore_index) ? 1 : 0;
  int excl;
  const int total = block_scan(c, excl, sh);
  if (threadIdx.x == 0) cnt[blockIdx.x] = total;
}

// One workgroup: cnt[] becomes its own exclusive prefix sum, n_rows the total.
__global__ __launch_bounds__(256) void scan_counts_kernel(int* cnt, int64_t nseg, int64_t* n_rows) {
  __shared__ int sh[4];
  int64_t running = 0;
  for (int64_t base = 0; base < nseg; base += 256) {
    const int64_t i = base + threadIdx.x;
    const int v = i < nseg ? cnt[i] : 0;
    int excl;
    const int total = block_scan(v, excl, sh);
    if (i < nseg) cnt[i] = (int)(running + excl);
    running += total;
  }
  if (threadIdx.x == 0) n_rows[0] = running;
}

__global__ __launch_bounds__(256) void pack_kept_kernel(const int64_t* y, int64_t N, int64_t ignore_index,
                                                        const int* offs, const int64_t* n_rows, int* perm, int64_t* yc) {
  __shared__ int sh[4];
  const int64_t base = (int64_t)blockIdx.x * kSegTokens + (int64_t)threadIdx.x * kPerThread;
  int64_t lab[kPerThread];
  int c = 0;
#pragma unroll
  for (int k = 0; k < kPerThread; ++k) {
    lab[k] = base + k < N ? y[base + k] : ignore_index;
    c += lab[k] != ignore_index ? 1 : 0;
  }
  int excl;
  block_scan(c, excl, sh);
  int64_t j = (int64_t)offs[blockIdx.x] + excl;
  const int64_t kept = n_rows[0];
#pragma unroll
  for (int k = 0; k < kPerThread; ++k) {
    if (base + k >= N) break;
    // j kept tokens come before token base + k: a dropped one is number base + k - j among the dropped
    const int64_t at = lab[k] != ignore_index ? j++ : kept + (base + k - j);
    perm[at] = (int)(base + k);
    yc[at] = lab[k];
  }
}

// Rows of the chunks (lce_internal.h): out[c] among `kept` packed rows, out[1024 + c] among all N.
LCE_DEV void store_chunk_rows(int c, int64_t kept, int64_t N, int64_t nc, int64_t* out) {
  const int64_t left = kept - (int64_t)c * nc;
  out[c] = left < 0 ? 0 : (left > nc ? nc : left);
  const int64_t all = N - (int64_t)c * nc;  // the chunk's rows when the dropped tokens follow the kept ones
  out[1024 + c] = all < 0 ? 0 : (all > nc ? nc : all);
}

__global__ __launch_bounds__(1024) void chunk_rows_kernel(const int64_t* n_rows, int64_t N, int64_t nc, int chunks, int64_t* out) {
  if ((int)threadIdx.x < chunks) store_chunk_rows((int)threadIdx.x, packed_rows(n_rows, N), N, nc, out);
}

// All of it in one launch, for N <= 1024 * ITER: one workgroup of 16 waves, each on ITER * 64 consecutive tokens that it
// holds in registers, counted and numbered by ballots.  Bound by latency, as the four kernels are that do it for any N (counts,
// their scan, packing, the chunks' rows: 14 us of launches at N = 16384): 5 us up to N = 8192, 7.5 at 16384, 14.5 at 32768.
template <int ITER>
__global__ __launch_bounds__(1024) void compact_labels_kernel(const int64_t* y, int N, int64_t ignore_index, int64_t* n_rows,
                                                              int* perm, int64_t* yc, int64_t nc, int chunks,
                                                              int64_t* chunk_rows) {
  __shared__ int sh[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int base = wave * (ITER * 64) + lane;
  int64_t lab[ITER];
#pragma unroll
  for (int it = 0; it < ITER; ++it) lab[it] = base + it * 64 < N ? y[base + it * 64] : ignore_index;
  int mine = 0;
#pragma unroll
  for (int it = 0; it < ITER; ++it) mine += __popcll(__ballot(lab[it] != ignore_index));
  if (lane == 0) sh[wave] = mine;
  __syncthreads();
  int j = 0, kept = 0;  // kept tokens before this wave's, and of all
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    if (w < wave) j += sh[w];
    kept += sh[w];
  }
#pragma unroll
  for (int it = 0; it < ITER; ++it) {
    const int i = base + it * 64;
    const bool keep = lab[it] != ignore_index;
    const unsigned long long mask = __ballot(keep);
    const int before = j + __popcll(mask & ((1ull << lane) - 1));
    if (i < N) {
      const int at = keep ? before : kept + (i - before);  // a dropped token is number i - before among the dropped
      perm[at] = i;
      yc[at] = lab[it];
    }
    j += __popcll(mask);
  }
  if (threadIdx.x == 0) n_rows[0] = kept;
  if ((int)threadIdx.x < chunks) store_chunk_rows((int)threadIdx.x, kept, N, nc, chunk_rows);
}

// One workgroup per packed row (grid-stride).  Rows are moved in 16-byte pieces; `chunks` pieces per row.
// The last row of x may end with its last element (a caller's matrix need not own the stride padding of its
// last row): of that row only the whole pieces are moved as such, the rest 16 bits at a time, zero-filled.
__global__ __launch_bounds__(256) void gather_rows_kernel(const char* x, int64_t ldx_bytes, const int* perm,
                                                          const int64_t* n_rows, int64_t N, char* xc,
                                                          int64_t ldxc_bytes, int chunks, int64_t row_bytes,
                                                          const float* lse, float* lse_c, int always) {
  const int64_t rows = packed_rows(n_rows, N);
  const bool copy_x = rows != N || always != 0;
  for (int64_t j = blockIdx.x; j < rows; j += gridDim.x) {
    const int64_t src = packed_token(perm, j, N);
    if (lse != nullptr && threadIdx.x == 0) lse_c[j] = lse[src];
    if (copy_x) {
      const u32x4_t* s = reinterpret_cast<const u32x4_t*>(x + src * ldx_bytes);
      u32x4_t* d = reinterpret_cast<u32x4_t*>(xc + j * ldxc_bytes);
      const int whole = src == N - 1 ? (int)(row_bytes / 16) : chunks;
      for (int c = threadIdx.x; c < whole; c += 256) d[c] = s[c];
      if (whole < chunks && threadIdx.x < 8) {  // the piece that the end of the last row cuts through
        const int64_t b = (int64_t)whole * 16 + threadIdx.x * 2;
        const unsigned short v = b < row_bytes ? *reinterpret_cast<const unsigned short*>(x + src * ldx_bytes + b) : 0;
        *reinterpret_cast<unsigned short*>(xc + j * ldxc_bytes + b) = v;
      }
    }
  }
}

// fp32 activations reach the tile kernels as bf16 pairs, x = hi + lo (lce_gemm.h), in a copy that is made even when no token is
// dropped (`perm` / `n_rows` may be null: all rows, in their order): row j = [hi | lo] of x[perm[j]], each part `part` elements
// long (a multiple of 8, zero-padded).  One workgroup per packed row (grid-stride), 8 elements to a thread: two 16-byte loads,
// two 16-byte stores; the run that the end of a row cuts is read element by element.  Bound by memory traffic, 4 bytes read and
// 4 written per element.
__global__ __launch_bounds__(256) void gather_rows_split_kernel(const float* x, int64_t ldx, int64_t H, const int* perm,
                                                                const int64_t* n_rows, int64_t N, unsigned short* xc,
                                                                int64_t part, const float* lse, float* lse_c) {
  const int64_t rows = n_rows != nullptr ? packed_rows(n_rows, N) : N;
  for (int64_t j = blockIdx.x; j < rows; j += gridDim.x) {
    const int64_t src = perm != nullptr ? packed_token(perm, j, N) : j;
    if (lse != nullptr && threadIdx.x == 0) lse_c[j] = lse[src];
    const float* s = x + src * ldx;
    unsigned short* c = xc + j * 2 * part;
    for (int64_t k = threadIdx.x * 8; k < part; k += 256 * 8) {
      float v[8];
      if (k + 8 <= H) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(s + k), b = *reinterpret_cast<const f32x4_t*>(s + k + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = a[i];
          v[4 + i] = b[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = k + i < H ? s[k + i] : 0.f;
      }
      u32x4_t hi, lo;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        hi[i] = pack2<BF16>(v[2 * i], v[2 * i + 1]);
        lo[i] = pack2<BF16>(bf16_lo(v[2 * i]), bf16_lo(v[2 * i + 1]));
      }
      *reinterpret_cast<u32x4_t*>(c + k) = hi;
      *reinterpret_cast<u32x4_t*>(c + part + k) = lo;
    }
  }
}

// One workgroup per token (grid-stride): token i moves packed row i to its place (if there is a packed
// row i) and clears its own row of dx if it was dropped.  8-byte pieces, `chunks` per row.
__global__ __launch_bounds__(256) void scatter_rows_kernel(const char* dxc, int64_t lddxc_bytes, const int* perm,
                                                           const int64_t* n_rows, int64_t N, const int64_t* y,
                                                           int64_t ignore_index, char* dx, int64_t lddx_bytes,
                                                           int chunks) {
  const int64_t rows = packed_rows(n_rows, N);
  if (rows == N) return;  // nothing was dropped: the tile kernel wrote dx itself
  for (int64_t i = blockIdx.x; i < N; i += gridDim.x) {
    if (dxc != nullptr && i < rows) {
      const u32x2_t* s = reinterpret_cast<const u32x2_t*>(dxc + i * lddxc_bytes);
      u32x2_t* d = reinterpret_cast<u32x2_t*>(dx + packed_token(perm, i, N) * lddx_bytes);
      for (int c = threadIdx.x; c < chunks; c += 256) d[c] = s[c];
    }
    if (y[i] == ignore_index) {
      u32x2_t* d = reinterpret_cast<u32x2_t*>(dx + i * lddx_bytes);
      u32x2_t z;
      z[0] = 0u;
      z[1] = 0u;
      for (int c = threadIdx.x; c < chunks; c += 256) d[c] = z;
    }
  }
}

// The upstream gradient that fp16 gradients are formed for before the real one is known (lce.h): the labels are counted by
// workgroups whose 1024 threads have 8 labels each in flight, 64 KiB at a time.
LCE_DEV unsigned count_valid(const int64_t* y, int64_t N, int64_t ignore_index, unsigned* sh) {  // (thread 0 has the sum)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned mine = 0;
  for (int64_t base = (int64_t)blockIdx.x * 8 * 1024 + threadIdx.x; base < N; base += (int64_t)gridDim.x * 8 * 1024) {
    int64_t lab[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) lab[u] = base + u * 1024 < N ? y[base + u * 1024] : ignore_index;
#pragma unroll
    for (int u = 0; u < 8; ++u) mine += lab[u] != ignore_index ? 1u : 0u;
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mine += (unsigned)__shfl_xor((int)mine, d);
  if (lane == 0) sh[wave] = mine;
  __syncthreads();
  unsigned n = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) n += sh[w];
  return n;
}

LCE_DEV float power_of_two_below(unsigned n) {
  return __builtin_bit_cast(float, (unsigned)(127 + 31 - __builtin_clz(n > 0 ? n : 1)) << 23);
}

// Up to kStandInOne labels: one launch, bound by the latency of one workgroup's loads.  (It stands for a chain of eight
// elementwise and reduction launches: fp16 forward + backward, N=1024, H=1024, V=32000 333 -> 307 us; N=4096 862 -> 835 us.)
__global__ __launch_bounds__(1024) void stand_in_kernel(const int64_t* y, int64_t N, int64_t ignore_index, float* out) {
  __shared__ unsigned sh[16];
  const unsigned n = count_valid(y, N, ignore_index, sh);
  if (threadIdx.x == 0) out[0] = power_of_two_below(n);
}

// More labels than that: one compute unit reads them at 30 to 60 GB/s, so the counts of up to 256 workgroups are added up in
// *out itself, as a whole number, which the launch before cleared and the one after turns into the power of two.  (With the
// call's host time, us, one workgroup / three launches / the eight of torch: 2^16 labels 12 / - / 45, 2^17 19 / - / 48, 2^18
// 35 / 18 / 48, 2^20 291 / 18 / 47, 2^24 4633 / 28 / 94.)
constexpr int64_t kStandInOne = (int64_t)1 << 17;
__global__ void stand_in_clear_kernel(float* out) { reinterpret_cast<unsigned*>(out)[0] = 0; }
__global__ __launch_bounds__(1024) void stand_in_count_kernel(const int64_t* y, int64_t N, int64_t ignore_index, float* out) {
  __shared__ unsigned sh[16];
  const unsigned n = count_valid(y, N, ignore_index, sh);
  if (threadIdx.x == 0) atomicAdd(reinterpret_cast<unsigned*>(out), n);
}
__global__ void stand_in_finish_kernel(float* out) { out[0] = power_of_two_below(reinterpret_cast<const unsigned*>(out)[0]); }

unsigned row_grid(int64_t N, int num_cus) {
  int64_t g = (int64_t)num_cus * 8;
  if (g > N) g = N;
  return (unsigned)(g < 1 ? 1 : g);
}

}  // namespace

int64_t compact_segments(int64_t N) { return (N + kSegTokens - 1) / kSegTokens; }

hipError_t launch_compact_labels(const int64_t* y, int64_t N, int64_t ignore_index, int* cnt, int64_t* n_rows,
                                 int* perm, int64_t* yc, hipStream_t s, int64_t nc, int chunks, int64_t* chunk_rows) {
  if (chunks < 0 || chunks > 1024) return hipErrorInvalidValue;
  if (N <= 32 * 1024) {
    auto kern = N <= 4 * 1024 ? compact_labels_kernel<4> : N <= 16 * 1024 ? compact_labels_kernel<16> : compact_labels_kernel<32>;
    hipLaunchKernelGGL(kern, dim3(1), dim3(1024), 0, s, y, (int)N, ignore_index, n_rows, perm, yc, nc, chunks, chunk_rows);
    return hipGetLastError();
  }
  const int64_t nseg = compact_segments(N);
  hipLaunchKernelGGL(count_kept_kernel, dim3((unsigned)nseg), dim3(256), 0, s, y, N, ignore_index, cnt);
  hipLaunchKernelGGL(scan_counts_kernel, dim3(1), dim3(256), 0, s, cnt, nseg, n_rows);
  hipLaunchKernelGGL(pack_kept_kernel, dim3((unsigned)nseg), dim3(256), 0, s, y, N, ignore_index, cnt, n_rows, perm, yc);
  if (chunks > 0) hipLaunchKernelGGL(chunk_rows_kernel, dim3(1), dim3(1024), 0, s, n_rows, N, nc, chunks, chunk_rows);
  return hipGetLastError();
}

hipError_t launch_stand_in(const int64_t* y, int64_t N, int64_t ignore_index, float* out, hipStream_t s) {
  if (N <= kStandInOne) {
    hipLaunchKernelGGL(stand_in_kernel, dim3(1), dim3(1024), 0, s, y, N, ignore_index, out);
    return hipGetLastError();
  }
  const int64_t trips = (N + 8191) / 8192;
  hipLaunchKernelGGL(stand_in_clear_kernel, dim3(1), dim3(1), 0, s, out);
  hipLaunchKernelGGL(stand_in_count_kernel, dim3((unsigned)(trips < 256 ? trips : 256)), dim3(1024), 0, s, y, N, ignore_index, out);
  hipLaunchKernelGGL(stand_in_finish_kernel, dim3(1), dim3(1), 0, s, out);
  return hipGetLastError();
}

hipError_t launch_gather_rows_split(const float* x, int64_t ldx, int64_t H, const int* perm, const int64_t* n_rows,
                                    int64_t N, void* xc, int64_t ldxc, const float* lse, float* lse_c, int num_cus,
                                    hipStream_t s) {
  if (ldxc % 16 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(gather_rows_split_kernel, dim3(row_grid(N, num_cus)), dim3(256), 0, s, x, ldx, H, perm, n_rows, N,
                     reinterpret_cast<unsigned short*>(xc), ldxc / 2, lse, lse_c);
  return hipGetLastError();
}

hipError_t launch_gather_rows(const void* x, int64_t ldx_bytes, int64_t row_bytes, const int* perm,
                              const int64_t* n_rows, int64_t N, void* xc, int64_t ldxc_bytes, const float* lse,
                              float* lse_c, int num_cus, hipStream_t s, bool always) {
  hipLaunchKernelGGL(gather_rows_kernel, dim3(row_grid(N, num_cus)), dim3(256), 0, s,
                     reinterpret_cast<const char*>(x), ldx_bytes, perm, n_rows, N, reinterpret_cast<char*>(xc),
                     ldxc_bytes, (int)(ldxc_bytes / 16), row_bytes, lse, lse_c, always ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_scatter_rows(const void* dxc, int64_t lddxc_bytes, const int* perm, const int64_t* n_rows,
                               int64_t N, const int64_t* y, int64_t ignore_index, void* dx, int64_t lddx_bytes,
                               int64_t row_bytes, int num_cus, hipStream_t s) {
  hipLaunchKernelGGL(scatter_rows_kernel, dim3(row_grid(N, num_cus)), dim3(256), 0, s,
                     reinterpret_cast<const char*>(dxc), lddxc_bytes, perm, n_rows, N, y, ignore_index,
                     reinterpret_cast<char*>(dx), lddx_bytes, (int)((row_bytes + 7) / 8));
  return hipGetLastError();
}

}  // namespace lce
