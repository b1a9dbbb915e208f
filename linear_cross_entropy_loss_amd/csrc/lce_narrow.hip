// Hidden sizes of up to 128: logits, loss partials and gradients without dz ever reaching memory.
//
// At such a size a logit costs less to multiply than to store: staged (lce_bwd_dz.hip), dz is written once and read twice, 6 bytes
// for 2 H multiply-adds, the stage fills the scratch bound and cuts the problem into slabs, and a tile's prologue and epilogue take
// several times its one or two K tiles.  Here one of the two matrices stays and the other streams past it.  A workgroup keeps
// 128 rows of the one, 32 to a wave, as fragments in registers, and works through tiles of 128 rows of the other, double buffered in
// LDS, the next one in flight for as long as a tile takes; two workgroups share a compute unit, so that one's exponentials run under
// the other's matrix instructions.
//   forward   tokens stay, the vocabulary streams: S = W x^T, then the partials of the forward's other kernels, slice by slice
//   dx        the same, S -> dz in registers, dx += dz W from the tile that is in LDS anyway
//   dW        the vocabulary stays, tokens stream: S = x W, dz, dW += dz^T x
// The gradients evaluate the logits once more each (10 N H V multiply-adds instead of 8) for no traffic but x, W and their results.
// An accumulator block of S has the streaming index along its registers, in the order that the fragments of the second product
// want along K once lanes l and l + 32 have exchanged quads: dz goes from one matrix instruction to the next without LDS.
// dz is rounded once to the compute type, as in the staged kernels, and has their bits.
// Large problems have their tokens with an ignored label packed away first (plan_narrow in lce_api.hip says where): the number of rows is
// read from the device, and the cuts of dW follow it.  bf16 N=65536, H=128, V=32768, us of a backward, all rows / packed: none ignored
// 2088 / 2117, 5 % 2089 / 2078, 85 % 1845 / 739; staged 4206, 4052, 1414.
//
// Bound by vector instructions, of which an exponential is four, with the matrix instructions only partly under them: 128 x 128
// logits take two workgroups of a compute unit 3.3 us for the forward and 3.1 for a gradient at a hidden size of 64 (0.6 of 1.4
// to 1.7 they would at the exponentials' rate), 4.4 and 4.6 at 128.  us, kernels of a step, staged / this: bf16 N=300, H=64, V=1000
// 64 / 28; N=2048, H=64, V=32768 219 / 104; N=1152, H=64, V=220160 641 / 320; N=16384, H=64, V=16384 839 / 319; N=8192, H=128, V=8192 285 / 167;
// fp16 N=18432, H=128, V=9344 764 / 320.  With three and four K tiles there is room for one workgroup on a compute unit only, and
// staging is faster where the bound allows it (N=4096, H=256, V=16384 205 / 271; the other way N=16384, H=256, V=4096 372 / 273).
#include <type_traits>

#include "lce_gemm_small.h"
#include "lce_internal.h"
#include "lce_fwd_epilogue.h"

namespace lce {

namespace {

constexpr int kNarrowTile = 128;
// K tiles (64 deep) of a hidden size.
template <int KT> constexpr int narrow_buf() { return KT * kNarrowTile * kBK * 2; }
constexpr int kNarrowScalars = 3 * kNarrowTile + 4;  // floats: three numbers of each token of a tile, and whether labels meet the workgroup's columns
template <int KT> constexpr int narrow_lds() { return 2 * narrow_buf<KT>() + 2 * kNarrowScalars * 4; }

// threadIdx.x from the lane's number and the wave's, worked out where it is used: not held in a register through the loops.
LCE_DEV int narrow_tid(int wave) {
  int zero = 0;
  asm volatile("" : "+v"(zero));
  return wave * 64 + (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, (unsigned)zero));
}

// Byte that is XOR-ed into the place of a 16-byte piece in row r of an LDS tile: eight consecutive rows have the same piece in
// eight different bank groups (plain reads, a row to a lane), four of them 32-byte pieces in four (transposing reads).
LCE_DEV int narrow_swizzle(int r) { return ((r & 3) << 5) | (((r >> 2) & 1) << 4); }

// A tile of 128 rows c of a matrix, all of its H columns, on its way to LDS.
//   !TRANS  stored [c][h]: LDS rows are c, 128 bytes (64 h), one block of 128 rows for each K tile
//   TRANS   stored [h][c]: LDS rows are h, 256 bytes (128 c)
template <class T, bool TRANS, int KT> struct NarrowTile {
  u32x4_t v[4 * KT];
  unsigned off[TRANS ? 1 : KT];  // this thread's first piece, in bytes (!TRANS: of each K tile, out of range past H)
  int step, lds;                 // bytes between its pieces (uniform); its place in LDS
  LCE_DEV void init(int wave, int64_t ld, int64_t H64) {
    const int t = narrow_tid(wave), H = (int)H64;
    if (TRANS) {
      const int h = t >> 4;  // (rows past H lie behind the matrix' end)
      off[0] = (unsigned)((h * ld + (t & 15) * 8) * 2);
      step = (int)(16 * ld * 2);
      lds = h * 256 + (((t & 15) << 4) ^ narrow_swizzle(h));
    } else {
      const int c = t >> 3;
#pragma unroll
      for (int k = 0; k < KT; ++k) {
        const int h = k * kBK + (t & 7) * 8;
        off[k] = h < H ? (unsigned)((c * ld + h) * 2) : 0x80000000u;
      }
      step = (int)(32 * ld * 2);
      lds = c * 128 + (((t & 7) << 4) ^ narrow_swizzle(c));
    }
  }
  // base: element (row 0 of the tile, h = 0) resp. (h = 0, column 0); left: columns c of the matrix from there on
  LCE_DEV void load(const void* base, const void* end, int64_t left) {
    const int64_t range64 = reinterpret_cast<const char*>(end) - reinterpret_cast<const char*>(base);
    const int range = range64 <= 0 ? 0 : range64 > 0x7fffffff ? 0x7fffffff : (int)range64;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, range, 0x00020000);
    const unsigned o = TRANS && (narrow_tid(0) & 15) * 8 >= left ? 0x80000000u : off[0];
#pragma unroll
    for (int i = 0; i < 4 * KT; ++i)
      v[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(TRANS ? o : off[TRANS ? 0 : i >> 2]), (TRANS ? i : i & 3) * step, 0);
  }
  LCE_DEV void store(char* buf) const {
#pragma unroll
    for (int i = 0; i < 4 * KT; ++i)
      *reinterpret_cast<u32x4_t*>(buf + lds + (TRANS ? i * (16 * 256) : (i >> 2) * (kNarrowTile * 128) + (i & 3) * (32 * 128))) = v[i];
  }
};

// Fragments from LDS, 8 consecutive numbers to a lane, by four offsets of the lane and constants: the swizzle meets the lowest bits
// of what differs from one fragment to the next.
//   Plain   32 LDS rows, columns col + 8 * (lane / 32)
//   Trans   32 LDS columns, rows row + 8 * (lane / 32), by transposing reads
template <int STRIDE> struct NarrowPlain {
  int off[4];  // by (col / 16) % 4
  LCE_DEV void init() {
    const int l = narrow_tid(0), r = l & 31;
#pragma unroll
    for (int k = 0; k < 4; ++k) off[k] = r * STRIDE + ((k * 32 + 16 * (l >> 5)) ^ narrow_swizzle(r));
  }
  // rows from 32 * blk on, columns from 16 * ks on
  LCE_DEV s16x8_t read(const char* m, int blk, int ks) const {
    return *reinterpret_cast<const s16x8_t*>(m + off[ks & 3] + blk * (kBlk * STRIDE) + (ks >> 2) * 128);
  }
};
template <int STRIDE> struct NarrowTrans {
  int off[2][2];  // by the parity of the column block; rows 0 .. 3 and 4 .. 7 of a lane's eight
  LCE_DEV void init() {
    const int l = narrow_tid(0), g = l >> 4, s = l & 15, j = s >> 2, c = s & 3, r = 8 * (g >> 1) + j;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int u = 0; u < 2; ++u) off[p][u] = (r + 4 * u) * STRIDE + ((p * 64 + 32 * (g & 1) + 8 * c) ^ narrow_swizzle(r + 4 * u));
  }
  // columns from 32 * blk on, rows from 16 * ks on
  LCE_DEV s16x8_t read(const char* m, int blk, int ks) const {
    const char* p = m + (blk >> 1) * 128 + ks * (16 * STRIDE);
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LCE_LDS(s16x4_t)*)(p + off[blk & 1][0]));
    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LCE_LDS(s16x4_t)*)(p + off[blk & 1][1]));
    s16x8_t v;
    v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
    v[4] = hi[0]; v[5] = hi[1]; v[6] = hi[2]; v[7] = hi[3];
    return v;
  }
};
// The two products' reads of a streaming tile: rows c of block i and k-step ks along h; rows h of block hb and k-step ks along c.
template <bool TRANS> struct NarrowReader;
template <> struct NarrowReader<true> {
  NarrowTrans<256> t;
  NarrowPlain<256> p;
  LCE_DEV void init() { t.init(); p.init(); }
  LCE_DEV s16x8_t a(const char* buf, int i, int ks) const { return t.read(buf, i, ks); }
  LCE_DEV s16x8_t b(const char* buf, int hb, int ks) const { return p.read(buf, hb, ks); }
};
template <> struct NarrowReader<false> {
  static constexpr int kBlock = kNarrowTile * 128;  // a K tile's rows
  NarrowTrans<128> t;
  NarrowPlain<128> p;
  LCE_DEV void init() { t.init(); p.init(); }
  LCE_DEV s16x8_t a(const char* buf, int i, int ks) const { return p.read(buf + (ks >> 2) * kBlock, i, ks & 3); }
  LCE_DEV s16x8_t b(const char* buf, int hb, int ks) const { return t.read(buf + (hb >> 1) * kBlock, hb & 1, ks); }
};

// The stationary rows of a wave, from `base` (row 0 of its 32, h = 0) of a matrix stored [r][h].
template <int KT> LCE_DEV void narrow_stay(s16x8_t (&q)[4 * KT], const void* base, const void* end, int64_t ld, int64_t H) {
  const int64_t range64 = reinterpret_cast<const char*>(end) - reinterpret_cast<const char*>(base);
  const int range = range64 <= 0 ? 0 : range64 > 0x7fffffff ? 0x7fffffff : (int)range64;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, range, 0x00020000);
  const int l = narrow_tid(0);
#pragma unroll
  for (int ks = 0; ks < 4 * KT; ++ks) {
    const int h = ks * 16 + 8 * (l >> 5);
    const unsigned off = h < (int)H ? (unsigned)(((l & 31) * ld + h) * 2) : 0x80000000u;
    q[ks] = __builtin_bit_cast(s16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, 0, 0));
  }
}

template <class T, bool TRANS, int KT> LCE_DEV void narrow_logits(const NarrowReader<TRANS>& rd, const char* buf, const s16x8_t (&q)[4 * KT], f32x16_t (&s)[kNB][1]) {
#pragma unroll
  for (int i = 0; i < kNB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[i][0][r] = 0.f;
  s16x8_t f[2][2];  // fragments of two blocks and of the next two
#pragma unroll
  for (int i = 0; i < 2; ++i) f[0][i] = rd.a(buf, i, 0);
#pragma unroll
  for (int n = 0; n < 8 * KT; ++n) {
    const int ks = n >> 1, i0 = 2 * (n & 1);
    if (n + 1 < 8 * KT) {
#pragma unroll
      for (int i = 0; i < 2; ++i) f[(n + 1) & 1][i] = rd.a(buf, 2 - i0 + i, (n + 1) >> 1);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) s[i0 + i][0] = mfma32<T>(f[n & 1][i], q[ks], s[i0 + i][0]);
    __builtin_amdgcn_sched_barrier(0);  // (no fragments further ahead: they would not fit the registers)
  }
}

template <class T, bool WVH, bool MON, int KT>
__global__ __launch_bounds__(kThreads, 2) void fwd_narrow_kernel(const FwdArgs a, int tiles_p, int tiles_q, int nseg) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename elem_of<T>::type E;
  const int64_t rows = a.n_rows ? packed_rows(a.n_rows, a.N) : a.N;
  const bool packed = rows != a.N;
  const E* x = reinterpret_cast<const E*>(packed ? a.xc : a.x);
  const int64_t ldx = packed ? a.ldxc : a.ldx;
  int tq, seg;
  segment_coords((int)blockIdx.x, tiles_q, nseg, tq, seg);
  const int first = (int)((int64_t)tiles_p * seg / nseg), last = (int)((int64_t)tiles_p * (seg + 1) / nseg);
  const int64_t t0 = (int64_t)tq * kNarrowTile;
  if (a.row0 + t0 >= rows) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t tw = t0 + wave * kBlk, tok = a.row0 + tw + (lane & 31);
  const E* w = reinterpret_cast<const E*>(a.w);
  const void* w_end = WVH ? matrix_end<E>(w, a.Vw, a.ldw, a.H) : matrix_end<E>(w, a.H, a.ldw, a.Vw);
  const int64_t vb = a.v0 - a.wv0;
  NarrowTile<T, !WVH, KT> next;
  auto fetch = [&](int tp) {
    const int64_t v = vb + (int64_t)tp * kNarrowTile;
    next.load(w + (WVH ? v * a.ldw : v), w_end, a.Vw - v);
  };
  s16x8_t q[4 * KT];
  NarrowReader<!WVH> rd;
  rd.init();
  next.init(wave, a.ldw, a.H);
  fetch(first);
  narrow_stay<KT>(q, x + (a.row0 + tw) * ldx, matrix_end<E>(x, rows, ldx, a.H), ldx, a.H);
  const int64_t yy = tok < rows ? a.y[tok] : a.ignore_index;
  next.store(lds);
  __syncthreads();
  for (int tp = first; tp < last; ++tp) {
    char* buf = lds + ((tp - first) & 1) * narrow_buf<KT>();
    fetch(tp + 1);  // (past the last tile too, which nothing uses: behind a branch the registers would be held through the loop)
    f32x16_t acc[kNB][1];
    narrow_logits<T, !WVH, KT>(rd, buf, q, acc);
    // (with the sums of the other kernels, bit for bit: by columns but in the tile of 256 columns that straddles the end)
    const int64_t slice_v0 = a.v0 + (int64_t)tp * kNarrowTile;
    if (slice_v0 / kTile * kTile + kTile <= a.V) {
      FwdColumnState st;
#pragma unroll
      for (int slot = 0; slot < 16; ++slot) fwd_epilogue_slot<T, 0, MON, 1>(a, st, acc, slice_v0, tw, slot);
      const int64_t rel = yy - slice_v0;
      const bool here = yy != a.ignore_index && rel >= 0 && rel < kNarrowTile && ((rel >> 2) & 1) == (lane >> 5);
      fwd_store_target<1>(a, acc, tok, 0, here ? (int)rel : -1);
    } else {
      fwd_epilogue<T, true, MON, 1>(a, rows, acc, slice_v0, tw);
    }
    next.store(lds + ((tp + 1 - first) & 1) * narrow_buf<KT>());
    __syncthreads();
  }
}

// dz of a wave's S: 128 streaming rows x 32 stationary rows, in place.  dx: the stationary row is a token, with its scalars in this lane,
// the streaming ones are columns from v0 on; dW: the other way round, the tokens' scalars in LDS.
constexpr int kNoColumn = -0x7fffffff;
// (label: kNoColumn where there is no column to look for)
LCE_DEV void narrow_scalars(const BwdArgs& a, int64_t rows, int64_t tok, float& nlse, float& gain, int& label) {
  const int64_t yy = tok < rows ? a.y[tok] : a.ignore_index;
  const bool valid = yy != a.ignore_index;
  const float l = valid ? a.lse[tok] : 0.f;
  nlse = valid ? fmaf(-l, kLog2e, (float)a.dz_shift) : -INFINITY;
  gain = 1.f + 2.f * a.z_reg * l;
  if (a.dz_shift != 0) gain = fminf(fmaxf(gain, -63.f), 63.f);  // (as in lce_bwd_dz.hip)
  label = valid && yy >= 0 && yy < a.V ? (int)yy : kNoColumn;
}

// The gradient of one 128-row tile of the stationary matrix over streaming tiles [first, last): acc[hb], rows h along registers,
// stationary rows along lanes.  rows: the tokens that are worked on, all of x's or the packed ones.
template <class T, bool WVH, bool DW, bool ZREG, int KT>
LCE_DEV void narrow_gradient(const BwdArgs& a, int64_t rows, int wave, int tile, int first, int last, char* lds, f32x16_t (&acc)[2 * KT]) {
  typedef typename elem_of<T>::type E;
  constexpr bool TRANS = !DW && !WVH;  // the streaming matrix is W stored (H, V)
  const bool packed = rows != a.N;
  const E* x = reinterpret_cast<const E*>(packed ? a.xc : a.x);
  const int64_t ldx = packed ? a.ldxc : a.ldx;
  const E* w = reinterpret_cast<const E*>(a.w);
  const void* x_end = matrix_end<E>(x, rows, ldx, a.H);
  const void* w_end = WVH ? matrix_end<E>(w, a.Vw, a.ldw, a.H) : matrix_end<E>(w, a.H, a.ldw, a.Vw);
  const int tid = narrow_tid(wave), lane = tid & 63, half = lane >> 5;
  const int64_t r0 = (int64_t)tile * kNarrowTile, rw = r0 + wave * kBlk;
  float* const sh = reinterpret_cast<float*>(lds + 2 * narrow_buf<KT>());  // dW: [2][3][128] nlse, gain, label
  const float c1 = a.scale * kLog2e, one = __builtin_bit_cast(float, (127 + a.dz_shift) << 23);

  NarrowTile<T, TRANS, KT> next;
  // dx: of this lane's token; dW: of the next tile's token threadIdx.x (the upper half of the threads: of none that is used)
  float nlse = 0.f, gain = 0.f;
  int label = 0;
  auto fetch = [&](int tc) {
    const int64_t c = (int64_t)tc * kNarrowTile;
    if (DW) {
      next.load(x + c * ldx, x_end, 0);
      narrow_scalars(a, rows, c + (tid & (kNarrowTile - 1)), nlse, gain, label);
    } else {
      next.load(w + (WVH ? c * a.ldw : c), w_end, a.Vw - c);
    }
  };
  auto put = [&](int n) {
    next.store(lds + (n & 1) * narrow_buf<KT>());
    if (DW && tid < kNarrowTile) {
      float* at = sh + (n & 1) * kNarrowScalars + tid;
      at[0] = nlse;
      at[kNarrowTile] = gain;
      at[2 * kNarrowTile] = __builtin_bit_cast(float, label);
      const int met = __any(label >= (int)r0 && label < (int)r0 + kNarrowTile);
      if ((tid & 63) == 0) at[3 * kNarrowTile - 63 * wave] = __builtin_bit_cast(float, met);  // [3 * 128 + wave]
    }
  };
  s16x8_t q[4 * KT];
  NarrowReader<TRANS> rd;
  rd.init();
  next.init(wave, DW ? ldx : a.ldw, a.H);
  if (DW && !WVH) {
    // (the columns of W that stay, through LDS)
    NarrowTile<T, true, KT> stay;
    NarrowTrans<256> across;
    across.init();
    stay.init(wave, a.ldw, a.H);
    stay.load(w + r0, w_end, a.Vw - r0);
    stay.store(lds);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) across.off[0][k] = (wave & 1) ? across.off[1][k] : across.off[0][k];
#pragma unroll
    for (int ks = 0; ks < 4 * KT; ++ks) q[ks] = across.read(lds + (wave >> 1) * 128, 0, ks);
    __syncthreads();
  } else if (DW) {
    narrow_stay<KT>(q, w + rw * a.ldw, w_end, a.ldw, a.H);
  } else {
    narrow_stay<KT>(q, x + rw * ldx, x_end, ldx, a.H);
  }
#pragma unroll
  for (int hb = 0; hb < 2 * KT; ++hb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[hb][r] = 0.f;
  if (first >= last) return;
  fetch(first);
  if (!DW) narrow_scalars(a, rows, rw + (lane & 31), nlse, gain, label);
  put(0);
  __syncthreads();
  for (int tc = first; tc < last; ++tc) {
    const int n = tc - first;
    const char* buf = lds + (n & 1) * narrow_buf<KT>();
    const float* scal = sh + (n & 1) * kNarrowScalars;
    // (past the last tile too, which nothing uses: behind a branch the registers would be held through the loop)
    if (KT == 1) fetch(tc + 1);
    f32x16_t s[kNB][1];
    narrow_logits<T, TRANS, KT>(rd, buf, q, s);
    // dx: this tile's columns of the vocabulary, and whether a token of the wave has its label among them
    const int64_t v0 = (int64_t)tc * kNarrowTile;
    const int rel = DW ? 0 : (label == kNoColumn ? -1 : (int)(label - v0));
    const bool hit = DW ? __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(scal)[3 * kNarrowTile] | reinterpret_cast<const int*>(scal)[3 * kNarrowTile + 1]) != 0
                        : __any(rel >= 0 && rel < kNarrowTile);
    const int cols = DW ? kNarrowTile : (a.vw - v0 < kNarrowTile ? (int)(a.vw - v0) : kNarrowTile);
    const int my_v = DW ? (int)(rw + (lane & 31)) : 0;
    // (a copy of the loop without what labels and the vocabulary's end ask for, which most tiles do not meet -- where the registers
    // of both fit)
    constexpr bool kOneCopy = KT == 2;
    auto second = [&](auto general) {
      constexpr bool GENERAL = decltype(general)::value;
#pragma unroll
      for (int i = 0; i < kNB; ++i) {
        if (KT == 2 && i == 1) fetch(tc + 1);  // (its registers do not fit before some logits are done with)
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
          const int ks = 2 * i + (g >> 1);  // k-step along the streaming rows
          s16x8_t f[3];  // (two fragments at a time: more do not fit the registers)
          f[0] = rd.b(buf, 0, ks);
          f[1] = rd.b(buf, 1, ks);
          float d[8];
#pragma unroll
          for (int h2 = 0; h2 < 2; ++h2) {
            const int c0 = i * kBlk + 8 * (g + h2) + 4 * half;  // first streaming row of this lane's quad
            f32x4_t nl, ga;
            if (DW) {
              nl = *reinterpret_cast<const f32x4_t*>(scal + c0);
              if (ZREG) ga = *reinterpret_cast<const f32x4_t*>(scal + kNarrowTile + c0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float z = s[i][0][(g + h2) * 4 + j];
              float e = __builtin_amdgcn_exp2f(fmaf(z, c1, DW ? nl[j] : nlse));
              if (ZREG) e *= DW ? ga[j] : gain;
              d[4 * h2 + j] = e;
            }
            if (GENERAL) {
              if (DW) {
                const f32x4_t la = *reinterpret_cast<const f32x4_t*>(scal + 2 * kNarrowTile + c0);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const float lj = la[j];
                  d[4 * h2 + j] = __builtin_bit_cast(int, lj) == my_v ? d[4 * h2 + j] - one : d[4 * h2 + j];
                }
              } else if (!kOneCopy || hit) {
#pragma unroll
                for (int j = 0; j < 4; ++j) d[4 * h2 + j] = rel == c0 + j ? d[4 * h2 + j] - one : d[4 * h2 + j];
              }
            }
            if (GENERAL && !DW && (!kOneCopy || cols < kNarrowTile)) {
#pragma unroll
              for (int j = 0; j < 4; ++j) d[4 * h2 + j] = c0 + j < cols ? d[4 * h2 + j] : 0.f;
            }
          }
          const auto s0 = __builtin_amdgcn_permlane32_swap(pack2<T>(d[0], d[1]), pack2<T>(d[4], d[5]), false, false);
          const auto s1 = __builtin_amdgcn_permlane32_swap(pack2<T>(d[2], d[3]), pack2<T>(d[6], d[7]), false, false);
          u32x4_t o;
          o[0] = s0[0];
          o[1] = s1[0];
          o[2] = s0[1];
          o[3] = s1[1];
          const s16x8_t dz = __builtin_bit_cast(s16x8_t, o);
          if (KT == 2) f[2] = rd.b(buf, 2, ks);
          acc[0] = mfma32<T>(f[0], dz, acc[0]);
          if (KT == 2) f[0] = rd.b(buf, 3, ks);
          acc[1] = mfma32<T>(f[1], dz, acc[1]);
          if constexpr (KT == 2) {
            acc[2] = mfma32<T>(f[2], dz, acc[2]);
            acc[3] = mfma32<T>(f[0], dz, acc[3]);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    };
    if (kOneCopy || hit || cols < kNarrowTile) second(std::true_type());
    else second(std::integral_constant<bool, kOneCopy>());
    put(n + 1);
    __syncthreads();
  }
}

// Element (r, h) of dx (a token's row; of packed tokens the one that perm names) or dW (a column of the vocabulary), four h at a time.
template <class T, bool WVH> LCE_DEV void narrow_out(const BwdArgs& a, int64_t rows, bool dw, float coef, int64_t r, int64_t h, f32x4_t v) {
  typedef typename elem_of<T>::type E;
  if (r >= (dw ? a.V : rows) || h >= a.H) return;
  if (!dw && rows != a.N) r = packed_token(a.perm, r, a.N);
  v *= coef;
  const bool f32 = (dw ? a.dw_dtype : a.dx_dtype) == DT_F32;
  char* out = reinterpret_cast<char*>(dw ? a.dw : a.dx);
  if (!dw || WVH) {  // (a quad that H cuts through is written whole, into the stride padding of its row)
    const int64_t o = r * (dw ? a.lddw : a.lddx) + h;
    if (f32) {
      *reinterpret_cast<f32x4_t*>(out + o * 4) = v;
    } else {
      u32x2_t b;
      b[0] = pack2<T>(v[0], v[1]);
      b[1] = pack2<T>(v[2], v[3]);
      *reinterpret_cast<u32x2_t*>(out + o * 2) = b;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (h + j < a.H) {
        const int64_t o = (h + j) * a.lddw + r;
        if (f32) reinterpret_cast<float*>(out)[o] = v[j];
        else reinterpret_cast<unsigned short*>(out)[o] = to_bits<T>(v[j]);
      }
  }
}

template <class T, bool WVH, bool ZREG, int KT>
__global__ __launch_bounds__(kThreads, 2) void grads_narrow_kernel(const BwdArgs a, const SmallGrads g) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const bool in_first = (int)blockIdx.x < g.first_span, dw = in_first == (g.dw_first != 0);
  const int j = (int)blockIdx.x - (in_first ? 0 : g.first_span), nseg = dw ? g.dw_nseg : g.dx_nseg;
  const int64_t rows = packed_rows(a.n_rows, a.N);
  const int tok_tiles = (int)((rows + kNarrowTile - 1) / kNarrowTile), voc_tiles = (int)((a.vw + kNarrowTile - 1) / kNarrowTile);
  const int tiles = dw ? voc_tiles : tok_tiles, stream = dw ? tok_tiles : voc_tiles;
  if (j >= tiles * nseg) return;  // (there are as many for dx as all tokens ask for)
  int tile, seg;
  segment_coords(j, tiles, nseg, tile, seg);
  const int first = (int)((int64_t)stream * seg / nseg), last = (int)((int64_t)stream * (seg + 1) / nseg);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x16_t acc[2 * KT];
  if (dw) narrow_gradient<T, WVH, true, ZREG, KT>(a, rows, wave, tile, first, last, lds, acc);
  else narrow_gradient<T, WVH, false, ZREG, KT>(a, rows, wave, tile, first, last, lds, acc);
  const int lane = narrow_tid(0), r = wave * kBlk + (lane & 31), hq = 4 * (lane >> 5);
  float* part = nseg > 1 ? g.part + ((dw ? (int64_t)g.dx_blocks : 0) + (int64_t)tile * nseg + seg) * (kNarrowTile * kBK * KT) : nullptr;
  const float coef = final_factor_of(a);
#pragma unroll
  for (int hb = 0; hb < 2 * KT; ++hb)
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const int h = hb * kBlk + 8 * rq + hq;
      f32x4_t v;
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = acc[hb][rq * 4 + k];
      if (part != nullptr) *reinterpret_cast<f32x4_t*>(part + r * (kBK * KT) + h) = v;
      else narrow_out<T, WVH>(a, rows, dw, coef, (int64_t)tile * kNarrowTile + r, h, v);
    }
}

// Adds the parts of the tiles that are cut along the streaming matrix, in order; kParts workgroups to a tile.
constexpr int kParts = 8;
template <class T, bool WVH, int KT>
__global__ __launch_bounds__(256) void narrow_tail_kernel(const BwdArgs a, const SmallGrads g, int dx_tiles) {
  int tile = (int)blockIdx.x / kParts;
  const int piece = (int)blockIdx.x % kParts;
  const bool dw = tile >= dx_tiles;
  if (dw) tile -= dx_tiles;
  const int64_t rows = packed_rows(a.n_rows, a.N);
  if (!dw && (int64_t)tile * kNarrowTile >= rows) return;
  const int nseg = dw ? g.dw_nseg : g.dx_nseg;
  constexpr int kBlockFloats = kNarrowTile * kBK * KT, kQuads = kBlockFloats / 4 / kParts;
  const float* part = g.part + ((dw ? (int64_t)g.dx_blocks : 0) + (int64_t)tile * nseg) * kBlockFloats;
  const float coef = final_factor_of(a);
#pragma unroll
  for (int u = 0; u < kQuads / 256; ++u) {
    // (dW stored (H, V): consecutive threads on consecutive columns of the vocabulary)
    const int i = piece * kQuads + u * 256 + (int)threadIdx.x;
    const bool by_r = dw && !WVH;
    const int r = by_r ? i % kNarrowTile : i / (kBK * KT / 4), h = (by_r ? i / kNarrowTile : i % (kBK * KT / 4)) * 4;
    const float* at = part + r * (kBK * KT) + h;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nseg; s0 += 8) {  // (eight in flight; those that there are not are read again and dropped)
      f32x4_t t[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) t[k] = *reinterpret_cast<const f32x4_t*>(at + (int64_t)(s0 + k < nseg ? s0 + k : s0) * kBlockFloats);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (s0 + k < nseg) v += t[k];
    }
    narrow_out<T, WVH>(a, rows, dw, coef, (int64_t)tile * kNarrowTile + r, h, v);
  }
}

template <class T, bool WVH, int KT> hipError_t launch_grads(const BwdArgs& a, SmallGrads g, bool want_dx, bool want_dw, hipStream_t s) {
  const int64_t tok = want_dx ? (a.N + kNarrowTile - 1) / kNarrowTile : 0, voc = want_dw ? (a.vw + kNarrowTile - 1) / kNarrowTile : 0;
  const int64_t dx_items = tok * g.dx_nseg, dw_items = voc * g.dw_nseg;
  g.first_span = (int)pad_to(g.dw_first ? dw_items : dx_items, 8);  // (workgroup j of either gradient is on XCD j % 8)
  const int64_t grid = g.first_span + (g.dw_first ? dx_items : dw_items);
  if (grid <= 0) return hipSuccess;
  hipError_t e;
  if (a.z_reg != 0.f) {
    static LdsOptIn optin;
    auto kern = grads_narrow_kernel<T, WVH, true, KT>;
    e = optin.ensure(reinterpret_cast<const void*>(kern), narrow_lds<KT>());
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kThreads), narrow_lds<KT>(), s, a, g);
  } else {
    static LdsOptIn optin;
    auto kern = grads_narrow_kernel<T, WVH, false, KT>;
    e = optin.ensure(reinterpret_cast<const void*>(kern), narrow_lds<KT>());
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kThreads), narrow_lds<KT>(), s, a, g);
  }
  e = hipGetLastError();
  const int64_t dx_tails = g.dx_nseg > 1 ? tok : 0, tails = dx_tails + (g.dw_nseg > 1 ? voc : 0);
  if (e != hipSuccess || tails == 0) return e;
  hipLaunchKernelGGL((narrow_tail_kernel<T, WVH, KT>), dim3((unsigned)(tails * kParts)), dim3(256), 0, s, a, g, (int)dx_tails);
  return hipGetLastError();
}
template <class T, bool WVH> hipError_t launch_grads_kt(const BwdArgs& a, const SmallGrads& g, bool dx, bool dw, hipStream_t s) {
  return a.H <= kBK ? launch_grads<T, WVH, 1>(a, g, dx, dw, s) : launch_grads<T, WVH, 2>(a, g, dx, dw, s);
}

template <class T, bool WVH, bool MON, int KT> hipError_t launch_fwd(const FwdArgs& a, int64_t rows, hipStream_t s) {
  const int tiles_p = (int)(pad_to(a.vw, kTile) / kNarrowTile), tiles_q = (int)((rows + kNarrowTile - 1) / kNarrowTile);
  int nseg = (kSmallSlots + tiles_q - 1) / tiles_q;
  if (nseg > tiles_p) nseg = tiles_p;
  auto kern = fwd_narrow_kernel<T, WVH, MON, KT>;
  static LdsOptIn optin;
  hipError_t e = optin.ensure(reinterpret_cast<const void*>(kern), narrow_lds<KT>());
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_q * nseg)), dim3(kThreads), narrow_lds<KT>(), s, a, tiles_p, tiles_q, nseg);
  return hipGetLastError();
}
template <class T, bool WVH, bool MON> hipError_t launch_fwd_kt(const FwdArgs& a, int64_t rows, hipStream_t s) {
  return a.H <= kBK ? launch_fwd<T, WVH, MON, 1>(a, rows, s) : launch_fwd<T, WVH, MON, 2>(a, rows, s);
}
template <class T, bool WVH> hipError_t launch_fwd_mon(const FwdArgs& a, int64_t rows, hipStream_t s) {
  return a.monitoring ? launch_fwd_kt<T, WVH, true>(a, rows, s) : launch_fwd_kt<T, WVH, false>(a, rows, s);
}

}  // namespace

hipError_t launch_fwd_narrow(const FwdArgs& a, int64_t rows, hipStream_t s) {
  if (a.H > kNarrowHidden || a.w_dtype != a.x_dtype || rows <= 0) return hipErrorInvalidValue;
  if (a.x_dtype == DT_BF16) return a.w_vh ? launch_fwd_mon<BF16, true>(a, rows, s) : launch_fwd_mon<BF16, false>(a, rows, s);
  if (a.x_dtype == DT_F16) return a.w_vh ? launch_fwd_mon<F16, true>(a, rows, s) : launch_fwd_mon<F16, false>(a, rows, s);
  return hipErrorInvalidValue;
}

hipError_t launch_bwd_narrow(const BwdArgs& a, const SmallGrads& g, bool want_dx, bool want_dw, hipStream_t s) {
  if (a.H > kNarrowHidden || a.w_dtype != a.x_dtype || a.perm_always || a.dxc != nullptr || a.v0 != 0 || a.wv0 != 0 || a.vw != a.V ||
      ((g.dx_nseg > 1 || g.dw_nseg > 1) && g.part == nullptr))
    return hipErrorInvalidValue;
  if (a.x_dtype == DT_BF16) return a.w_vh ? launch_grads_kt<BF16, true>(a, g, want_dx, want_dw, s) : launch_grads_kt<BF16, false>(a, g, want_dx, want_dw, s);
  if (a.x_dtype == DT_F16) return a.w_vh ? launch_grads_kt<F16, true>(a, g, want_dx, want_dw, s) : launch_grads_kt<F16, false>(a, g, want_dx, want_dw, s);
  return hipErrorInvalidValue;
}

}  // namespace lce
