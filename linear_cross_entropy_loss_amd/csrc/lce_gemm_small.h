// The logit contraction on 128 (P) x 128 (Q) output tiles, one workgroup per tile, for problems with few tiles.
//
// The persistent kernels (lce_gemm3.h) are made for long launches: their code is 25 to 90 KB, straight through, and every
// compute unit fetches it from L2 when a launch starts, which takes 10 to 14 us, and a 256 x 256 tile is much work for one
// compute unit where there are fewer tiles than those.  Here a tile is a quarter of that, two workgroups share a compute
// unit, and the code of a kernel is a few KB: the K loop is two K tiles long, the epilogue handles a quarter of the
// accumulators.  What that costs is LDS traffic, five fragment reads for four matrix instructions (eight for sixteen there).
//
// A wave has all 128 P rows (one slice of the vocabulary, as the waves of the persistent kernels have) of 32 Q rows, so that
// the epilogues are those of the persistent kernels on one accumulator column.  Operands are staged in the same LDS layouts by
// the same stagers, 16 KiB each per stage.  Two K tiles are in flight in registers while a third is multiplied: with few
// workgroups the loop is bound by the latency of memory, not by the matrix cores.
#pragma once

#include <type_traits>

#include "lce_gemm3.h"

namespace lce {

constexpr int kSmallTile = 128;
constexpr int kSmallOperandBytes = kSmallTile * kBK * 2;
constexpr int kSmallStageBytes = 2 * kSmallOperandBytes;
constexpr int kSmallLds = 2 * kSmallStageBytes;  // 64 KiB: two workgroups to a compute unit

// The P operand from fp32 rows, rounded to the compute type (pairs: to the hi or the lo part that the step multiplies) on its way to
// LDS, with the rounding of convert_w_slab_kernel.  As Stager3 otherwise: a thread moves eight numbers at a time, two loads and
// one store, into the same LDS layouts.
template <class T, bool KC, int CHUNKS> struct StagerF32 {
  struct Regs {
    u32x4_t v[CHUNKS][2];
  };
  static constexpr int kRowPieces = CHUNKS * 4, kRowsAtOnce = kThreads / kRowPieces;
  const char* base;
  const char* end;
  unsigned range, voff, voff_cur, iter_stride;
  int kpos, lds_off;
  int64_t k_stride;
  bool lo;  // pairs: which part of the numbers is stored

  LCE_DEV void init(int64_t ld) {
    const int t = threadIdx.x;
    if (KC) {
      const int c = t & 7, r = t >> 3;
      voff = (unsigned)((r * ld + c * 8) * 4);
      iter_stride = (unsigned)(32 * ld * 4);
      k_stride = kBK * 4;
      lds_off = r * 128 + ((c ^ (r & 7) ^ ((r >> 3) & 1)) << 4);
      kpos = c * 8;
    } else {
      const int c = t % kRowPieces, k = t / kRowPieces, j = k & 3;
      voff = (unsigned)((k * ld + c * 8) * 4);
      iter_stride = (unsigned)(kRowsAtOnce * ld * 4);
      k_stride = (int64_t)kBK * ld * 4;
      lds_off = k * (kRowPieces * 16) + ((c << 4) ^ (((j & 1) << 7) | ((j >> 1) << 6) | ((j & 1) << 5)));
      kpos = 0;
    }
    voff_cur = voff;
    base = end = nullptr;
    range = 0;
    lo = false;
  }
  LCE_DEV void retarget(int k_rem) {
    const int64_t left = end - base;
    range = left <= 0 ? 0u : left > 0x7fffffff ? 0x7fffffffu : (unsigned)left;
    if (KC) voff_cur = kpos < k_rem ? voff : 0x80000000u;
  }
  LCE_DEV void load(Regs& r, int i0, int i1) const {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, (int)range, 0x00020000);
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      r.v[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)voff_cur, (int)(i * iter_stride), 0);
      r.v[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)voff_cur + 16, (int)(i * iter_stride), 0);
    }
  }
  LCE_DEV void store(const Regs& r, char* tile, int i0, int i1) const {
    constexpr int step = KC ? 32 * 128 : kRowsAtOnce * kRowPieces * 16;
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      float f[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const unsigned u = r.v[i][k >> 2][k & 3];
        f[k] = __builtin_bit_cast(float, u);
        if (is_pair<T>::value && lo) f[k] = bf16_lo(f[k]);
      }
      u32x4_t o;
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = pack2<T>(f[2 * k], f[2 * k + 1]);
      *reinterpret_cast<u32x4_t*>(tile + lds_off + i * step) = o;
    }
  }
};

// NP, NQ: blocks of 32 P / Q rows of a wave, four accumulator blocks together: 4, 1 for the logits; 2, 2 for the gradients, whose
// epilogues do not need a slice of the vocabulary in one wave and whose fragment reads are then four for four products.
// Q_BLOCKED, SWAP: Problem::kQBlocked and kSwapAB of Pipe3.
template <class T, bool P_KC, bool Q_KC = true, bool Q_BLOCKED = false, int NP = 4, int NQ = 1, bool SWAP = false,
          bool P_F32 = false> struct SmallPipe {
  static_assert(NP * NQ == kNB, "four accumulator blocks to a wave");
  typedef typename elem_of<T>::type E;
  static constexpr bool kSplit = is_pair<T>::value;
  static constexpr bool kQRowBlocks = Q_BLOCKED && !Q_KC;
  static constexpr int kWavesP = kNB / NP;
  typedef typename std::conditional<P_F32, StagerF32<T, P_KC, 4>, Stager3<T, E, P_KC, true, 4>>::type PStager;
  typedef Stager3<T, E, Q_KC, true, 4> QStager;
  PStager ps;
  QStager qs;
  FragReader<P_KC, kSmallTile> pr;
  FragReader<Q_KC, kSmallTile> qr;
  typename PStager::Regs sp[2];  // K tiles t + 1 and t + 2 while t is multiplied; set t & 1
  typename QStager::Regs sq[2];
  int k_rem, split_s;
  int64_t p_lo, q_lo;
  int q_phase;     // as in Pipe3
  int64_t q_jump;

  s16x8_t pf[2][NP], qf[2][NQ];  // fragments of this k-step and the next

  LCE_DEV void advance() {
    if constexpr (kSplit) {
      if (split_s != 2) {
        ps.base += split_s == 0 ? 0 : p_lo;
        qs.base += split_s == 0 ? q_lo : -q_lo;
        ++split_s;
        if constexpr (P_F32) ps.lo = split_s == 1;  // (the K tile stored next is two before the one loaded next: one after it, modulo 3)
        ps.retarget(k_rem);
        qs.retarget(k_rem);
        return;
      }
      ps.base -= p_lo;
      split_s = 0;
      if constexpr (P_F32) ps.lo = false;
    }
    ps.base += ps.k_stride;
    if constexpr (kQRowBlocks) {
      qs.base += q_phase == 3 ? q_jump : qs.k_stride;
      q_phase = (q_phase + 1) & 3;
    } else {
      qs.base += qs.k_stride;
    }
    k_rem -= kBK;
    ps.retarget(k_rem);
    qs.retarget(k_rem);
  }
  // Chunks 0 .. 7 of a staged K tile: those of P and of Q in turn.
  template <int SET> LCE_DEV void load_chunks(int c0, int c1) {
#pragma unroll
    for (int c = c0; c < c1; ++c) {
      if (c & 1) qs.load(sq[SET], c >> 1, (c >> 1) + 1);
      else ps.load(sp[SET], c >> 1, (c >> 1) + 1);
    }
  }
  template <int SET> LCE_DEV void store_chunks(char* stage, int c0, int c1) {
#pragma unroll
    for (int c = c0; c < c1; ++c) {
      if (c & 1) qs.store(sq[SET], stage + kSmallOperandBytes, c >> 1, (c >> 1) + 1);
      else ps.store(sp[SET], stage, c >> 1, (c >> 1) + 1);
    }
  }
  LCE_DEV void read_frags(const char* stage, int ks) {
#pragma unroll
    for (int j = 0; j < NQ; ++j) qf[ks & 1][j] = qr.read(stage + kSmallOperandBytes, j, ks);
#pragma unroll
    for (int i = 0; i < NP; ++i) pf[ks & 1][i] = pr.read(stage, i, ks);
  }
  LCE_DEV void multiply(int ks, f32x16_t (&acc)[NP][NQ]) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int jj = 0; jj < NQ; ++jj) {
        const int j = (i & 1) ? NQ - 1 - jj : jj;
        acc[i][j] = SWAP ? mfma32<T>(qf[ks & 1][j], pf[ks & 1][i], acc[i][j]) : mfma32<T>(pf[ks & 1][i], qf[ks & 1][j], acc[i][j]);
      }
  }
  static constexpr int kReads = NQ * (Q_KC ? 1 : 2) + NP * (P_KC ? 1 : 2);  // LDS reads of a k-step's fragments
  // What goes behind each of a k-step's four matrix instructions: a quarter of the next one's reads, stores and loads in turn.
  template <int STORES, int LOADS> LCE_DEV void order() {
    if constexpr (P_F32) {  // (with the conversions in between, left to the compiler)
      __builtin_amdgcn_sched_barrier(0);
      return;
    }
    __builtin_amdgcn_sched_group_barrier(LCE_SG_MFMA, 1, 0);
    __builtin_amdgcn_sched_group_barrier(LCE_SG_DS_RD, kReads - 3 * (kReads / 4), 0);
    if (STORES > 0) __builtin_amdgcn_sched_group_barrier(LCE_SG_DS_WR, 1, 0);
#pragma unroll
    for (int i = 1; i < kNB; ++i) {
      __builtin_amdgcn_sched_group_barrier(LCE_SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(LCE_SG_DS_RD, kReads / 4, 0);
      if (i < STORES) __builtin_amdgcn_sched_group_barrier(LCE_SG_DS_WR, 1, 0);
      if (i >= kNB - LOADS) __builtin_amdgcn_sched_group_barrier(LCE_SG_VMEM_RD, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // One K tile, t, held in `cur`, the fragments of its first k-step in registers: K tile t + 1 goes from set SET to `next`, which
  // takes K tile t + 3 in its place, chunk by chunk; the barrier opens the last k-step, and the fragments of K tile t + 1's
  // first k-step are read during it.  (Left to the compiler, which put all stores first and all loads last: N=1536, V=2560, H=2048
  // 31 us, so 24; N=48, V=50304, H=2048 43, so 39, which is 5.3 TB/s of weight.)
  template <int SET> LCE_DEV void step(const char* cur, char* next, f32x16_t (&acc)[NP][NQ]) {
    read_frags(cur, 1);
    store_chunks<SET>(next, 0, 3);
    load_chunks<SET>(0, 3);
    multiply(0, acc);
    order<3, 3>();
    read_frags(cur, 2);
    store_chunks<SET>(next, 3, 6);
    load_chunks<SET>(3, 6);
    multiply(1, acc);
    order<3, 3>();
    read_frags(cur, 3);
    store_chunks<SET>(next, 6, 8);
    load_chunks<SET>(6, 8);
    multiply(2, acc);
    order<2, 2>();
    advance();
    __syncthreads();
    read_frags(next, 0);
    multiply(3, acc);
    order<0, 0>();
  }
  // p, q: first element of the tile's operands; *_end: one past the last valid byte; ktiles: even, or 0.  Q_BLOCKED: ldq and q_phase_
  // as in Pipe3.
  LCE_DEV void run(const void* p, const void* p_end, int64_t ldp, const void* q, const void* q_end, int64_t ldq, int64_t k_valid,
                   int ktiles, int64_t p_lo_, int64_t q_lo_, char* lds, f32x16_t (&acc)[NP][NQ], int q_phase_ = 0) {
    const int wave = (int)(threadIdx.x >> 6);
    ps.init(ldp);
    if constexpr (Q_BLOCKED) {
      qs.init_blocked(kSplit ? 2 : 1);
      q_jump = ldq * ((kSplit ? 2 : 1) * kTile * kBK * QStager::kEs) - 3 * qs.k_stride;
      q_phase = q_phase_;
    } else {
      qs.init(ldq);
    }
    pr.init(wave % kWavesP * (NP * kBlk));
    qr.init(wave / kWavesP * (NQ * kBlk));
    ps.base = reinterpret_cast<const char*>(p);
    ps.end = reinterpret_cast<const char*>(p_end);
    qs.base = reinterpret_cast<const char*>(q);
    qs.end = reinterpret_cast<const char*>(q_end);
    k_rem = (int)k_valid;
    split_s = 0;
    p_lo = p_lo_;
    q_lo = q_lo_;
    ps.retarget(k_rem);
    qs.retarget(k_rem);
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int j = 0; j < NQ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    load_chunks<0>(0, 8);
    advance();
    load_chunks<1>(0, 8);
    advance();
    store_chunks<0>(lds, 0, 8);
    load_chunks<0>(0, 8);
    advance();
    __syncthreads();
    read_frags(lds, 0);
    // (K tiles past the last one are fetched as zeros: masked in the K-contiguous operand, out of range in the other)
    for (int t = 0; t < ktiles; t += 2) {
      step<1>(lds, lds + kSmallStageBytes, acc);
      step<0>(lds + kSmallStageBytes, lds, acc);
    }
    __syncthreads();  // (the epilogue may use the stages)
  }
};

}  // namespace lce
