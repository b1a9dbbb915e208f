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

#include "lce_gemm3.h"

namespace lce {

constexpr int kSmallTile = 128;
constexpr int kSmallOperandBytes = kSmallTile * kBK * 2;
constexpr int kSmallStageBytes = 2 * kSmallOperandBytes;
constexpr int kSmallLds = 2 * kSmallStageBytes;  // 64 KiB: two workgroups to a compute unit

template <class T, bool P_KC> struct SmallPipe {
  typedef typename elem_of<T>::type E;
  static constexpr bool kSplit = is_pair<T>::value;
  typedef Stager3<T, E, P_KC, true, 4> PStager;
  typedef Stager3<T, E, true, true, 4> QStager;
  PStager ps;
  QStager qs;
  FragReader<P_KC, kSmallTile> pr;
  FragReader<true, kSmallTile> qr;
  typename PStager::Regs sp[2];  // K tiles t + 1 and t + 2 while t is multiplied; set t & 1
  typename QStager::Regs sq[2];
  int k_rem, split_s;
  int64_t p_lo, q_lo;

  LCE_DEV void fetch(int set) {  // the K tile the stream is at, and on to the next
    ps.load(sp[set], 0, 4);
    qs.load(sq[set], 0, 4);
    if constexpr (kSplit) {
      if (split_s != 2) {
        ps.base += split_s == 0 ? 0 : p_lo;
        qs.base += split_s == 0 ? q_lo : -q_lo;
        ++split_s;
        ps.retarget(k_rem);
        qs.retarget(k_rem);
        return;
      }
      ps.base -= p_lo;
      split_s = 0;
    }
    ps.base += ps.k_stride;
    qs.base += qs.k_stride;
    k_rem -= kBK;
    ps.retarget(k_rem);
    qs.retarget(k_rem);
  }
  LCE_DEV void stash(int set, char* stage) {
    ps.store(sp[set], stage, 0, 4);
    qs.store(sq[set], stage + kSmallOperandBytes, 0, 4);
  }
  LCE_DEV void multiply(const char* stage, f32x16_t (&acc)[kNB][1]) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const s16x8_t q = qr.read(stage + kSmallOperandBytes, 0, ks);
#pragma unroll
      for (int i = 0; i < kNB; ++i) acc[i][0] = mfma32<T>(pr.read(stage, i, ks), q, acc[i][0]);
    }
  }
  // p, q: first element of the tile's operands; *_end: one past the last valid byte; ktiles: even, as in Pipe3, or 0.
  LCE_DEV void run(const void* p, const void* p_end, int64_t ldp, const void* q, const void* q_end, int64_t ldq, int64_t k_valid,
                   int ktiles, int64_t p_lo_, int64_t q_lo_, char* lds, f32x16_t (&acc)[kNB][1]) {
    ps.init(ldp);
    qs.init(ldq);
    pr.init(0);
    qr.init((int)(threadIdx.x >> 6) * kBlk);
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
    for (int i = 0; i < kNB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][0][r] = 0.f;
    fetch(0);
    fetch(1);
    stash(0, lds);
    fetch(0);
    __syncthreads();
    // (K tiles past the last one are fetched as zeros: masked in the K-contiguous operand, out of range in the other)
    for (int t = 0; t < ktiles; t += 2) {
      stash(1, lds + kSmallStageBytes);
      fetch(1);
      multiply(lds, acc);
      __syncthreads();
      stash(0, lds);
      fetch(0);
      multiply(lds + kSmallStageBytes, acc);
      __syncthreads();
    }
  }
};

}  // namespace lce
