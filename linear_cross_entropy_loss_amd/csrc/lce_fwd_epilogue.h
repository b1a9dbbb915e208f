// What the forward's tile kernels do with a finished accumulator: per-slice partials of the loss (lce_fwd.hip, lce_narrow.hip).
#pragma once

#include "lce_gemm.h"
#include "lce_internal.h"

namespace lce {

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

LCE_DEV float fast_exp2(float v) { return __builtin_amdgcn_exp2f(v); }
LCE_DEV float fast_log(float v) { return __builtin_amdgcn_logf(v) * kLn2; }

// Reduces a wave's finished 128(v) x 32 NQ(token) accumulator -- the slice that starts at column slice_v0, the tokens from
// row tw of this launch's chunk on -- to the per-slice partials.  Accumulator rows (v) lie along registers and columns
// (tokens) along lanes, so each lane reduces its own tokens in registers and
// meets the other half of the vocabulary slice in lane ^ 32.
//
// VTAIL is the variant for the one tile column that straddles V (V % 256 != 0).
// A register quad covers 4 columns of a run of 8 (lanes l and l+32 hold the two
// halves), so every run but at most one is inside or outside the vocabulary as a
// whole, uniformly over the wave, and is taken or skipped with a scalar branch;
// the one run that V cuts through is handled element by element.
// MON: the monitoring partials (slice max, sum softmax*z, sum z^2) are formed as well.
template <class T, bool VTAIL, bool MON, int NQ>
LCE_DEV void fwd_epilogue(const FwdArgs& a, int64_t rows, f32x16_t (&acc)[kNB][NQ], int64_t slice_v0, int64_t tw) {
  const int lane = opaque_tid() & 63;
  // columns of this wave's slice inside the vocabulary: nq whole runs of 8, then `cut` more columns
  const int64_t left = a.V - slice_v0;
  const int vrem = VTAIL ? (int)(left < 0 ? 0 : (left > kWaveTile ? kWaveTile : left)) : kWaveTile;
  const int nq = vrem >> 3, cut = vrem & 7;
  const int mine = cut - 4 * (lane >> 5);  // elements of this lane's quad of the cut run that exist (<= 0: none)

  const float c1 = a.scale * kLog2e;
  const int64_t slice = slice_v0 / kChunkV;
#pragma unroll
  for (int qb = 0; qb < NQ; ++qb) {
    const int64_t tokl = tw + qb * kBlk + (lane & 31);  // row inside the chunk
    const int64_t tok = a.row0 + tokl;
    const int64_t o = slice * a.nc + tokl;
    if (VTAIL && vrem == 0) {  // nothing of this slice exists
      if (lane < 32) {
        a.part_lse[o] = -INFINITY;
        if (MON) {
          a.part_max[o] = -INFINITY;
          a.part_pz[o] = 0.f;
          a.part_sq[o] = 0.f;
        }
      }
      continue;
    }
    // Column of the target inside this wave's 128-wide slice, or -1.
    const int64_t yy = tok < rows ? a.y[tok] : a.ignore_index;
    const int64_t rel = yy - slice_v0;
    const int yl = (yy != a.ignore_index && rel >= 0 && rel < kWaveTile) ? (int)rel : -1;

    float m = -INFINITY;
#pragma unroll
    for (int pb = 0; pb < kNB; ++pb)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq)
        if (!VTAIL || pb * 4 + rq < nq) {
#pragma unroll
          for (int j = 0; j < 4; ++j) m = fmaxf(m, acc[pb][qb][rq * 4 + j]);
        } else if (pb * 4 + rq == nq && cut != 0) {
#pragma unroll
          for (int j = 0; j < 4; ++j) m = j < mine ? fmaxf(m, acc[pb][qb][rq * 4 + j]) : m;
        }
    m = fmaxf(m, __shfl_xor(m, 32));
    m *= a.scale;  // logit_scale > 0, so max commutes with the scaling
    const float mo = m * kLog2e;
    float s = 0.f, pz = 0.f, sq = 0.f;
    if (MON) {
#pragma unroll
      for (int pb = 0; pb < kNB; ++pb)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq)
          if (!VTAIL || pb * 4 + rq < nq) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float e = fast_exp2(fmaf(acc[pb][qb][rq * 4 + j], c1, -mo));
              const float z = acc[pb][qb][rq * 4 + j] * a.scale;
              s += e;
              pz = fmaf(e, z, pz);
              sq = fmaf(z, z, sq);
            }
          } else if (pb * 4 + rq == nq && cut != 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float e = fast_exp2(fmaf(acc[pb][qb][rq * 4 + j], c1, -mo));
              const float z = acc[pb][qb][rq * 4 + j] * a.scale;
              s += j < mine ? e : 0.f;
              pz = j < mine ? fmaf(e, z, pz) : pz;
              sq = j < mine ? fmaf(z, z, sq) : sq;
            }
          }
      pz += __shfl_xor(pz, 32);
      sq += __shfl_xor(sq, 32);
    } else {
#pragma unroll
      for (int pb = 0; pb < kNB; ++pb)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq)
          if (!VTAIL || pb * 4 + rq < nq) {
#pragma unroll
            for (int j = 0; j < 4; ++j) s += fast_exp2(fmaf(acc[pb][qb][rq * 4 + j], c1, -mo));
          } else if (pb * 4 + rq == nq && cut != 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float e = fast_exp2(fmaf(acc[pb][qb][rq * 4 + j], c1, -mo));
              s += j < mine ? e : 0.f;
            }
          }
    }
    s += __shfl_xor(s, 32);
    if (lane < 32) {
      a.part_lse[o] = m + fast_log(s);
      if (MON) {
        a.part_max[o] = m;
        a.part_pz[o] = pz / s;
        a.part_sq[o] = sq;
      }
    }
    if (yl >= 0 && ((yl >> 2) & 1) == (lane >> 5)) {
      const int want_pb = yl >> 5, want_r = ((yl >> 3) & 3) * 4 + (yl & 3);
      float zt = 0.f;
#pragma unroll
      for (int pb = 0; pb < kNB; ++pb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (pb == want_pb && r == want_r) zt = acc[pb][qb][r];
      a.tgt[tok] = zt * a.scale;
    }
  }
}


// The logit of the target column, written by the one lane that holds it (rare: a wave holds the target of
// one token in a thousand at a vocabulary of 131072).  `yl`: the column inside this wave's 128-wide slice if
// this lane's half holds it, else -1.
template <int NQ>
LCE_DEV void fwd_store_target(const FwdArgs& a, f32x16_t (&acc)[kNB][NQ], int64_t tok, int qb, int yl) {
  if (yl >= 0) {
    const int want = (yl >> 5) * 16 + ((yl >> 3) & 3) * 4 + (yl & 3);  // (block, register) index
    float zt = 0.f;
#pragma unroll
    for (int pb = 0; pb < kNB; ++pb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        // (a volatile read: the compiler would otherwise hoist the 64 accumulator reads above the branch)
        float v;
        asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[pb][qb][r]));
        if (want == pb * 16 + r) zt = v;
      }
    a.tgt[tok] = zt * a.scale;
  }
}

// The same reduction for the kernels whose last K tile is multiplied column by column (Pipe3::step_last_columns:
// all but the tile column that straddles V): one block column of the accumulator at a time -- 32 tokens along the lanes, this
// wave's 128 vocabulary entries of each token in 4 x 16 registers of lanes l and l + 32 -- cut into 16 slots of
// straight-line code that run behind the matrix instructions of the next column.  A lane folds its 64 values
// in two chunks of 32 (slots 8c .. 8c + 7 of chunk c) into a running (max, sum of exp2) pair, so that only 32
// accumulator values are in vector registers at a time, and meets the other half of the slice in lane ^ 32.
struct FwdColumnState {
  float v[32];   // the chunk being summed
  float m, s;    // running max (unscaled logits) and sum of exp2(scaled logit - scaled max)
  float mo;      // scaled max of the chunk being summed
  float e[4], f; // exponentials of the last slot, not yet added; factor for the sum at a chunk change
  float pz, sq;  // monitoring: sum exp2(..) * scaled logit (moves with the max like s) and sum of squared scaled logits
};
// Slot 0..15 of block column QB: the running (max, sum) of this lane's 64 values -- and, MON, the two monitoring
// sums, which leave the arithmetic on (max, sum) as it is, so that the loss does not depend on the monitoring flag
// bit for bit.  The exponentials of a slot are added up in the next one, when they are there.
template <int QB, bool MON, int NQ>
LCE_DEV void fwd_slot_sum(const FwdArgs& a, FwdColumnState& st, f32x16_t (&acc)[kNB][NQ], int slot) {
  const float c1 = a.scale * kLog2e;
  const int c = slot >> 3, sub = slot & 7;  // chunk c: accumulator blocks 2c, 2c + 1, slots 8c .. 8c + 7
  if (slot > 0) {
    st.s += (st.e[0] + st.e[1]) + (st.e[2] + st.e[3]);
    if (MON) {
      const int prev = 4 * ((slot - 1) & 7);  // (the chunk of the previous slot is still in st.v)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = st.v[prev + r] * a.scale;
        st.pz = fmaf(st.e[r], z, st.pz);
        st.sq = fmaf(z, z, st.sq);
      }
    }
  }
  if (sub == 0) {
#pragma unroll
    for (int r = 0; r < 32; ++r) st.v[r] = acc[2 * c + (r >> 4)][QB][r & 15];
    float cm = st.v[0];
#pragma unroll
    for (int r = 1; r < 32; ++r) cm = fmaxf(cm, st.v[r]);
    const float mn = c == 0 ? cm : fmaxf(st.m, cm);
    st.mo = mn * c1;  // logit_scale > 0, so max commutes with the scaling
    if (c == 0) {
      st.s = 0.f;
      if (MON) st.pz = st.sq = 0.f;
    } else {
      st.f = fast_exp2(fmaf(st.m, c1, -st.mo));  // moves the sums to the new max
      st.s *= st.f;
      if (MON) st.pz *= st.f;
    }
    st.m = mn;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) st.e[r] = fast_exp2(fmaf(st.v[4 * sub + r], c1, -st.mo));
  if (slot == 15) {
    st.s += (st.e[0] + st.e[1]) + (st.e[2] + st.e[3]);
    if (MON) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = st.v[28 + r] * a.scale;
        st.pz = fmaf(st.e[r], z, st.pz);
        st.sq = fmaf(z, z, st.sq);
      }
    }
  }
}
// After slot 15: the other half of the slice.  Leaves the slice's max (unscaled) in st.m, its sum of exp2 in st.s
// and, MON, the slice's monitoring sums in st.pz, st.sq.
template <bool MON>
LCE_DEV void fwd_merge_halves(const FwdArgs& a, FwdColumnState& st) {
  const float c1 = a.scale * kLog2e;
  // after the swaps both lanes of a pair hold the lower lane's value in [0] and the upper lane's in [1]
  const unsigned mb = __builtin_bit_cast(unsigned, st.m), sb = __builtin_bit_cast(unsigned, st.s);
  const auto mm = __builtin_amdgcn_permlane32_swap(mb, mb, false, false);
  const auto ss = __builtin_amdgcn_permlane32_swap(sb, sb, false, false);
  // (elements copied to scalars first: a bit cast applied to a vector element reads element 0 whichever is named)
  const unsigned m0u = mm[0], m1u = mm[1], s0u = ss[0], s1u = ss[1];
  const float m0 = __builtin_bit_cast(float, m0u), m1 = __builtin_bit_cast(float, m1u);
  const float s0 = __builtin_bit_cast(float, s0u), s1 = __builtin_bit_cast(float, s1u);
  const float mt = fmaxf(m0, m1), mo = mt * c1;
  const float f0 = fast_exp2(fmaf(m0, c1, -mo)), f1 = fast_exp2(fmaf(m1, c1, -mo));
  st.s = s0 * f0 + s1 * f1;
  st.m = mt;
  if (MON) {
    const unsigned pb = __builtin_bit_cast(unsigned, st.pz), qb = __builtin_bit_cast(unsigned, st.sq);
    const auto pp = __builtin_amdgcn_permlane32_swap(pb, pb, false, false);
    const auto qq = __builtin_amdgcn_permlane32_swap(qb, qb, false, false);
    const unsigned p0u = pp[0], p1u = pp[1], q0u = qq[0], q1u = qq[1];
    st.pz = __builtin_bit_cast(float, p0u) * f0 + __builtin_bit_cast(float, p1u) * f1;
    st.sq = __builtin_bit_cast(float, q0u) + __builtin_bit_cast(float, q1u);
  }
}
// tw: first token row of the wave inside this launch's chunk (like slice_v0 uniform over the wave).
template <class T, int QB, bool MON, int NQ>
LCE_DEV void fwd_epilogue_slot(const FwdArgs& a, FwdColumnState& st, f32x16_t (&acc)[kNB][NQ], int64_t slice_v0, int64_t tw, int slot) {
  fwd_slot_sum<QB, MON, NQ>(a, st, acc, slot);
  if (slot == 15) {
    fwd_merge_halves<MON>(a, st);
    // one store per token and partial: the upper lanes get an offset that the range check of the buffer store drops
    const int lane = threadIdx.x & 63;
    const int64_t o = slice_v0 / kChunkV * a.nc + tw + QB * kBlk;
    const int voff = lane < 32 ? lane * 4 : (int)0x80000000;
    auto store = [&](float* base, float v) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(base + o, 0, kBlk * 4, 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc, voff, 0, 0);
    };
    store(a.part_lse, fmaf(st.m, a.scale, fast_log(st.s)));
    if (MON) {
      store(a.part_max, st.m * a.scale);
      store(a.part_pz, st.pz / st.s);
      store(a.part_sq, st.sq);
    }
  }
}

}  // namespace

}  // namespace lce
