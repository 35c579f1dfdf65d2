// Results of an fp32 wave that are not all finite, computed again number by number.
//
// The fp32 kernels run on three bf16 parts per number (see Elem<float>).  An infinity has no remainder
// there, and its products with the parts of another number, zeros and either sign among them, add up
// to NaN, also in the number that was split beside it; a number that rounds to infinity in bf16 and
// products past the end of fp32 go the same way.  fp32 itself knows better: an infinite value makes its
// own column infinite, a score of -inf has the probability zero.  So each wave looks at what it has
// computed (one instruction per result register), and one that finds something not
// finite does its part again here, with fp32 multiply-adds and the same formulas.  (Wave by wave: to
// agree on it the waves of a workgroup would have to meet, which took 1.7 % of a step at n = 110.)
//
// Only such waves come here, and what bounds these loops is of no interest; a sum that has become NaN
// stays so, and its loop ends there (n = 512: with v NaN throughout a step took 154 ms without that;
// with q, k and v NaN it takes 2.9 with it, as for finite numbers).  They keep few numbers alive: the
// kernels' own code in a second version for the fp32 matrix pipe in their place took the forward at
// d = 32 from three waves per SIMD to two.
#pragma once
#include "tri_args.hpp"
#include "tri_common.hpp"

namespace tri {

// 0 as long as everything that went in is finite.  VALUES: how many of a lane's 16 values stand for
// something (8 in the output tile of head dim 16, whose upper rows no operand is defined for and
// which hold whatever the registers did).
template <int VALUES>
TRI_DEV float finite_check(const f32x16& v, float acc) {
#pragma unroll
  for (int e = 0; e < VALUES; ++e) acc = __builtin_fmaf(v[e], 0.f, acc);
  return acc;
}

// What a kernel hands to the functions at the end of this file: where the launch put its arguments,
// and the lane, neither of which it has to keep through its own work for that (kept, the
// arguments spilled up to 40 scalar registers, and the fp32 step at n = 110, d = 64 took 1.6 % longer).
typedef const __attribute__((address_space(4))) uint32_t* ArgWords;
TRI_DEV ArgWords arg_words() { return (ArgWords)__builtin_amdgcn_kernarg_segment_ptr(); }
TRI_DEV int fresh_lane() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}
template <typename Args>
TRI_DEV Args read_args(ArgWords at) {
  static_assert(sizeof(Args) % 4 == 0);
  struct {
    uint32_t w[sizeof(Args) / 4];
  } copy;
#pragma unroll
  for (unsigned i = 0; i < sizeof(Args) / 4; ++i) copy.w[i] = at[i];
  return __builtin_bit_cast(Args, copy);
}

// x . y, rows of D numbers (rolled: nothing of a row stays in registers)
template <int D>
TRI_DEV float plain_dot(const float* x, const float* y, float acc) {
#pragma unroll 1
  for (int c = 0; c < D; c += 4) {
    const f32x4 xv = *reinterpret_cast<const f32x4*>(x + c), yv = *reinterpret_cast<const f32x4*>(y + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_fmaf(xv[e], yv[e], acc);
  }
  return acc;
}
template <int W>
TRI_DEV void plain_axpy(float (&acc)[W], float p, const float* x) {
#pragma unroll
  for (int c = 0; c < W; c += 4) {
    const f32x4 xv = *reinterpret_cast<const f32x4*>(x + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[c + e] = __builtin_fmaf(p, xv[e], acc[c + e]);
  }
}
template <int W>
TRI_DEV void plain_store(float* dst, const float (&acc)[W], float mul) {
#pragma unroll
  for (int c = 0; c < W; c += 4) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[c + e] * mul;
    *reinterpret_cast<f32x4*>(dst + c) = v;
  }
}

// A pair row's part of a problem, and its raw scores as the kernels define them: sqrt(d) bias + q . k,
// with the mask value on top for keys that are not attended; a fully masked row has the mask value
// (here: none) alone.  Key tiles without an attended key are left out, as in the kernels.
template <int D, typename Args>
struct PlainRow {
  const float *q, *k, *v, *packq;
  const uint32_t* keep;
  int64_t sq, sk, sv;
  bool flagged;
  int NP;
  float sqrt_d;
  TRI_DEV PlainRow(const Args& a, int bh, int i) {
    const int b = bh / a.H, h = bh % a.H;
    q = reinterpret_cast<const float*>(a.q) + b * a.sq.b + h * a.sq.h + i * a.sq.i;
    k = reinterpret_cast<const float*>(a.k) + b * a.sk.b + h * a.sk.h + i * a.sk.i;
    v = reinterpret_cast<const float*>(a.v) + b * a.sv.b + h * a.sv.h + i * a.sv.i;
    sq = a.sq.j, sk = a.sk.j, sv = a.sv.j;
    packq = reinterpret_cast<const float*>(a.packq) + (int64_t)bh * a.NP * a.NP * 1024;
    keep = a.keep + ((int64_t)b * a.N + i) * a.nwords;
    flagged = a.rowflag[(int64_t)b * a.N + i] != 0;
    NP = a.NP;
    sqrt_d = a.sqrt_d;
  }
  TRI_DEV bool live(int key) const { return keep[key >> 5] != 0; }
  TRI_DEV float score(int j, int key) const {
    if (flagged) return 0.f;
    const int r = key >> 4 & 1, g = key >> 3 & 1;  // (the layout of the packed bias: see BiasPrepArgs)
    const float bias = packq[((((int64_t)(j >> 5) * NP + (key >> 5)) * 2 + r) * 64 + (j & 31) + 32 * g) * 8 + (key & 7)];
    const float s = plain_dot<D>(q + j * sq, k + key * sk, bias * sqrt_d);
    return keep[key >> 5] >> (key & 31) & 1u ? s : s + 4.0f * Elem<float>::kMaskElem;
  }
};

// Queries j_blk .. j_blk + 31 of one pair row by a wave: lane t takes query t % 32 and half of the
// columns.
template <int D>
TRI_DEV void plain_fwd_row(const FwdArgs& a, int bh, int i, int j_blk, int lane) {
  constexpr int W = D / 2 < 32 ? D / 2 : 32;
  const int j = j_blk + lane % 32, half = lane / 32;
  if (j >= a.N) return;
  const PlainRow<D, FwdArgs> row(a, bh, i);
  float top = kNeg, sum = 0.f;
  for (int key = 0; key < a.N && top == top; ++key)
    if (row.live(key)) {
      const float s = row.score(j, key);
      top = s == s ? fmaxf(top, s) : s;
    }
  float* o = reinterpret_cast<float*>(a.o) + (((int64_t)bh * a.N + i) * a.N + j) * D;
#pragma unroll 1
  for (int c0 = half * (D / 2); c0 < (half + 1) * (D / 2); c0 += W) {
    float acc[W] = {};
    sum = 0.f;
    for (int key = 0; key < a.N; ++key) {
      if (!row.live(key)) continue;
      const float p = fast_exp2((row.score(j, key) - top) * a.c);
      sum += p;
      plain_axpy(acc, p, row.v + key * row.sv + c0);
      if (sum != sum) break;
    }
    plain_store(o + c0, acc, 1.0f / sum);
  }
  if (half == 0) a.lse[((int64_t)bh * a.N + i) * a.N + j] = kLn2 * (top * a.c + fast_log2(sum)) + (row.flagged ? a.neg_inf : 0.f);
}

// P and dS of one query and key, from the per-query words of the dq kernel
template <int D>
TRI_DEV float plain_dscore(const BwdArgs& a, const PlainRow<D, BwdArgs>& row, const float* dout, int64_t words, int j, int key, float& p) {
  const float nlse = reinterpret_cast<const float*>(a.lse2)[words + j], ndelta = reinterpret_cast<const float*>(a.delta)[words + j];
  p = fast_exp2((row.score(j, key) + nlse) * a.c);
  return p * plain_dot<D>(dout, row.v + key * row.sv, ndelta);
}
TRI_DEV const float* plain_dout(const BwdArgs& a, int bh, int i) {
  return reinterpret_cast<const float*>(a.dout) + bh / a.H * a.sdo.b + bh % a.H * a.sdo.h + i * a.sdo.i;
}

// dq of queries j_blk .. j_blk + 31, lanes as above
template <int D>
TRI_DEV void plain_dq_row(const BwdArgs& a, int bh, int i, int j_blk, int lane) {
  constexpr int W = D / 2 < 32 ? D / 2 : 32;
  const int j = j_blk + lane % 32, half = lane / 32;
  if (j >= a.N) return;
  const PlainRow<D, BwdArgs> row(a, bh, i);
  const float* dout = plain_dout(a, bh, i) + j * a.sdo.j;
  const int64_t words = ((int64_t)bh * a.N + i) * a.N;
  float* dq = reinterpret_cast<float*>(a.dq) + bh / a.H * a.sdq.b + bh % a.H * a.sdq.h + i * a.sdq.i + j * a.sdq.j;
#pragma unroll 1
  for (int c0 = half * (D / 2); c0 < (half + 1) * (D / 2); c0 += W) {
    float acc[W] = {};
    for (int key = 0; key < a.N; ++key) {
      if (!row.live(key)) continue;
      float p;
      const float ds = plain_dscore<D>(a, row, dout, words, j, key, p);
      plain_axpy(acc, ds, row.k + key * row.sk + c0);
      if (ds != ds) break;
    }
    plain_store(dq + c0, acc, a.scale);
  }
}

// dk and dv of keys k_blk .. k_blk + 31: lane t takes key t % 32, and dk or dv
template <int D>
TRI_DEV void plain_dkv_row(const BwdArgs& a, int bh, int i, int k_blk, int lane) {
  constexpr int W = D < 32 ? D : 32;
  const int key = k_blk + lane % 32;
  const bool is_dk = lane < 32;
  if (key >= a.N) return;
  const PlainRow<D, BwdArgs> row(a, bh, i);
  const float* dout = plain_dout(a, bh, i);
  const int64_t words = ((int64_t)bh * a.N + i) * a.N;
  const Str5& st = is_dk ? a.sdk : a.sdv;
  float* out = reinterpret_cast<float*>(is_dk ? a.dk : a.dv) + bh / a.H * st.b + bh % a.H * st.h + i * st.i + key * st.j;
#pragma unroll 1
  for (int c0 = 0; c0 < D; c0 += W) {
    float acc[W] = {};
    if (row.live(key))
      for (int j = 0; j < a.N; ++j) {
        float p;
        const float ds = plain_dscore<D>(a, row, dout + j * a.sdo.j, words, j, key, p);
        const float* from = is_dk ? row.q + j * row.sq : dout + j * a.sdo.j;
        const float w = is_dk ? ds : p;
        plain_axpy(acc, w, from + c0);
        if (w != w) break;
      }
    plain_store(out + c0, acc, is_dk ? a.scale : 1.0f);
  }
}

// db of a block of queries and keys, summed over the pair rows of its chunk in order; the lanes take the
// pairs of the block in turn
template <int D, int BJ, int BKB>
TRI_DEV void plain_db_block(const BwdArgs& a, int bh, int chunk, int j_blk, int k_blk, int i_begin, int i_end, int lane) {
  for (int x = lane; x < BJ * BKB; x += 64) {
    const int j = j_blk + x % BJ, key = k_blk + x / BJ;
    if (j >= a.N || key >= a.N) continue;
    float acc = 0.f;
    for (int i = i_begin; i < i_end && acc == acc; ++i) {
      const PlainRow<D, BwdArgs> row(a, bh, i);
      if (!row.live(key)) continue;
      float p;
      acc += plain_dscore<D>(a, row, plain_dout(a, bh, i) + j * a.sdo.j, ((int64_t)bh * a.N + i) * a.N, j, key, p);
    }
    if (a.nchunks == 1) reinterpret_cast<float*>(a.db)[bh / a.H * a.sdb_b + bh % a.H * a.sdb_h + j * a.sdb_j + key * a.sdb_k] = acc;
    else a.dbpart[(((int64_t)chunk * a.BH + bh) * a.N + j) * a.N + key] = acc;
  }
}

// The same for a wave that found something not finite.  Called, not inlined: with these loops in their
// bodies the kernels' own loops got other registers (at d = 64 dk/dv 2 % slower, the step
// 0.7 %); at d = 128 dk/dv, which spills, is 2 % slower with the look at its results alone.
#define TRI_CALLED __device__ __attribute__((noinline))
template <int D, int R>
TRI_CALLED void plain_fwd(ArgWords at, int bh, int i0, int j_blk, int lane) {
  const FwdArgs a = read_args<FwdArgs>(at);
  for (int r = 0; r < R && i0 + r < a.N; ++r) plain_fwd_row<D>(a, bh, i0 + r, j_blk, lane);
}
template <int D, int R>
TRI_CALLED void plain_dq(ArgWords at, int bh, int i0, int j_blk, int lane) {
  const BwdArgs a = read_args<BwdArgs>(at);
  for (int r = 0; r < R && i0 + r < a.N; ++r) plain_dq_row<D>(a, bh, i0 + r, j_blk, lane);
}
template <int D, int R>
TRI_CALLED void plain_dkv(ArgWords at, int bh, int i0, int k_blk, int lane) {
  const BwdArgs a = read_args<BwdArgs>(at);
  for (int r = 0; r < R && i0 + r < a.N; ++r) plain_dkv_row<D>(a, bh, i0 + r, k_blk, lane);
}
template <int D, int BJ, int BKB>
TRI_CALLED void plain_db(ArgWords at, int bh, int chunk, int j_blk, int k_blk, int i_begin, int i_end, int lane) {
  plain_db_block<D, BJ, BKB>(read_args<BwdArgs>(at), bh, chunk, j_blk, k_blk, i_begin, i_end, lane);
}

}  // namespace tri
