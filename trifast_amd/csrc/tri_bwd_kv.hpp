// Backward kernel 2 of 3: dk and dv.
//
// Work unit: (batch*head, R consecutive pair rows i, block of NW*32 keys).  Wave w
// owns one tile of 32 keys for all R rows: its K and V rows (B operands) and the
// dk, dv accumulators stay in registers, and the queries of the rows are streamed
// through LDS in tiles of BJ (direct global->LDS loads, double-buffered, swizzled;
// rows of Q and dO, the lse and delta operand words left by the dq kernel, and the packed
// bias tiles).  With one pair row per workgroup the 16-bit types also have a version whose tiles are 32 queries, whatever BJ says, in
// a ring of four (RING, see bwd_kv_ring).  Scores are computed UN-transposed here, S = Q K^T, so that a lane
// owns one key (column) and 16 queries of every 32-query tile: P and dS are then
// already in B-operand layout for the two products that contract over queries,
//   dv^T += dO^T P,   dk^T += Q^T dS,   dk = dk^T / sqrt(d),
// whose A operands dO^T, Q^T come from the natural tiles through transposing LDS
// reads.  The per-element additive terms ride on the matrix pipe: the bias tile
// (fp32, raw-score domain, converted once per stage and shared by the R rows) is
// the accumulator init of the score MFMA, and the per-query terms -lse*sqrt(d) and
// -delta enter through one extra MFMA each (see rank1_operand, OffsetMask), so that
// P = exp2(c * acc) and dS = P * dP' are one multiply each.  Masked keys get a large
// negative score from the MFMA that adds -lse, which makes their P and dS zero.
//
// Replaces _bwd_kv of reference src/trifast/triton.py:143-263.
#pragma once
#include <type_traits>

#include "tri_args.hpp"
#include "tri_common.hpp"
#include "tri_f32_plain.hpp"
#include "tri_tile.hpp"

namespace tri {

// LDS bytes of a stage: Q rows of the R pair rows | dO rows | lse2 | -delta | packed bias tiles
// (fp32: the rows as three parts, words and bias in registers)
constexpr int bwd_kv_stage_bytes(int D, int es, int NW, int R, int BJ) {
  return 2 * R * BJ * lds_row_bytes(D, es) + (es == 4 ? 0 : 2 * R * BJ * 4 + NW * (BJ / 32) * 2048);
}

// The ring of 32-query stages (one pair row, 16-bit types; whole loads for every wave): a stage's rows and bias tiles, then lse2 and -delta
// of its queries once per wave.
constexpr int kBwdKVStages = 4;
// Where there is a version with the ring, and the rows that take it: all at head dim 64. At 32 and 128 its stages, twice as many, cost
// more than their waits where the other version's last stage of 64 queries is more than half full, and save the empty half of it where it is not
// (this kernel alone, stages of 64 / ring, bf16, h = 4, us: d = 128, n = 100 29.9 / 31.4, 256 160.4 / 163.5, 300 293.5 / 304.3, 384 436 / 446, 500 934 / 956,
// 768 2740 / 2790; n = 160 76.9 / 72.2, 200 124.0 / 117.9, 600 1551 / 1527; d = 32, n = 300 73.5 / 78.3, 384 111 / 114; h = 8, n = 96 14.6 / 13.9; h = 2, n = 600 211 / 211,
// with padding 195 / 184, 850 562 / 570, with padding 505 / 479; d = 64, n = 384 186.2 / 182.6, 401 267 / 237, 512 387 / 386, 700 1007 / 957, 900 2148 / 2022).
constexpr bool bwd_kv_ring(int D, int es, int R) { return es == 2 && R == 1 && D >= 32; }
constexpr bool bwd_kv_ring_always(int D) { return D == 64; }
constexpr bool bwd_kv_ring_pays(int n) { return (n - 1) % 64 < 32; }
constexpr int bwd_kv_ring_stage_bytes(int D, int es, int NW) { return ring_stage_bytes(D, es, NW, 1) + NW * 256; }
// LDS bytes of a workgroup
constexpr int bwd_kv_lds_bytes(int D, int es, int NW, int R, int BJ, int nbuf, bool ring) {
  return ring ? kBwdKVStages * bwd_kv_ring_stage_bytes(D, es, NW) : nbuf * bwd_kv_stage_bytes(D, es, NW, R, BJ);
}

// Two waves per SIMD (at most 256 registers) wherever the tile fits them or nearly
// does: a few registers over would otherwise halve the occupancy.
template <typename T, int D, int R, int BJ>
constexpr int bwd_kv_min_waves() {
  constexpr int row_bytes = D * (int)sizeof(T);
  if (sizeof(T) == 4) return R == 1 && D != 64 ? 2 : 1;
  return (row_bytes >= 512 || (row_bytes == 128 && R == 1) || (row_bytes <= 64 && R * BJ <= 64)) ? 2 : 1;
}

template <typename T, int D, int NW, int R, int BJ, int NBUF, bool RING>
__global__ __launch_bounds__(NW * 64, (bwd_kv_min_waves<T, D, R, BJ>())) void tri_bwd_kv_kernel(const BwdArgs a) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using Tile = typename OperandOffsets<T, D>::Tile;
  constexpr int KP = E::KP;
  constexpr int DS = D / (2 * KP);
  constexpr int DM = (D + 31) / 32;
  constexpr int PS = 32 / (2 * KP);
  constexpr int JU = BJ / 32;
  constexpr int ROWB = lds_row_bytes(D, (int)sizeof(T));
  // one stage: Q rows of the R pair rows | dO rows | lse2 | -delta | packed bias tiles
  constexpr int OFF_Q = 0, OFF_DO = R * BJ * ROWB, OFF_LSE = 2 * R * BJ * ROWB;
  constexpr int WORDS = sizeof(T) == 4 ? 0 : R * BJ * 4;
  constexpr int OFF_DELTA = OFF_LSE + WORDS, OFF_B = OFF_DELTA + WORDS;
  constexpr int BIAS_B = sizeof(T) == 4 ? 0 : 2 * 64 * 8 * (int)sizeof(T);
  constexpr int STAGE = OFF_B + NW * JU * BIAS_B;
  static_assert(STAGE == bwd_kv_stage_bytes(D, (int)sizeof(T), NW, R, BJ), "the launcher sizes LDS with bwd_kv_stage_bytes");
  static_assert(sizeof(T) == 4 || (R * BJ) % 64 == 0, "lse/delta rows are loaded in whole waves");
  extern __shared__ __attribute__((aligned(16))) unsigned char tri_smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kl = lane & 31, g = lane >> 5;
  const int N = a.N;
  int bx, by;
  xcd_remap(gridDim.x, bx, by);
  const int i0 = by * R;
  if (i0 >= N) return;
  const int bh = blockIdx.z;
  const int b = bh / a.H, h = bh % a.H;
  const int k_wave = bx * (NW * 32) + wave * 32;
  const int key = k_wave + kl;
  const bool wave_active = k_wave < N;
  const int kt = min(k_wave >> 5, a.NP - 1);

  const T* qbh = reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h;
  const T* kbh = reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h;
  const T* vbh = reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h;
  const T* dobh = reinterpret_cast<const T*>(a.dout) + b * a.sdo.b + h * a.sdo.h;
  const T* pack_bh = reinterpret_cast<const T*>(a.packk) + (int64_t)bh * a.NP * a.NP * 1024;
  const float* lse2_bh = reinterpret_cast<const float*>(a.lse2) + (int64_t)bh * N * N;    // 32-bit words, moved as floats
  const float* delta_bh = reinterpret_cast<const float*>(a.delta) + (int64_t)bh * N * N;

  // per-row state: K and V tiles as B operands (lane owns key k_wave + kl).  A
  // fully masked row drops the q.k and bias terms from its scores: its K operand
  // is zero here (K itself is not needed for dk, dv) and it skips the bias.
  bool flagged[R], tile_live[R];
  frag kf[R][DS], vf[R][DS];
  typename E::ofrag keyop[R];  // ones | mask element of this lane's key: B operand of the offset-and-mask MFMA
  f32x16 dkacc[R][DM], dvacc[R][DM];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = min(i0 + r, N - 1);  // rows past the end repeat the last one and are not stored
    // (wave-uniform values, pinned to scalar registers so that the branches on
    // them are real branches and not lane masks)
    flagged[r] = __builtin_amdgcn_readfirstlane(a.rowflag[(int64_t)b * N + i]) != 0;
    const int w = k_wave >> 5;
    const uint32_t word = __builtin_amdgcn_readfirstlane((wave_active && w < a.nwords) ? a.keep[((int64_t)b * N + i) * a.nwords + w] : 0u);
    tile_live[r] = word != 0;
    {
      typename OffsetMask<T>::Keys ko;
      ko.init(kl, g);
      keyop[r] = ko.masked(word);
    }
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const int dofs = 2 * KP * s + KP * g;
      const int kc = min(key, N - 1);
      kf[r][s] = flagged[r] ? E::zero() : E::load(kbh + i * a.sk.i + (int64_t)kc * a.sk.j + dofs);
      vf[r][s] = E::load(vbh + i * a.sv.i + (int64_t)kc * a.sv.j + dofs);
    }
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      dkacc[r][mt] = zero16();
      dvacc[r][mt] = zero16();
    }
  }

  // lane-constant LDS offsets: Q and dO rows as natural operands (tile row m stands
  // for query perm32(m)) and again through transposing reads
  OperandOffsets<T, D> ofs;
  ofs.init(perm32(kl), lane);

  // per-lane source pointers of the stage tiles for queries 0..BJ-1
  std::conditional_t<sizeof(T) == 4, SplitStream<D, R * BJ, NW>, TileStream<T, D, R * BJ, NW>> qstream, dostream;
  qstream.init([&](int x) { return qbh + min(i0 + x / BJ, N - 1) * a.sq.i + (int64_t)(x % BJ) * a.sq.j; }, wave, lane);
  dostream.init([&](int x) { return dobh + min(i0 + x / BJ, N - 1) * a.sdo.i + (int64_t)(x % BJ) * a.sdo.j; }, wave, lane);
  FloatStream<sizeof(T) == 4 ? 64 : R * BJ, NW> lstream, dstream;  // (16-bit types)
  if constexpr (sizeof(T) == 2) {
    lstream.init([&](int x) { return lse2_bh + (int64_t)min(i0 + x / BJ, N - 1) * N + x % BJ; }, wave, lane);
    dstream.init([&](int x) { return delta_bh + (int64_t)min(i0 + x / BJ, N - 1) * N + x % BJ; }, wave, lane);
  }
  float lw_x[R][JU], dw_x[R][JU], lw_cur[R][JU], dw_cur[R][JU];  // fp32: the words of this lane's queries, next and current stage
  const T* bias_lane = pack_bh + ((int64_t)kt * 2 * 64 + lane) * 8;

  // Stage loads: direct global->LDS.  A ragged last stage clamps query indices: a
  // clamped row duplicates the last valid one, and the compute of that stage gives
  // the duplicates P = dS = 0.
  f32x4 bias_x[JU][4];   // fp32: packed bias words on their way
  f32x16 bias_cur[JU];   // fp32: the bias tiles of the stage in use
  auto issue_loads = [&](int jt0, int buf) {
    unsigned char* st = tri_smem + buf * STAGE;
    auto q_row = [&](int x) { return qbh + min(i0 + x / BJ, N - 1) * a.sq.i + (int64_t)min(jt0 + x % BJ, N - 1) * a.sq.j; };
    auto do_row = [&](int x) { return dobh + min(i0 + x / BJ, N - 1) * a.sdo.i + (int64_t)min(jt0 + x % BJ, N - 1) * a.sdo.j; };
    if (jt0 + BJ <= N) {
      if constexpr (sizeof(T) == 4) {
        // (into registers; store_loads() writes them once the stage in use has been computed)
        qstream.load((int64_t)jt0 * a.sq.j);
        dostream.load((int64_t)jt0 * a.sdo.j);
      } else {
        qstream.issue(st + OFF_Q, (int64_t)jt0 * a.sq.j, wave);
        dostream.issue(st + OFF_DO, (int64_t)jt0 * a.sdo.j, wave);
      }
      if constexpr (sizeof(T) == 2) {
        lstream.issue(reinterpret_cast<float*>(st + OFF_LSE), jt0, wave);
        dstream.issue(reinterpret_cast<float*>(st + OFF_DELTA), jt0, wave);
      }
    } else {
      asm volatile("" ::);  // keeps this rare path a real branch
      if constexpr (sizeof(T) == 4) {
        qstream.load_rows(q_row);
        dostream.load_rows(do_row);
      } else {
        Tile::template fill<R * BJ, NW>(st + OFF_Q, q_row, wave, lane);
        Tile::template fill<R * BJ, NW>(st + OFF_DO, do_row, wave, lane);
      }
      if constexpr (sizeof(T) == 2) {
        fill_floats<R * BJ, NW>(reinterpret_cast<float*>(st + OFF_LSE), [&](int x) {
          return lse2_bh + (int64_t)min(i0 + x / BJ, N - 1) * N + min(jt0 + x % BJ, N - 1); }, wave, lane);
        fill_floats<R * BJ, NW>(reinterpret_cast<float*>(st + OFF_DELTA), [&](int x) {
          return delta_bh + (int64_t)min(i0 + x / BJ, N - 1) * N + min(jt0 + x % BJ, N - 1); }, wave, lane);
      }
    }
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < JU; ++u) {
          const int64_t at = (int64_t)min(i0 + r, N - 1) * N + min(jt0 + 32 * u + perm32(kl), N - 1);
          lw_x[r][u] = lse2_bh[at];
          dw_x[r][u] = delta_bh[at];
        }
    }
#pragma unroll
    for (int u = 0; u < JU; ++u) {
      const T* p = bias_lane + (int64_t)min((jt0 >> 5) + u, a.NP - 1) * a.NP * 1024;
#pragma unroll
      for (int r2 = 0; r2 < 2; ++r2) {
        if constexpr (sizeof(T) == 4) {
          // (fp32: into registers, which leaves LDS room for another workgroup)
          bias_x[u][2 * r2] = *reinterpret_cast<const f32x4*>(p + r2 * 512);
          bias_x[u][2 * r2 + 1] = *reinterpret_cast<const f32x4*>(p + r2 * 512 + 4);
        } else {
          unsigned char* dst = st + OFF_B + (wave * JU + u) * BIAS_B + r2 * (BIAS_B / 2);
          __builtin_amdgcn_global_load_lds((const TRI_G1 void*)(p + r2 * 512), (TRI_L3 void*)dst, 16, 0, 0);
        }
      }
    }
  };
  auto store_loads = [&](int buf) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < JU; ++u) {
          lw_cur[r][u] = lw_x[r][u];
          dw_cur[r][u] = dw_x[r][u];
        }
#pragma unroll
      for (int u = 0; u < JU; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) bias_cur[u][e] = bias_x[u][e / 4][e % 4] * a.sqrt_d;
      qstream.store(tri_smem + buf * STAGE + OFF_Q);
      dostream.store(tri_smem + buf * STAGE + OFF_DO);
    }
  };
  // sqrt(d) * bias through the matrix pipe (16-bit types): the packed words of a bias tile are a B
  // operand as they are, against a constant A operand with sqrt(d) where the contraction slot is
  // the row's own index (sqrt(32) and sqrt(128) as hi + lo parts).  With one pair row per
  // workgroup a bias tile serves one tile of scores, and converting it on the vector ALU, 32
  // instructions beside the 56 of the tile itself, costs more: n = 768, h = 8, d = 64 2.78 -> 2.56 ms, n = 384, b = 2 825 -> 724 us.
  constexpr int NPART = D == 32 || D == 128 ? 2 : 1;
  frag bsel[2][NPART];
  if constexpr (sizeof(T) == 2) {
    typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
    const T hi = (T)a.sqrt_d;
    const T part[2] = {hi, (T)(a.sqrt_d - (float)hi)};
#pragma unroll
    for (int r2 = 0; r2 < 2; ++r2)
#pragma unroll
      for (int pp = 0; pp < NPART; ++pp) {
        const int e = perm32(kl) - 16 * r2 - 8 * g;
        const uint32_t bits = (uint32_t)__builtin_bit_cast(uint16_t, part[pp]) << (16 * (e & 1));
        u32x4v w;
#pragma unroll
        for (int x = 0; x < 4; ++x) w[x] = (e >= 0 && e < 8 && (e >> 1) == x) ? bits : 0u;
        asm volatile("" : "+v"(w));
        bsel[r2][pp] = __builtin_bit_cast(frag, w);
      }
  }
  auto bias_from_lds = [&](const unsigned char* st, int u) -> f32x16 {
    const unsigned char* src = st + OFF_B + (wave * JU + u) * BIAS_B;
    f32x16 bv = zero16();
#pragma unroll
    for (int r2 = 0; r2 < 2; ++r2) {
      const frag x = *reinterpret_cast<const frag*>(src + r2 * (BIAS_B / 2) + lane * 16);
#pragma unroll
      for (int pp = 0; pp < NPART; ++pp) bv = E::mfma(bsel[r2][pp], x, bv);
    }
    return bv;
  };
  // the per-query operand word (lse or delta term) of the query this lane's A
  // operand row stands for, in tile (r, u)
  const float c = a.c;
  typename OffsetMask<T>::Queries lseop;  // the query's -lse word | ones: A operand of that MFMA
  lseop.init(0u, g);
  auto query_word = [&](const unsigned char* st, int off, int r, int u) -> uint32_t {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(uint32_t, (off == OFF_LSE ? lw_cur : dw_cur)[r][u]);
    return reinterpret_cast<const uint32_t*>(st + off)[r * BJ + 32 * u + perm32(kl)];
  };

  // One stage of compute.  The JU*R tiles run as a software pipeline inside the
  // wave: the two MFMA chains (scores, dP) of tile t+1 are issued before the
  // exponentials of tile t.  EDGE stages hold queries past the end.
  // COMMON stages belong to a wave none of whose rows is fully masked or has a dead key
  // tile: the stage then has no branch, and the MFMA chains of the next tile are
  // scheduled into the vector arithmetic of the current one (branches would split them
  // into blocks of their own).
  auto compute_stage = [&](auto edge_tag, auto common_tag, int jt0, int buf) __attribute__((always_inline)) {
    constexpr bool EDGE = decltype(edge_tag)::value;
    constexpr bool COMMON = decltype(common_tag)::value && !EDGE;
    const unsigned char* st = tri_smem + buf * STAGE;
    if (!wave_active) return;
    constexpr int TS = JU * R;
    f32x16 biasv[JU];
#pragma unroll
    for (int u = 0; u < JU; ++u) {
      if constexpr (sizeof(T) == 4) biasv[u] = bias_cur[u];
      else biasv[u] = bias_from_lds(st, u);
    }

    // scores: bias tile (accumulator init) - lse*sqrt(d) (per query, one MFMA) + Q K^T;
    // dP - delta: -delta (per query, one MFMA) + dO V^T
    auto chains = [&](int t, f32x16& sc, f32x16& dp) {
      const int u = t / R, r = t % R;
      const unsigned char* qt = st + OFF_Q + (r * BJ + 32 * u) * ROWB;
      const unsigned char* dot = st + OFF_DO + (r * BJ + 32 * u) * ROWB;
      uint32_t lw = query_word(st, OFF_LSE, r, u);
      if constexpr (EDGE) {
        // queries past the end: a huge lse makes their P and dS zero
        if (jt0 + 32 * u + perm32(kl) >= N) lw = split_word<T>(E::kMaskElem);
      }
      const typename E::ofrag ones = E::osplat(1.0f);
      // -lse per query and the key mask through one MFMA (see OffsetMask; the roles of
      // the two operands are swapped here: rows are queries, columns are keys)
      lseop.set(lw, g);
      if (COMMON || !flagged[r]) {
        sc = E::mfma(lseop.get(), keyop[r], biasv[u]);
      } else {
        // rare: kept a real branch so that the common case starts from the bias
        // tile in place (a select between the two inits would copy 16 registers)
        asm volatile("" ::);
        sc = E::mfma(lseop.get(), keyop[r], zero16());
      }
      dp = E::mfma(rank1_operand<T>(query_word(st, OFF_DELTA + (sizeof(T) == 4), r, u), g), ones, zero16());
#pragma unroll
      for (int sd = 0; sd < DS; ++sd) {
        sc = E::mfma(ofs.natural(qt, sd), kf[r][sd], sc);
        dp = E::mfma(ofs.natural(dot, sd), vf[r][sd], dp);
      }
    };

    f32x16 sc, dp;
    chains(0, sc, dp);
#pragma unroll
    for (int t = 0; t < TS; ++t) {
      const int u = t / R, r = t % R;
      f32x16 sn, dn;
      if (t + 1 < TS) chains(t + 1, sn, dn);
      if (COMMON || (tile_live[r] && (!EDGE || jt0 + 32 * u < N))) {
        float p[16], ds[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          p[v] = fast_exp2(sc[v] * c);
          ds[v] = p[v] * dp[v];
        }
#pragma unroll
        for (int s2 = 0; s2 < PS; ++s2) {
          const frag pf = E::pack(&p[KP * s2]);
          const frag dsf = E::pack(&ds[KP * s2]);
#pragma unroll
          for (int mt = 0; mt < DM; ++mt) {
            dvacc[r][mt] = E::mfma(ofs.transposed(st + OFF_DO + (r * BJ + 32 * u) * ROWB, s2, mt), pf, dvacc[r][mt]);
            dkacc[r][mt] = E::mfma(ofs.transposed(st + OFF_Q + (r * BJ + 32 * u) * ROWB, s2, mt), dsf, dkacc[r][mt]);
          }
        }
      }
      if (t + 1 < TS) { sc = sn; dp = dn; }
    }
  };

  // The stages as a ring of four tiles of 32 queries: while a tile's sums are made the scores and dP of the tile after it start, from a stage
  // that has landed, and the loads of the two stages behind that one are in flight, with a counted wait and one barrier per stage.
  // What bounded the double buffer was the wait for everything in flight at the end of each stage, 20 spilled registers and
  // the general loop that a ragged end takes; outputs are the same bits.  Whole steps, h = 4, d = 64, bf16: n = 401
  // 779 -> 735 us, b = 2, n = 512 with 300 valid 1961 -> 1916; h = 2: n = 1000 3962 -> 3902, d = 128, n = 600 2522 -> 2506; h = 8,
  // n = 768 in fp16 7854 -> 7844 (the chip lowers its clock there).  Without the scores a stage ahead n = 1000 takes 3924 and n = 768 7935; three
  // stages and three waves per SIMD, which spill 12 registers, 4473 and 9054.
  auto ring_loop = [&](auto common_tag, auto stages_tag) __attribute__((always_inline)) {
    constexpr bool COMMON = decltype(common_tag)::value;
    using Ring = StageRing<T, D, NW, 1, decltype(stages_tag)::value>;
    constexpr int NS = Ring::NS, RSTAGE = bwd_kv_ring_stage_bytes(D, (int)sizeof(T), NW), NLD = Ring::NLD + 1;
    const int ns = (N + 31) >> 5;
    Ring ring;
    ring.init(a.sq, a.sdo, qbh, dobh, pack_bh + (int64_t)kt * 1024, a.NP * 1024, N, i0, wave, lane, tri_smem);
    const uint32_t* const words = reinterpret_cast<const uint32_t*>(g ? delta_bh : lse2_bh) + (int64_t)i0 * N;
    auto issue = [&](int boff) {
      const uint32_t* src = words + min(32 * ring.pos + kl, N - 1);
      const uint32_t dst = __builtin_amdgcn_readfirstlane(ring.lds0 + (uint32_t)(boff + Ring::FSTAGE + wave * 256));
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(dst), "v"(src) : "memory", "m0");
      ring.issue(boff, ns, wave, lane);
    };
    const typename E::ofrag ones = E::osplat(1.0f);
    auto chains = [&](int stage, int boff, f32x16& sc, f32x16& dp) __attribute__((always_inline)) {
      const unsigned char* st = tri_smem + boff;
      const uint32_t* w = reinterpret_cast<const uint32_t*>(st + Ring::FSTAGE + wave * 256) + perm32(kl);
      uint32_t lw = w[0];
      if (32 * stage + perm32(kl) >= N) lw = split_word<T>(E::kMaskElem);  // queries past the end: P = dS = 0
      lseop.set(lw, g);
      f32x16 bv = zero16();
      if (COMMON || !flagged[0]) {
        const unsigned char* src = st + Ring::FOFF_B + wave * 2048;
#pragma unroll
        for (int r2 = 0; r2 < 2; ++r2) {
          const frag x = *reinterpret_cast<const frag*>(src + r2 * 1024 + lane * 16);
#pragma unroll
          for (int pp = 0; pp < NPART; ++pp) bv = E::mfma(bsel[r2][pp], x, bv);
        }
      }
      sc = E::mfma(lseop.get(), keyop[0], bv);
      dp = E::mfma(rank1_operand<T>(w[32], g), ones, zero16());
#pragma unroll
      for (int sd = 0; sd < DS; ++sd) {
        sc = E::mfma(ofs.natural(st, sd), kf[0][sd], sc);
        dp = E::mfma(ofs.natural(st + Ring::FOFF_V, sd), vf[0][sd], dp);
      }
    };
    auto sums = [&](int boff, const f32x16& sc, const f32x16& dp) __attribute__((always_inline)) {
      const unsigned char* st = tri_smem + boff;
      float p[16], ds[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        p[v] = fast_exp2(sc[v] * c);
        ds[v] = p[v] * dp[v];
      }
#pragma unroll
      for (int s2 = 0; s2 < PS; ++s2) {
        const frag pf = E::pack(&p[KP * s2]);
        const frag dsf = E::pack(&ds[KP * s2]);
#pragma unroll
        for (int mt = 0; mt < DM; ++mt) {
          dvacc[0][mt] = E::mfma(ofs.transposed(st + Ring::FOFF_V, s2, mt), pf, dvacc[0][mt]);
          dkacc[0][mt] = E::mfma(ofs.transposed(st, s2, mt), dsf, dkacc[0][mt]);
        }
      }
    };
#pragma unroll
    for (int st = 0; st < NS - 1; ++st) issue(st * RSTAGE);
    wait_dma_known();  // (the loads of the prologue are not in flight any more as far as the compiler's own waits go)
    auto up = [](int boff) { return boff == (NS - 1) * RSTAGE ? 0 : boff + RSTAGE; };
    auto down = [](int boff) { return boff == 0 ? (NS - 1) * RSTAGE : boff - RSTAGE; };
    int boff = 0;
    // Both versions of the loop, which may run side by side in a workgroup, meet at the same barriers and use the buffers alike: behind the
    // one of stage s the stages up to s + 1 have landed, the last reads of stage s - 1 are made, and stage s + 3 is
    // requested into its buffer.
    ring_sync<(NS - 2) * NLD>();
    auto advance = [&] {
      ring_sync<(NS - 3) * NLD>();
      issue(down(boff));
    };
    int s = 0;
    if constexpr (COMMON) {
      f32x16 sa, da, sb, db;
      chains(0, 0, sa, da);
      auto trip = [&](int stage, const f32x16& s0, const f32x16& d0, f32x16& s1, f32x16& d1) __attribute__((always_inline)) {
        advance();
        chains(stage + 1, up(boff), s1, d1);
        sums(boff, s0, d0);
        boff = up(boff);
      };
      for (; s + 2 < ns; s += 2) {
        trip(s, sa, da, sb, db);
        trip(s + 1, sb, db, sa, da);
      }
      if (s + 1 < ns) {
        trip(s, sa, da, sb, db);
        sums(boff, sb, db);
      } else {
        sums(boff, sa, da);
      }
    } else {
      for (; s < ns; ++s) {
        if (s + 1 < ns) advance();
        if (tile_live[0]) {
          f32x16 sc, dp;
          chains(s, boff, sc, dp);
          sums(boff, sc, dp);
        }
        boff = up(boff);
      }
    }
    wait_dma();  // (the last prefetches are still on their way into LDS)
  };

  if constexpr (RING) {
    constexpr std::integral_constant<int, kBwdKVStages> stages{};
    if (wave_active && !flagged[0] && tile_live[0]) ring_loop(std::true_type{}, stages);
    else ring_loop(std::false_type{}, stages);
  } else {
    // Stages that lie inside the query range run in the main loop; a ragged last
    // stage runs after it with the edge handling.
    const int nfull = N / BJ;  // whole stages
    const bool ragged = N % BJ != 0;
    if constexpr (NBUF == 2) {
      issue_loads(0, 0);
      store_loads(0);
      wait_dma();
      __syncthreads();
      // (the whole loop exists twice; a wave picks its version once.  Both run the same
      // stages and barriers.)
      auto whole_stages = [&](auto common_tag) __attribute__((always_inline)) {
        int s = 0;
        for (; s + 1 < nfull; s += 2) {
          issue_loads((s + 1) * BJ, 1);
          compute_stage(std::false_type{}, common_tag, s * BJ, 0);
          store_loads(1);
          wait_dma();
          __syncthreads();
          if ((s + 2) * BJ < N) issue_loads((s + 2) * BJ, 0);
          compute_stage(std::false_type{}, common_tag, (s + 1) * BJ, 1);
          if ((s + 2) * BJ < N) store_loads(0);
          wait_dma();
          __syncthreads();
        }
        return s;
      };
      bool common = wave_active;
#pragma unroll
      for (int r = 0; r < R; ++r) common = common && !flagged[r] && tile_live[r];
      const int s = common ? whole_stages(std::true_type{}) : whole_stages(std::false_type{});
      // buffer 0 now holds stage s: the last whole one, the ragged one, or a spare
      if (s < nfull) {
        if (ragged) issue_loads((s + 1) * BJ, 1);
        compute_stage(std::false_type{}, std::false_type{}, s * BJ, 0);
        if (ragged) {
          store_loads(1);
          wait_dma();
          __syncthreads();
          compute_stage(std::true_type{}, std::false_type{}, (s + 1) * BJ, 1);
        }
      } else if (ragged) {
        compute_stage(std::true_type{}, std::false_type{}, s * BJ, 0);
      }
    } else {
      // one stage only (the double buffer does not fit in LDS): load, then compute
      for (int s = 0; s < nfull; ++s) {
        issue_loads(s * BJ, 0);
        store_loads(0);
        wait_dma();
        __syncthreads();
        compute_stage(std::false_type{}, std::false_type{}, s * BJ, 0);
        __syncthreads();
      }
      if (ragged) {
        issue_loads(nfull * BJ, 0);
        store_loads(0);
        wait_dma();
        __syncthreads();
        compute_stage(std::true_type{}, std::false_type{}, nfull * BJ, 0);
      }
    }
  }

  if (!wave_active) return;
  float check = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = i0 + r;
    if (i >= N) continue;
    T* dkrow = reinterpret_cast<T*>(a.dk) + b * a.sdk.b + h * a.sdk.h + i * a.sdk.i + key * a.sdk.j;
    T* dvrow = reinterpret_cast<T*>(a.dv) + b * a.sdv.b + h * a.sdv.h + i * a.sdv.i + key * a.sdv.j;
    store_rows_any<T, D, DM>(dkrow, dkacc[r], a.scale, g, key < N);
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) check = finite_check<(D < 32 ? 8 : 16)>(dkacc[r][mt], check);
    }
    store_rows_any<T, D, DM>(dvrow, dvacc[r], 1.0f, g, key < N);
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) check = finite_check<(D < 32 ? 8 : 16)>(dvacc[r][mt], check);
    }
  }
  if constexpr (sizeof(T) == 4) {
    if (__any(!(check == 0.f))) plain_dkv<D, R>(arg_words(), bh, i0, k_wave, fresh_lane());
  }
}

}  // namespace tri
