// Row-resident backward: dq, dk and dv of one pair row from ONE computation of the
// scores and of dP (the dq kernel and the dk/dv kernel each recompute both).
//
// Work unit: (batch*head, pair row i), one workgroup of four waves, one wave per
// SIMD with the whole register file.  (Rows of up to 64 bytes and 512 keys have a kernel of their own, of one or two
// waves: tri_bwd_row_short.hpp.)  The keys of the row are dealt to the waves
// in tiles of 32 (wave w owns key tiles w, w+4, ...; at most KT of them): their
// dk, dv accumulators stay in registers for the whole row, their V rows too (B
// operands; in a private piece of LDS where the registers do not hold them all), and
// the K row of the pair row sits in LDS for the whole workgroup (read as B operand of
// the scores and, transposed, as A operand of dq).  The queries of the row are
// streamed through LDS in tiles of 32 (Q, dO rows, direct global->LDS loads, three
// stages: in use, ready, in flight).  Per (query tile, key tile), with the scores
// un-transposed (a lane owns one key and 16 queries):
//   S  = Q K^T + sqrt(d) (bias - lse)      every term through the matrix pipe (below)
//   P  = exp2(c S)
//   dP = dO V^T - delta
//   dS = P * dP
//   dv^T += dO^T P,  dk^T += Q^T dS        P, dS are B operands as they are
//   dq^T += K^T dS^T                       dS goes through a 2 KiB LDS tile of the wave
//                                          and comes back transposed (ds_read_tr)
// Everything additive is a matrix product, which leaves the per-tile vector work free of
// conversions, selects and adds (matrix and full-rate vector time add up within a wave,
// so this costs what it saves for the bias; it makes masked rows cost what unmasked ones
// do and frees the registers the converted tiles took).  The packed bias words of a tile are A operands as they
// are (a lane owns a query and eight keys) against a constant B operand that holds
// sqrt(d) where the contraction slot is the column's key; -lse sqrt(d) and -delta (per
// query) and the key mask (per key) are rank-1 products of operand words.  That leaves
// the vector ALU one multiply and one exp2 per score, one multiply per dS and the two
// conversions.  dq of a query tile is the sum of the four waves' partial tiles: they
// meet in LDS once per query tile (one barrier) and each wave adds a quarter of the tile, its
// own part first and then the others' in wave order (deterministic, no atomics), behind the
// MFMAs that start the next query tile.
// The four waves share the LDS pipe, and an LDS instruction occupies it for four cycles
// whatever its width (transposing reads move half of what 16-byte reads do): operands
// that do not change over the key tiles of a query tile (Q^T, dO^T) are read once per
// query tile where the registers allow.
//
// The prologue also computes delta = rowsum(o * do) of the row and leaves it, with
// the row's log-sum-exp, in the per-query planes the db kernel reads.
//
// In rows of one pass the loop over the query tiles has no branch: the compiler sinks what stands in front of one behind it, out of the schedule.
// Lanes and waves without a share are masked with exec inside asm statements, pointers advance by masked steps, transposing reads past the
// columns of a short row return bytes nobody uses; nothing of the loop lies in scratch (a reload waits for every load in flight).  (Not so
// in rows of 128 bytes with four key tiles per wave, which the tuner alone takes: 11 reloads per query tile and a branch around the words; rows of several
// passes branch on the first one; of the short rows 32 wide those of two waves with eight key tiles reload 16 bytes.)  It
// is why masked key operands are made in the step and not kept.  Before that, on one card, this kernel alone, h = 4: d = 16, n = 700
// 786 -> 652 us, n = 1024 1964 -> 1607; d = 32, n = 600 546 -> 530, n = 768 951 -> 939, n = 1024 1995 -> 1980 (bound by issue and clock);
// d = 64, n = 300 219 -> 195, h = 8, n = 256 240 -> 228, fp16, two of n = 384 with half of the keys masked 1172 -> 1140.
//
// Rows up to 128*KT keys fit (1024 keys at head dim 32).  Longer rows run the kernel in
// several passes (MULTI), one launch per 128*KT keys: dk and dv of a pass's keys are complete
// after it, dq is the sum over the passes and travels from one to the next as two numbers of
// the element type per value (the rounded running sum in dq itself, the rounding error in a
// workspace plane), which keeps 16 bits of it.  The per-query words are then read from the
// global planes (the first pass writes them) instead of LDS, where the longer row leaves
// them no room.  Replaces _bwd_q and _bwd_kv of reference
// src/trifast/triton.py:274-383 and :143-263 in one pass.
#pragma once
#include <type_traits>
#include <utility>

#include "tri_args.hpp"
#include "tri_common.hpp"
#include "tri_tile.hpp"

// -DTRI_ROW_TIMING builds the kernel as a probe of itself (benchmark/microbench/row_timeline.py):
// wave 0 of every workgroup reads the 100 MHz counter at the marks below and the shader clock
// between the steps of the query-tile loop, and leaves the readings where the db argument
// points (a buffer of the caller's; db itself is not computed by this kernel).  Of a reading only the low
// word is kept, and what is known before the loop is written before it: with all of them held to the end the
// loop spilled scalar registers, and its steps took 60 clocks longer (n = 1024, d = 32: 7910 clocks per query tile, now 7380).
#ifdef TRI_ROW_TIMING
#define TRI_ROW_MARK(var)               \
  __builtin_amdgcn_sched_barrier(0);    \
  const uint32_t var = (uint32_t)__builtin_amdgcn_s_memrealtime(); \
  __builtin_amdgcn_sched_barrier(0)
#define TRI_ROW_TICK(k)                                      \
  do {                                                       \
    __builtin_amdgcn_sched_barrier(0);                       \
    const uint32_t now_ = (uint32_t)__builtin_amdgcn_s_memtime(); \
    tacc[k] += now_ - tprev;                                 \
    tprev = now_;                                            \
    __builtin_amdgcn_sched_barrier(0);                       \
  } while (0)
#else
#define TRI_ROW_MARK(var) (void)0
#define TRI_ROW_TICK(k) (void)0
#endif

namespace tri {

constexpr int kRowWaves = 4;

// ---- the MFMA order of one step of the kernel below ------------------------------------
enum RowOp { R_SOFF, R_SB, R_SQK, R_DOFF, R_DP, R_ACC, R_DQ };
struct RowSched {
  int n;             // MFMAs of the step
  int kind[48], idx[48];
  int dq_reads_at;   // the LDS reads for dq follow this MFMA
  int last_sqk;      // the last MFMA that reads the K rows of the next tile
  int v_reads_at;    // V operands kept in LDS are read after this MFMA
  int last_sb;       // the last MFMA that reads bias words (0 without any)
  int last_acc;      // the last dv/dk MFMA (-1 without any)
};
// Two dependent chains start a tile (scores: per-query offset and key mask, bias parts,
// q.k; dP: -delta, dO.v) and three finish the one before (dv/dk, dq).  Dependent MFMAs are
// kept apart: first the head of the score chain alternates with the dv/dk MFMAs, then dq,
// the q.k part and the dP chain take turns.  (delta_early: -delta stands behind the bias parts instead, three MFMAs in front of the
// first that adds to it.)
constexpr RowSched make_row_sched(bool has_prev, bool has_next, int nsb, int ds, int nacc, int ndq, bool delta_early) {
  RowSched s{};
  s.dq_reads_at = -1;
  s.last_sqk = -1;
  s.v_reads_at = -1;
  s.last_sb = 0;
  s.last_acc = -1;
  int lk[16] = {}, li[16] = {}, ns = 0;
  if (has_next) {
    lk[ns] = R_SOFF;
    li[ns++] = 0;
    for (int i = 0; i < nsb; ++i) {
      lk[ns] = R_SB;
      li[ns++] = i;
    }
    if (delta_early) {
      lk[ns] = R_DOFF;
      li[ns++] = 0;
    }
  }
  const int na = has_prev ? nacc : 0;
  int is = 0, ia = 0;
  if (is < ns) {
    if (lk[is] == R_SB) s.last_sb = s.n;
    s.kind[s.n] = lk[is];
    s.idx[s.n++] = li[is++];
  }
  while (is < ns || ia < na) {
    if (is < ns) {
      if (lk[is] == R_SB) s.last_sb = s.n;
      s.kind[s.n] = lk[is];
      s.idx[s.n++] = li[is++];
    }
    if (ia < na) {
      s.last_acc = s.n;
      s.kind[s.n] = R_ACC;
      s.idx[s.n++] = ia++;
    }
  }
  const int nq = has_prev ? ndq : 0, nk = has_next ? ds : 0, np = has_next ? 1 + ds : 0;
  int iq = 0, ik = 0, ip = delta_early ? 1 : 0, first_dq = -1;
  while (iq < nq || ik < nk || ip < np) {
    if (iq < nq) {
      if (first_dq < 0) first_dq = s.n;
      s.kind[s.n] = R_DQ;
      s.idx[s.n++] = iq++;
    }
    if (ik < nk) {
      s.last_sqk = s.n;
      s.kind[s.n] = R_SQK;
      s.idx[s.n++] = ik++;
    }
    if (ip < np) {
      if (ip == 1) s.v_reads_at = s.n >= 4 ? s.n - 4 : 0;
      s.kind[s.n] = ip == 0 ? R_DOFF : R_DP;
      s.idx[s.n++] = ip == 0 ? 0 : ip - 1;
      ++ip;
    }
  }
  if (first_dq >= 0) s.dq_reads_at = first_dq >= 3 ? first_dq - 3 : 0;
  return s;
}
template <bool HAS_PREV, bool HAS_NEXT, int NSB, int DS, int NACC, int NDQ, bool DELTA_EARLY = false>
struct RowSchedOf {
  static constexpr RowSched value = make_row_sched(HAS_PREV, HAS_NEXT, NSB, DS, NACC, NDQ, DELTA_EARLY);
};

// Key tiles per wave whose V operands live in LDS instead of registers: the longest rows
// leave the vector registers no room for all of them (the accumulators fill the other file).
// (one tile more in LDS when the row takes several passes: the words of the queries then leave
// LDS the room, and the dq carried between the passes takes registers)
constexpr int bwd_row_v_lds_tiles(int D, int KT, bool multi = false) { return KT * (D / 16) < 16 ? 0 : D <= 32 ? KT - (multi ? 2 : 3) : 1; }
// Two waves per SIMD (256 registers each, the accumulators among the ordinary ones), of two workgroups, where a wave holds two key
// tiles of rows of up to 64 bytes (the launches of short rows that tri_bwd_row_rule.hpp gives four waves, and the last pass over a long row).
constexpr bool bwd_row_two_waves(int D, int KT) { return D <= 32 && KT <= 2; }
// LDS bytes of the kernel below.  dq partials: two buffers (one barrier per query tile) of
// three quarters of a tile per wave (the quarter a wave sums itself waits in its dS tile)
constexpr int bwd_row_red_bytes(int D) { return kRowWaves * 3 * ((D + 31) / 32) * 1024; }
// Tiles of a stage of the query stream: Q, dO and, in rows of 128 bytes of up to 384 keys, o: delta is formed from it per query tile then, and
// the row does not start with a trip to memory for the o and dO of all its queries, a fifth of its time there (training steps, d = 64,
// us: h = 8, b = 2, n = 384 in fp16 2039 -> 1996; h = 8, n = 256 370 -> 351; h = 4, n = 330 419 -> 403, 384 491 -> 478).  In narrower
// rows, whose loops are longer, the work per query tile costs as much (d = 32, n = 600 994 -> 1006, 768 1812 both, 850 2767 -> 2764; d = 16, n = 700 1261 -> 1259).
constexpr int bwd_row_stage_tiles(int D, int KT, bool multi) { return D == 64 && KT <= 3 && !multi ? 3 : 2; }
constexpr int bwd_row_base_lds_bytes(int D, int es, int KT, bool multi) {  // (without the per-query words)
  const int rowb = D * es, keys = kRowWaves * KT * 32;
  return keys * rowb + 3 * (bwd_row_stage_tiles(D, KT, multi) * 32 * rowb) + kRowWaves * 2048 + 2 * bwd_row_red_bytes(D) +
         kRowWaves * bwd_row_v_lds_tiles(D, KT, multi) * (D / 16) * 1024;
}
// The per-query operand words of the row (two planes of 4 bytes per query) live in LDS where
// there is room and the row takes one pass; else they come from the global planes that the
// prologue writes, one query tile ahead.
constexpr bool bwd_row_words_in_lds(int D, int es, int KT, bool multi) {
  return !multi && bwd_row_base_lds_bytes(D, es, KT, multi) + 2 * kRowWaves * KT * 32 * 4 <= 160 * 1024;
}
constexpr int bwd_row_lds_bytes(int D, int es, int KT, bool multi = false) {
  return bwd_row_base_lds_bytes(D, es, KT, multi) + (bwd_row_words_in_lds(D, es, KT, multi) ? 2 * kRowWaves * KT * 32 * 4 : 0);
}

// XCDs that work on a head together: the smallest power of two whose heads side by side (8 / share of
// them) deal the launch's heads out evenly (8 heads or 16: one, 12: two, 6: four, 3: all eight).  With
// all eight wherever 8 heads do not divide, the backward of 12 heads took 1.464 instead of 1.434 ms at
// n = 512 and 9.38 instead of 9.22 at n = 1024 (d = 32), that of 6 heads 0.754 and 0.741 at n = 512.
constexpr int bwd_row_xcd_share(int bh) { return bh % 8 == 0 ? 1 : bh % 4 == 0 ? 2 : bh % 2 == 0 ? 4 : 8; }
// workgroups of a launch
constexpr int64_t bwd_row_blocks(int bh, int n) {
  const int share = bwd_row_xcd_share(bh), heads = 8 / share;
  return (int64_t)8 * ((bh + heads - 1) / heads) * ((n + share - 1) / share);
}

// The start of a launch.  Rows take equally long, so compute units that start together fetch the K, V, dO and o of a row together, compute
// while memory is idle, and store dk and dv together, row after row.  The workgroups of the first round (`per_cu` on each of 32 compute
// units of each XCD) start one after the other instead, over about the time memory needs for their rows (16 bytes per element at 5
// TB/s): 2 n d clocks.  That much later the last of them ends, so launches with few rounds take half of it, and rows that
// compute for long, which gain least; one round has nothing to gain.  A wave sleeps at most 2 n d clocks once per launch.
// This kernel or that of the short rows alone, us, without -> with, h = 4 where not said: d = 16: h = 8, n = 160 35.8 -> 34.8; n = 300 83.4 -> 81.2, 384
// 110.9 -> 108.3, 700 649 -> 643, 1024 1583 -> 1572; d = 32: h = 16, n = 128 39.2 -> 37.9; h = 3, n = 256 41.1 -> 40.0; n = 300 94.2 -> 89.0, 449
// 264 -> 259, 600 533 -> 515, 1024 1917 -> 1890; d = 64 (fp16): h = 8, n = 256 209 -> 195; n = 200 87.4 -> 82.4, 300 183 -> 174, 384 265 -> 252.
// In 118 launches of n = 90 to 1024 (46, 46 and 26 by head dim, half of them with padding) none lost more than its scatter.  Not
// halved: d = 64, h = 2, n = 256 58.1 -> 61.8 (halved 56.4); d = 32, n = 512 298 -> 301 (296); twice the time: d = 64, h = 8, n = 256 216 -> 213.
// Passes over longer rows: n = 1280 4211 -> 4258, so not there.
TRI_DEV void stagger_rows(int block, int per_cu, int bh, int n, int d) {
  const int slot = block >> 3, round = 256 * per_cu;
  const int64_t rows = (int64_t)bh * n;
  if (slot >= 32 * per_cu || rows <= round) return;
  const bool half = n > 10 * d || (per_cu == 1 && rows < 4 * round);
  for (int z = slot * (n * d >> 7) / (half ? 16 * per_cu : 8 * per_cu); z > 0; --z) __builtin_amdgcn_s_sleep(1);  // (64 clocks)
}

// LDS bytes of bwd_uniform_row: each wave's four 32-row tiles and 64 floats of delta, then the
// sums of the row (two D x D products, three vectors)
constexpr int bwd_uniform_lds_bytes(int D, int es, int NW) {
  const int tiles = NW * (4 * 32 * D * es + 256), sums = (2 * D * D + 3 * D) * 4;
  return tiles + sums;
}

// dq, dk and dv of a fully masked row (the padding of a padded batch), by one workgroup.  All logits of
// the row are equal, so P = 1 / n for every query and key, dS_jk = (dO_j . V_k - delta_j) / n, and
// the row's gradients are products with sums over the row instead of sums over score tiles:
//   dq_j = s / n (M1 dO_j - delta_j sK),   M1 = sum_k K_k V_k^T,  sK = sum_k K_k
//   dk_k = s / n (M2 V_k - sQ),            M2 = sum_j Q_j dO_j^T, sQ = sum_j delta_j Q_j
//   dv_k = sO / n,                          sO = sum_j dO_j
// The sums run on the matrix pipe over 32-row tiles (wave w takes tiles w, w + NW, ...; every
// wave's part is added in wave order), in fp32; M1 and M2 go into the second products as hi + lo parts
// (scaled for fp16, see there).
// What is left is the memory traffic of the row and its latency.  A training step over n = 512 with
// 397 valid positions (bf16, h = 4, d = 32), with the same rule in db and the rows dealt evenly:
// 605 -> 543 us.
// (Several passes over a long row: the first one does all of it.)
template <typename T, int D, int NW>
TRI_DEV void bwd_uniform_row(const BwdArgs& a, int bh, int i, unsigned char* smem, int wave, int lane) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using Tile = LdsTile<T, D>;
  constexpr int DS = D / 16, DM = (D + 31) / 32, NV = 32 * Tile::CPR / 64;  // 16-byte loads per lane and tile
  const int N = a.N, b = bh / a.H, h = bh % a.H, jl = lane & 31, g = lane >> 5;
  const T* const rows[4] = {reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h + i * a.sk.i,
                            reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h + i * a.sv.i,
                            reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h + i * a.sq.i,
                            reinterpret_cast<const T*>(a.dout) + b * a.sdo.b + h * a.sdo.h + i * a.sdo.i};
  const int64_t step[4] = {a.sk.j, a.sv.j, a.sq.j, a.sdo.j};
  const T* const orow = reinterpret_cast<const T*>(a.o) + ((int64_t)bh * N + i) * N * D;
  uint32_t* const dplane = a.delta + ((int64_t)bh * N + i) * N;
  uint32_t* const lplane = a.lse2 + ((int64_t)bh * N + i) * N;
  const uint32_t flat = split_word<T>(-__builtin_amdgcn_logf((float)N) * (kLn2 * a.sqrt_d));

  constexpr int TILE = 32 * Tile::ROWB;
  unsigned char* const mine = smem + wave * (4 * TILE + 256);
  float* const delta = reinterpret_cast<float*>(mine + 4 * TILE);  // [32]
  float* const m1 = reinterpret_cast<float*>(smem + NW * (4 * TILE + 256));  // [D][D]
  float* const m2 = m1 + D * D;
  float* const sk = m2 + D * D;  // sK, sQ, sO
  float* const sq = sk + D;
  float* const so = sq + D;

  OperandOffsets<T, D> ofs;
  ofs.init(jl, lane);
  f32x16 acc1[DM][DM], acc2[DM][DM], ak[DM], aq[DM], ao[DM];
#pragma unroll
  for (int x = 0; x < DM; ++x) {
#pragma unroll
    for (int y = 0; y < DM; ++y) acc1[x][y] = acc2[x][y] = zero16();
    ak[x] = aq[x] = ao[x] = zero16();
  }
  const frag ones = resident_ones<T>();
  // (the loads run a tile ahead, where the registers allow: nothing else on the compute unit hides
  // their latency)
  constexpr bool AHEAD = D <= 32;
  vec xn[4][NV], on[NV];
  auto load_tile = [&](int t) {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int r = (u * 64 + lane) / Tile::CPR, c = (u * 64 + lane) % Tile::CPR, j = min(32 * t + r, N - 1);
#pragma unroll
      for (int w = 0; w < 4; ++w) xn[w][u] = *reinterpret_cast<const vec*>(rows[w] + (int64_t)j * step[w] + 8 * c);
      on[u] = *reinterpret_cast<const vec*>(orow + (int64_t)j * D + 8 * c);
    }
  };
  if constexpr (AHEAD) load_tile(wave);
  for (int t = wave; t < a.nwords; t += NW) {
    if constexpr (!AHEAD) load_tile(t);
    vec x[4][NV], ov[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
#pragma unroll
      for (int w = 0; w < 4; ++w) x[w][u] = xn[w][u];
      ov[u] = on[u];
    }
    if constexpr (AHEAD) load_tile(t + NW);
    // rows past the end count as zeros
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int r = (u * 64 + lane) / Tile::CPR, c = (u * 64 + lane) % Tile::CPR, j = 32 * t + r;
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) d += (float)ov[u][e] * (float)x[3][u][e];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        vec y = x[w][u];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = j < N ? y[e] : (T)0.f;
        *reinterpret_cast<vec*>(mine + w * TILE + Tile::off(r, 16 * c)) = y;
      }
      // (the lanes of a row are neighbours)
#pragma unroll
      for (int m = 1; m < Tile::CPR; m *= 2) d += __shfl_xor(d, m);
      if (c == 0) {
        delta[r] = j < N ? d : 0.f;
        if (j < N) {
          dplane[j] = split_word<T>(-d);
          lplane[j] = flat;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      frag kt[DM], vt[DM], qt[DM], dt[DM], dh, dl;
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
        kt[mt] = ofs.transposed(mine, s2, mt);
        vt[mt] = ofs.transposed(mine + TILE, s2, mt);
        qt[mt] = ofs.transposed(mine + 2 * TILE, s2, mt);
        dt[mt] = ofs.transposed(mine + 3 * TILE, s2, mt);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = delta[cidx(8 * s2 + e, g)];
        dh[e] = (T)d;
        dl[e] = (T)(d - (float)dh[e]);
      }
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
#pragma unroll
        for (int nt = 0; nt < DM; ++nt) {
          acc1[mt][nt] = E::mfma(kt[mt], vt[nt], acc1[mt][nt]);
          acc2[mt][nt] = E::mfma(qt[mt], dt[nt], acc2[mt][nt]);
        }
        ak[mt] = E::mfma(kt[mt], ones, ak[mt]);
        ao[mt] = E::mfma(dt[mt], ones, ao[mt]);
        aq[mt] = E::mfma(qt[mt], dh, aq[mt]);
        aq[mt] = E::mfma(qt[mt], dl, aq[mt]);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  // The waves' parts, in wave order.  A wave's turn is one run of reads, adds and writes without a branch, at immediates from two bases
  // that are made in the turn.  (One address per element, made before the turns, took every register of the kernel: at d = 64 they came
  // back from scratch one by one, and the loop over the query tiles of the other rows had a reload of its own.  This kernel alone, h = 4, d = 64,
  // bf16, us: n = 256 with 60 valid 399 -> 156, 199 valid 185 -> 118, n = 384 with 300 valid 388 -> 262; without padding n = 256, h = 8 197 -> 194, n = 330
  // 219 -> 215, b = 2, h = 8, n = 384 in fp16 1004 -> 978.)
  for (int w = 0; w < NW; ++w) {
    if (wave == w) {
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int row0 = 4 * (ln >> 5), col0 = ln & 31;
      float *const p1 = m1 + row0 * D + col0, *const pv = sk + row0;
      auto add = [&](auto first_tag, auto vectors_tag) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_tag)::value, VECTORS = decltype(vectors_tag)::value;
        auto sum = [](float& at, float x) { at = x + (FIRST ? 0.f : at); };
#pragma unroll
        for (int mt = 0; mt < DM; ++mt)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int row = 32 * mt + crow(v, 0);  // (the other half of the lanes: four rows on)
            if (row + 4 >= D) continue;
            if constexpr (VECTORS) {
              sum(pv[row], ak[mt][v]);
              sum(pv[D + row], aq[mt][v]);
              sum(pv[2 * D + row], ao[mt][v]);
            } else {
#pragma unroll
              for (int nt = 0; nt < DM; ++nt) {
                sum(p1[row * D + 32 * nt], acc1[mt][nt][v]);
                sum(p1[D * D + row * D + 32 * nt], acc2[mt][nt][v]);
              }
            }
          }
      };
      auto turn = [&](auto first_tag) __attribute__((always_inline)) {
        if (D % 32 == 0 || col0 < D) add(first_tag, std::false_type{});
        if (col0 == 0) add(first_tag, std::true_type{});
      };
      if (w == 0) turn(std::true_type{});
      else turn(std::false_type{});
    }
    __syncthreads();
  }
  // fp16 ends at 65504, which sums over a row of coherent numbers pass (768 keys with K = V = 10 in a
  // channel give 76800): M1 and M2 go in times a power of two that brings their largest entry to
  // 2^13 .. 2^14, which costs no bits, and the factor comes off with the store.
  int up1 = 0, up2 = 0;
  if constexpr (std::is_same_v<T, _Float16>) {
    float x1 = 0.f, x2 = 0.f;
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      const int row = min(32 * mt + jl, D - 1);
#pragma unroll
      for (int e = 0; e < D / 2; ++e) {
        x1 = fmaxf(x1, __builtin_fabsf(m1[row * D + D / 2 * g + e]));
        x2 = fmaxf(x2, __builtin_fabsf(m2[row * D + D / 2 * g + e]));
      }
    }
#pragma unroll
    for (int m = 1; m < 64; m *= 2) {
      x1 = fmaxf(x1, __shfl_xor(x1, m));
      x2 = fmaxf(x2, __shfl_xor(x2, m));
    }
    up1 = 14 - __builtin_amdgcn_frexp_expf(x1);
    up2 = 14 - __builtin_amdgcn_frexp_expf(x2);
  }
  // second products: row jl of M1, M2 as hi + lo parts; the vectors at this lane's rows of the result
  frag h1[DM][DS], l1[DM][DS], h2[DM][DS], l2[DM][DS];
  f32x16 vk[DM], vq[DM], vo[DM];
#pragma unroll
  for (int mt = 0; mt < DM; ++mt) {
    const int row = min(32 * mt + jl, D - 1);
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x1 = ldexpf(m1[row * D + 16 * s + 8 * g + e], up1), x2 = ldexpf(m2[row * D + 16 * s + 8 * g + e], up2);
        h1[mt][s][e] = (T)x1;
        l1[mt][s][e] = (T)(x1 - (float)h1[mt][s][e]);
        h2[mt][s][e] = (T)x2;
        l2[mt][s][e] = (T)(x2 - (float)h2[mt][s][e]);
      }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = min(32 * mt + crow(v, g), D - 1);
      vk[mt][v] = ldexpf(sk[r], up1);
      vq[mt][v] = ldexpf(-sq[r], up2);
      vo[mt][v] = so[r];
    }
  }
  const float inv = 1.0f / (float)N, mulq = ldexpf(a.scale * inv, -up1), mulk = ldexpf(a.scale * inv, -up2);
  T* const dqrow = reinterpret_cast<T*>(a.dq) + b * a.sdq.b + h * a.sdq.h + i * a.sdq.i;
  T* const dkrow = reinterpret_cast<T*>(a.dk) + b * a.sdk.b + h * a.sdk.h + i * a.sdk.i;
  T* const dvrow = reinterpret_cast<T*>(a.dv) + b * a.sdv.b + h * a.sdv.h + i * a.sdv.i;
  frag dn[DS], vn[DS], pn[DS];
  auto load_ops = [&](int t) {
    const int j = min(32 * t + jl, N - 1);
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const int c = 16 * s + 8 * g;
      dn[s] = E::load(rows[3] + (int64_t)j * step[3] + c);
      vn[s] = E::load(rows[1] + (int64_t)j * step[1] + c);
      pn[s] = E::load(orow + (int64_t)j * D + c);
    }
  };
  if constexpr (AHEAD) load_ops(wave);
  for (int t = wave; t < a.nwords; t += NW) {
    if constexpr (!AHEAD) load_ops(t);
    const int j = 32 * t + jl;
    frag df[DS], vf[DS];
    float d = 0.f;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      df[s] = dn[s];
      vf[s] = vn[s];
#pragma unroll
      for (int e = 0; e < 8; ++e) d += (float)pn[s][e] * (float)dn[s][e];
    }
    d = half_sum(d);
    if constexpr (AHEAD) load_ops(t + NW);
    f32x16 q[DM], k[DM];
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
#pragma unroll
      for (int v = 0; v < 16; ++v) q[mt][v] = -d * vk[mt][v];
      k[mt] = vq[mt];
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        q[mt] = E::mfma(l1[mt][s], df[s], q[mt]);
        k[mt] = E::mfma(l2[mt][s], vf[s], k[mt]);
        q[mt] = E::mfma(h1[mt][s], df[s], q[mt]);
        k[mt] = E::mfma(h2[mt][s], vf[s], k[mt]);
      }
    }
    store_rows_wide<T, D, DM>(dqrow + (int64_t)j * a.sdq.j, q, mulq, g, j < N);
    store_rows_wide<T, D, DM>(dkrow + (int64_t)j * a.sdk.j, k, mulk, g, j < N);
    store_rows_wide<T, D, DM>(dvrow + (int64_t)j * a.sdv.j, vo, inv, g, j < N);
  }
}

// delta = rowsum(o * do) of up to ROWS queries by NW waves.  A load takes whole rows side by side, 16 bytes of one per lane, so that the CPR
// lanes of a row each hold a part of its sum; they trade the parts of CPR rows in such a way that each ends with the sum of one of them.
// (A row per lane, 16 bytes at a time, touches 64 rows with every load.  Measured at d = 64, which forms delta per query tile now: h = 8, n = 256
// 228.4 -> 216.8 us; d = 32 within 0.6 %.)
template <typename T, int D, int ROWS, int NW>
struct DeltaRows {
  using E = Elem<T>;
  static constexpr int CPR = D / 8, RPL = NW * 64 / CPR;  // lanes per row; rows per load of the workgroup
  static constexpr int NLD = (ROWS + RPL - 1) / RPL, NB = (NLD + CPR - 1) / CPR;
  typename E::vec ov[NLD], dv[NLD];
  float lv[NB];
  // the query whose sum a lane has of batch x
  static TRI_DEV int query(int x, int tid) { return (x * CPR + tid % CPR) * RPL + tid / CPR; }
  TRI_DEV void load(const T* orow, const T* dorow, uint32_t do_step, const float* lse, int n, int tid) {
#pragma unroll
    for (int x = 0; x < NLD; ++x) {
      const int j = min(x * RPL + tid / CPR, n - 1);
      ov[x] = *reinterpret_cast<const typename E::vec*>(orow + (int64_t)j * D + 8 * (tid % CPR));
      dv[x] = *reinterpret_cast<const typename E::vec*>(dorow + (int64_t)j * do_step + 8 * (tid % CPR));
    }
#pragma unroll
    for (int x = 0; x < NB; ++x) lv[x] = lse[min(query(x, tid), n - 1)];
  }
  // words(query, delta, lse) for every query
  template <typename Words>
  TRI_DEV void finish(int tid, Words words) {
    static_assert(CPR <= 4, "the lanes of a row trade their parts within a quad");
    typedef T pair __attribute__((ext_vector_type(2)));
    const int c = tid % CPR;
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      float s[CPR];
#pragma unroll
      for (int y = 0; y < CPR; ++y) {
        s[y] = 0.f;
        const int ld = x * CPR + y;
        if (ld < NLD) {
#pragma unroll
          for (int e = 0; e < 8; e += 2) s[y] = pair_dot(pair{ov[ld][e], ov[ld][e + 1]}, pair{dv[ld][e], dv[ld][e + 1]}, s[y]);
        }
      }
#pragma unroll
      for (int m = CPR / 2; m > 0; m /= 2)
#pragma unroll
        for (int y = 0; y < m; ++y) {
          const float keep = c & m ? s[y + m] : s[y], give = c & m ? s[y] : s[y + m];
          s[y] = keep + (m == 2 ? dpp_move<0x4e>(give) : dpp_move<0xb1>(give));
        }
      if ((x * CPR + c) * RPL < ROWS) words(query(x, tid), s[0], lv[x]);
    }
  }
};

template <typename T, int D, int KT, bool MULTI = false>
__global__ __launch_bounds__(kRowWaves * 64, bwd_row_two_waves(D, KT) ? 2 : 1) void tri_bwd_row_kernel(const BwdArgs a) {
  // (two waves per SIMD: the accumulators are ordinary registers)
  constexpr bool TWO = bwd_row_two_waves(D, KT);
  static_assert(sizeof(T) == 2, "16-bit inputs only (the transposing LDS reads)");
  using E = Elem<T>;
  using frag = typename E::frag;
  using Tile = LdsTile<T, D>;
  using DsTile = LdsTile<T, 32, 2>;  // the wave's dS tile: 16-byte stores of whole rows, transposed reads
  constexpr int NW = kRowWaves;
  constexpr int KP = E::KP;
  constexpr int DS = D / (2 * KP);
  constexpr int DM = (D + 31) / 32;
  constexpr int PS = 2;
  constexpr int ROWB = Tile::ROWB;
  constexpr int KEYS = NW * KT * 32;         // keys (and queries) the workgroup can hold
  constexpr bool WORDS_LDS = bwd_row_words_in_lds(D, (int)sizeof(T), KT, MULTI);  // per-query words of the row in LDS (else from the global planes)
  constexpr int NT = bwd_row_stage_tiles(D, KT, MULTI);
  constexpr bool O_STAGE = NT == 3;
  constexpr int STAGE = NT * 32 * ROWB;       // Q tile | dO tile (| o tile)
  constexpr int OFF_K = 0;
  constexpr int OFF_ST = KEYS * ROWB;
  constexpr int OFF_DS = OFF_ST + 3 * STAGE;  // three stages: in use, ready, in flight
  constexpr int OFF_RED = OFF_DS + NW * 2048;
  constexpr int OFF_NL = OFF_RED + 2 * bwd_row_red_bytes(D);
  constexpr int PLANE = WORDS_LDS ? KEYS * 4 : 0;  // per-query words of the row
  constexpr int OFF_ND = OFF_NL + PLANE;
  constexpr int G2W = (NT * 32 * (ROWB / 16) / 64 + NW - 1) / NW;  // global->LDS loads per wave and stage
  constexpr int VL = bwd_row_v_lds_tiles(D, KT, MULTI);  // this wave's last VL key tiles keep V in LDS
  constexpr int VR = KT - VL;
  constexpr int OFF_V = OFF_ND + PLANE;
  static_assert(OFF_V + NW * VL * DS * 1024 == bwd_row_lds_bytes(D, (int)sizeof(T), KT, MULTI), "the launcher sizes LDS with bwd_row_lds_bytes");
  static_assert(bwd_row_lds_bytes(D, (int)sizeof(T), KT, MULTI) <= 160 * 1024, "LDS of one compute unit");
  static_assert(bwd_uniform_lds_bytes(D, (int)sizeof(T), NW) <= bwd_row_lds_bytes(D, (int)sizeof(T), KT, MULTI), "LDS of a fully masked row");
  static_assert((KT - 1) * NW * 32 * ROWB + 32 * ROWB <= 65536, "key tile offsets are LDS immediates");
  extern __shared__ __attribute__((aligned(16))) unsigned char tri_smem[];

  TRI_ROW_MARK(t_entry);
  if constexpr (!MULTI) stagger_rows(blockIdx.x, bwd_row_two_waves(D, KT) ? 2 : 1, a.BH, a.N, D);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the lane id for addresses inside the loop: opaque wherever it is used, so that nothing derived from it is hoisted out of the loop
  // and kept in registers (it would be spilled, and a reload from scratch waits for every load in flight)
  int lane_o = lane;
  const int kl = lane & 31, g = lane >> 5;
  const int N = a.N;
  const int NJ = a.nwords;  // 32-tiles of the row (queries and keys)
  // this pass: key tiles KT0 .. KT0 + 4 KT - 1 of the row (tiles past the row's end are empty)
  const int KT0 = MULTI ? a.key_tile0 : 0;
  const bool first_pass = !MULTI || (a.pass_flags & 1) == 0, last_pass = !MULTI || (a.pass_flags & 2) == 0;

  // Workgroups go to the 8 XCDs round-robin by linear id.  An XCD works on one head at a time, so
  // that the head's packed bias stays in its L2, and takes every `share`-th row of it, so that the
  // short work of fully masked rows (the padding at the end of every head) is spread evenly: with
  // a run of rows per XCD, half of the XCDs had none of it at n = 512, h = 4.
  const int share = bwd_row_xcd_share(a.BH), per_head = (N + share - 1) / share;
  const int L = blockIdx.x, slot = L >> 3;
  const int bh = slot / per_head * (8 / share) + (L & 7) / share, i = slot % per_head * share + (L & 7) % share;
  if (bh >= a.BH || i >= N) return;
  const int b = bh / a.H, h = bh % a.H;

  const T* qrow = reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h + i * a.sq.i;
  const T* krow = reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h + i * a.sk.i;
  const T* vrow = reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h + i * a.sv.i;
  const T* dorow = reinterpret_cast<const T*>(a.dout) + b * a.sdo.b + h * a.sdo.h + i * a.sdo.i;
  const T* const orow = reinterpret_cast<const T*>(a.o) + ((int64_t)bh * N + i) * N * D;
  const T* pack_bh = reinterpret_cast<const T*>(a.packq) + (int64_t)bh * a.NP * a.NP * 1024;

  unsigned char* const lds_k = tri_smem + OFF_K;
  uint32_t* const nl = reinterpret_cast<uint32_t*>(tri_smem + OFF_NL);  // operand words, see split_word
  uint32_t* const nd = reinterpret_cast<uint32_t*>(tri_smem + OFF_ND);

  // ---- prologue -----------------------------------------------------------------
  // K row -> LDS (rows past the end repeat the last key; their keep bits are clear)
  Tile::template fill<KEYS, NW>(lds_k, [&](int r) { return krow + (int64_t)min(32 * KT0 + r, N - 1) * a.sk.j; }, wave, lane);
  // query tiles 0 (and 1) -> the two stage buffers
  // (per-lane source pointers for query tile 0, computed once; a tile inside the row adds
  // one uniform offset, the ragged last one clamps the query index)
  // The loads are written as asm: the compiler makes every LDS read that follows a
  // global->LDS load it knows of wait for that load (the read might be of the bytes in
  // flight), which would turn the prefetch of the next query tile into a stall at the next
  // operand read.  Here the stage in flight is not read before the wait and barrier that end
  // the query tile.  The compiler's own waits stay correct: loads return in issue order, and
  // a load it does not know of only makes the counter it waits on larger.  (The source
  // addresses are rebuilt from the lane id every time: kept in registers from one query tile
  // to the next they would be spilled, and a reload from scratch waits for every load in flight.)
  // (No branch: what stands in front of one is sunk behind it by the compiler, out of the schedule of the loop below.)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(TRI_L3 unsigned char*)tri_smem;
  // the stage is two or three tiles (Q rows, dO rows, o rows) of LT wave loads of 1 KiB, dealt to the waves in turn: GX loads for each, or, where that
  // does not come out even (head dim 16), some without a share; fill[] are the first rows of the next stage to request, per load
  constexpr int LT = 32 * Tile::CPR / 64, GX = (NT * LT + NW - 1) / NW;
  const T* fill[GX];
  int64_t fill_step[GX];
  uint32_t fill_row[GX];  // bytes between rows (below 2^24: a limit of the entry points)
#pragma unroll
  for (int x = 0; x < GX; ++x) {
    const int tile = (x * NW + wave) / LT;
    fill[x] = tile == 0 ? qrow : O_STAGE && tile == 2 ? orow : dorow;
    const int64_t stride = tile == 0 ? a.sq.j : O_STAGE && tile == 2 ? D : a.sdo.j;
    fill_step[x] = 32 * stride;
    fill_row[x] = (uint32_t)stride * (uint32_t)sizeof(T);
  }
  int fill_rows = N - 1;  // the last row of the pair row, counted from them
  auto issue_stage = [&](int buf) {
    asm volatile("" : "+v"(lane_o));
    const uint32_t ln = (uint32_t)lane_o;
#pragma unroll
    for (int x = 0; x < GX; ++x) {
      const int gi = x * NW + wave;
      const uint32_t r = (uint32_t)(gi % LT * (64 / Tile::CPR)) + ln / Tile::CPR, cc = (ln % Tile::CPR) ^ (uint32_t)Tile::swz((int)r);
      // a 64-bit base per tile (scalar registers) and a 32-bit byte offset per lane; rows past
      // the end of the pair row (last tile only) read the last row again
      const uint32_t voff = __umul24((uint32_t)min((int)r, fill_rows), fill_row[x]) + 16 * cc;
      const T* base = fill[x];
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(OFF_ST + buf * STAGE + gi * 1024));
      // (waves without a share load with no lane; their counted wait is for nothing of theirs, the barrier behind it stands for the others')
      if constexpr (NT * LT % NW != 0) {
        const int mine = __builtin_amdgcn_readfirstlane(gi < NT * LT ? -1 : 0);
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" : : "s"(dst), "v"(voff), "s"(base), "s"(mine) : "memory", "m0");
      } else {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(voff), "s"(base) : "memory", "m0");
      }
    }
    // (behind the last query tile the last one is requested again, into a stage nobody reads any more)
    const int more = __builtin_amdgcn_readfirstlane(fill_rows >= 32 ? -1 : 0);
#pragma unroll
    for (int x = 0; x < GX; ++x) fill[x] += fill_step[x] & (int64_t)more;
    fill_rows -= 32 & more;
  };
  issue_stage(0);
  issue_stage(1);

  // (a fully masked row goes its own way; these words come through the scalar cache, all in flight together and apart from the
  // vector loads around them)
  if (uniform_word(a.rowflag, b * N + i) != 0) {
    wait_dma();  // (the loads on their way into the LDS it uses)
    __syncthreads();
    if (first_pass) bwd_uniform_row<T, D, NW>(a, bh, i, tri_smem, wave, lane);
    return;
  }
  // keep words of this wave's key tiles (bit k set = key k of the tile is attended)
  uint32_t kw[KT];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int kt = KT0 + NW * t + wave;
    kw[t] = uniform_word(a.keep, (b * N + i) * a.nwords + min(kt, NJ - 1));
  }
#pragma unroll
  for (int t = 0; t < KT; ++t)
    if (KT0 + NW * t + wave >= NJ) kw[t] = 0u;
  TRI_ROW_MARK(t_p1);

  // V rows of this lane's keys as B operands: in registers for the wave's first VR key
  // tiles, in a private piece of LDS (operand by operand, 16 bytes per lane) for the rest
  frag vf[VR > 0 ? VR : 1][DS];
  frag* const v_lds = reinterpret_cast<frag*>(tri_smem + OFF_V + wave * VL * DS * 1024) + lane;
  // (every load of the prologue is issued before the first one is used: the V rows here, then
  // the row's o and do where delta comes from them (queries past the end read the last one again): one trip to
  // memory for all of them, while the K row is on its way to LDS)
  frag vx[KT][DS];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int key = min(32 * (KT0 + NW * t + wave) + kl, N - 1);
#pragma unroll
    for (int s = 0; s < DS; ++s) vx[t][s] = *reinterpret_cast<const frag*>(vrow + (int64_t)key * a.sv.j + 2 * KP * s + KP * g);
  }
  const float* const lserow = a.lse + ((int64_t)bh * N + i) * N;
  static_assert(WORDS_LDS || !O_STAGE, "the words of a query are kept in LDS until the end of the row");
  DeltaRows<T, D, WORDS_LDS ? KEYS : 1, NW> dr;
  constexpr int LSE_N = O_STAGE ? (KEYS + NW * 64 - 1) / (NW * 64) : 1;
  float lse_x[LSE_N];
  if constexpr (O_STAGE) {
#pragma unroll
    for (int x = 0; x < LSE_N; ++x) lse_x[x] = lserow[min(x * NW * 64 + tid, N - 1)];
  } else if constexpr (WORDS_LDS) {
    dr.load(orow, dorow, (uint32_t)a.sdo.j, lserow, N, tid);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      if (t < VR) vf[t][s] = vx[t][s];
      else v_lds[((t - VR) * DS + s) * 64] = vx[t][s];
    }

  TRI_ROW_MARK(t_p2);
  // per-query terms of the row: -delta and -lse*sqrt(d) as MFMA operand words, kept in LDS for this kernel and written for the db kernel
  uint32_t* const dplane = a.delta + ((int64_t)bh * N + i) * N;
  uint32_t* const lplane = a.lse2 + ((int64_t)bh * N + i) * N;
  if (first_pass) {
    auto query_words = [&](int j, float dsum, float lse_j) {
      float nlv = E::kMaskElem, ndv = 0.f;  // queries past the end: P = dS = 0
      if (j < N) {
        ndv = -dsum;
        nlv = -lse_j * a.sqrt_d;
      }
      const uint32_t lw = split_word<T>(nlv), dw = split_word<T>(ndv);
      if (j < N) {
        dplane[j] = dw;
        lplane[j] = lw;
      }
      if constexpr (WORDS_LDS) {
        nl[j] = lw;
        nd[j] = dw;
      }
    };
    if constexpr (O_STAGE) {
#pragma unroll
      for (int x = 0; x < LSE_N; ++x) {
        const int j = x * NW * 64 + tid;
        if (KEYS % (NW * 64) != 0 && j >= KEYS) continue;
        const uint32_t lw = split_word<T>(j < N ? -lse_x[x] * a.sqrt_d : E::kMaskElem);  // queries past the end: P = dS = 0
        if (j < N) lplane[j] = lw;
        nl[j] = lw;
      }
    } else if constexpr (WORDS_LDS) {
      dr.finish(tid, query_words);
    } else {
      // (rows of 1024 keys are as fast this way, and with the loads above in a loop the compiler (ROCm 7.2.0) ends with a segmentation fault
      // in its pass over accumulator copies at d = 64 and four key tiles in bf16)
      for (int j = tid; j < N; j += NW * 64) {
        float dsum = 0.f;
#pragma unroll
        for (int x = 0; x < D / 8; ++x) {
          const typename E::vec ov = *reinterpret_cast<const typename E::vec*>(orow + (int64_t)j * D + 8 * x);
          const typename E::vec dv = *reinterpret_cast<const typename E::vec*>(dorow + (int64_t)j * a.sdo.j + 8 * x);
#pragma unroll
          for (int e = 0; e < 8; ++e) dsum += (float)ov[e] * (float)dv[e];
        }
        query_words(j, dsum, lserow[j]);
      }
    }
  }
  TRI_ROW_MARK(t_p3);
  // (words not in LDS: they come back from the global planes, which the first pass has just
  // written: its stores are waited for, with the loads, before the barrier below; the loads
  // are made at device scope so that no stale copy in the first-level cache can serve them)
  auto fetch_words = [&](int jt, uint32_t& lw, uint32_t& dw) {
    const int j = 32 * min(jt, NJ - 1) + perm32(kl);
    lw = split_word<T>(E::kMaskElem);  // queries past the end: P = dS = 0
    dw = split_word<T>(0.f);
    if (j < N) {
      lw = __hip_atomic_load(lplane + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      dw = __hip_atomic_load(dplane + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };

  // lane-constant LDS offsets.  Q, dO tiles: natural A operands (tile row m stands for
  // query perm32(m)) and transposed A operands; K tiles: natural B operand of this lane's
  // key and transposed A operand; the wave's dS tile: write offsets and transposed reads.
  OperandOffsets<T, D> ofq, ofk;
  ofq.init(perm32(kl), lane);
  ofk.init(kl, lane);
  ofk.shift(wave * 32 * ROWB);  // key tile t of this wave starts (4 t + wave) * 32 rows into K
  OperandOffsets<T, 32, 2> ofd;
  ofd.init(0, lane);
  // (one tile: the wave reads dS of a key tile back before it writes the next one)
  unsigned char* const ds_tile = tri_smem + OFF_DS + wave * 2048;
  const int ds_w0 = DsTile::off(kl, 16 * g), ds_w1 = DsTile::off(kl, 32 + 16 * g);


  // packed bias tiles of this lane: tile (jt, kt) is 2 x 16 bytes per lane
  typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
  // (as A operand: operand row m stands for query perm32(m), like the Q and dO operands)
  // (a tile's address is a wave-uniform base, computed on the scalar unit, plus this lane's
  // constant 32-bit byte offset: no vector arithmetic per tile)
  uint32_t bias_lane = (uint32_t)((perm32(kl) + 32 * g) * 8 * sizeof(T));
  auto bias_load = [&](int jt, int t, u32x4v* dst) {
    const int kt = min(KT0 + NW * t + wave, a.NP - 1);
    const char* tile = reinterpret_cast<const char*>(pack_bh + ((int64_t)min(jt, a.NP - 1) * a.NP + kt) * 1024);
    asm volatile("" : "+v"(bias_lane));  // (opaque here: the sum of the lane offset and the head's base is not hoisted as a 64-bit vector)
    dst[0] = *reinterpret_cast<const u32x4v*>(tile + (uint64_t)bias_lane);
    dst[1] = *reinterpret_cast<const u32x4v*>(tile + (uint64_t)bias_lane + 512 * sizeof(T));
  };
  const float c = a.c;

  // sqrt(d) * bias through the matrix pipe.  Half r of a packed bias tile gives a lane
  // (query, g) the keys 16 r + 8 g + 0..7 as its contraction slots; the constant B operand
  // of half r holds sqrt(d) in the slot that stands for the lane's own key (column) and
  // zero elsewhere.  sqrt(32) is not a 16-bit number: it goes in as hi + lo, one MFMA each.
  constexpr int NPART = D == 32 ? 2 : 1;
  constexpr int NSB = 2 * NPART;
  frag bsel[2][NPART];
  {
    const T hi = (T)a.sqrt_d;
    const T part[2] = {hi, (T)(a.sqrt_d - (float)hi)};
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int pp = 0; pp < NPART; ++pp) {
        const int e = kl - 16 * r - 8 * g;
        const uint32_t bits = (uint32_t)__builtin_bit_cast(uint16_t, part[pp]) << (16 * (e & 1));
        u32x4v w;
#pragma unroll
        for (int x = 0; x < 4; ++x) w[x] = (e >= 0 && e < 8 && (e >> 1) == x) ? bits : 0u;
        asm volatile("" : "+v"(w));  // resident: not rebuilt from the lane id at every use
        bsel[r][pp] = __builtin_bit_cast(frag, w);
      }
  }
  // rank-1 operands: per-query words (A side) and the ones / key-mask operand (B side)
  typename OffsetMask<T>::Queries s_off;
  s_off.init(0u, g);
  Rank1<T> d_off;
  d_off.init();
  typename OffsetMask<T>::Keys keys_op;
  keys_op.init(kl, g);

  // dq partial tiles of the four waves.  Wave q sums quarter q of every lane's values: head-dim
  // elements 32 mt + 8 q + 4 g + 0..3 of query 32 jt + kl, 8 bytes per lane (the four waves'
  // stores complete the rows).  The other three waves leave their parts of that quarter in
  // [buffer][summing wave q][slot][mt][lane] x 16 bytes, the slot being the writer's rank among
  // those three; the wave's own part waits in its dS tile, which is idle between the last key
  // tile of a query tile and the first of the next.  A wave adds its own part first, then the
  // others' in wave order (deterministic, no atomics).
  // The store is written as asm, as one instruction with its base in scalar registers.
  // Addresses are rebuilt from the lane id at every use: kept in registers across the
  // key-tile steps they would be spilled, and a reload from scratch waits for every load
  // in flight.
  static_assert(DM * 1024 <= 2048, "the own quarter of a dq tile fits the wave's dS tile");
  constexpr int RED_BYTES = bwd_row_red_bytes(D);
  // byte offsets in LDS, all wave-uniform and the same for every query tile: where this wave
  // leaves quarter q of its tile (per buffer), where its own quarter waits, and where the other
  // waves leave their parts of its quarter (three slots side by side)
  int part_wr[2][kRowWaves];
#pragma unroll
  for (int q = 0; q < kRowWaves; ++q)
#pragma unroll
    for (int bf = 0; bf < 2; ++bf)
      part_wr[bf][q] = q == wave ? OFF_DS + wave * 2048 : OFF_RED + bf * RED_BYTES + (q * 3 + (wave < q ? wave : wave - 1)) * DM * 1024;
  const int part_own = OFF_DS + wave * 2048, part_rd = OFF_RED + wave * 3 * DM * 1024;
  T* dqrow = reinterpret_cast<T*>(a.dq) + b * a.sdq.b + h * a.sdq.h + i * a.sdq.i;
  T* lorow = reinterpret_cast<T*>(a.dq_lo) + ((int64_t)bh * N + i) * N * D;  // (several passes only)
  typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
  // what the passes before this one left for this lane's elements of query tile jt: fetched at
  // the start of the query tile, added when its dq is summed
  struct DqCarry {
    typename E::vec4 hi[DM], lo[DM];
  };
  auto fetch_carry = [&](int jt, DqCarry& cy) {
    asm volatile("" : "+v"(lane_o));
    const int ln = lane_o;
    const int j = min(32 * jt + (ln & 31), N - 1);
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      const int d0 = min(32 * mt + 8 * wave + 4 * (ln >> 5), D - 4);
      cy.hi[mt] = *reinterpret_cast<const typename E::vec4*>(dqrow + (int64_t)j * a.sdq.j + d0);
      cy.lo[mt] = *reinterpret_cast<const typename E::vec4*>(lorow + (int64_t)j * D + d0);
    }
  };
  // this wave's dq tile of a query tile -> LDS, a quarter for each wave that sums one
  auto store_partials = [&](int buf, const f32x16 (&acc)[DM]) {
    asm volatile("" : "+v"(lane_o));
    const int ln = lane_o;
#pragma unroll
    for (int q = 0; q < kRowWaves; ++q)
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = acc[mt][4 * q + e];
        *(reinterpret_cast<f32x4*>(tri_smem + (buf ? part_wr[1][q] : part_wr[0][q]) + mt * 1024) + ln) = x;
      }
  };
  // the four parts of this wave's quarter: its own, then the other waves' in wave order
  struct DqParts {
    f32x4 v[4][DM];
  };
  auto load_partials = [&](int buf, DqParts& pp) {
    asm volatile("" : "+v"(lane_o));
    const int ln = lane_o;
    const f32x4* own = reinterpret_cast<const f32x4*>(tri_smem + part_own) + ln;
    const f32x4* others = reinterpret_cast<const f32x4*>(tri_smem + part_rd + (buf ? RED_BYTES : 0)) + ln;
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      pp.v[0][mt] = own[mt * 64];
#pragma unroll
      for (int k = 0; k < 3; ++k) pp.v[1 + k][mt] = others[(k * DM + mt) * 64];
    }
  };
  // Their sum (the own part first, then the others in wave order), scaled, as the stores will write it: dq, what rounding it to the
  // element type lost (between the passes over a long row), this lane's byte offset from
  // the start of the query tile in dq, and which lanes store.  The sum is cut into pieces of a
  // few instructions each (piece 0 .. kSumPieces-1, in this order): they run one per MFMA of a
  // step that has no vector work of its own, in the shadow of the matrix pipe.
  struct DqOut {
    f32x4 sum[DM];
    u32x2v hi[DM], lo[DM];
    uint32_t off;
    uint64_t live;  // the lanes that store
  };
  constexpr int kSumPieces = 6;
  auto sum_dq_piece = [&](int piece, int jt, DqParts& pp, const DqCarry& cy, DqOut& o) {
    if (piece == 0) {
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) o.sum[mt] = pp.v[0][mt] + pp.v[1][mt];
    } else if (piece == 1 || piece == 2) {
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) o.sum[mt] += pp.v[piece + 1][mt];
    } else if (piece == 3) {
#pragma unroll
      for (int mt = 0; mt < DM; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e) o.sum[mt][e] *= a.scale;
      if constexpr (MULTI) {
#pragma unroll
        for (int mt = 0; mt < DM; ++mt)
#pragma unroll
          for (int e = 0; e < 4; ++e) o.sum[mt][e] += (float)cy.hi[mt][e] + (float)cy.lo[mt][e];  // (zeros in the first pass)
      }
    } else if (piece == 4) {
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
        typename E::vec4 ov, lv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ov[e] = (T)o.sum[mt][e];
          lv[e] = MULTI ? (T)(o.sum[mt][e] - (float)ov[e]) : (T)0.f;
        }
        o.hi[mt] = __builtin_bit_cast(u32x2v, ov);
        o.lo[mt] = __builtin_bit_cast(u32x2v, lv);
      }
    } else {
      asm volatile("" : "+v"(lane_o));
      const int ln = lane_o;
      const int jl = ln & 31, d0 = 8 * wave + 4 * (ln >> 5);
      // (head dims that are no multiple of 32: a quarter past the end has no live lane)
      o.live = __builtin_amdgcn_ballot_w64((int)(jl < N - 32 * jt) & (int)(d0 < D)) & (jt < 0 ? 0ull : ~0ull);
      // (row strides of the gradients are below 2^24 bytes, like those of the inputs)
      o.off = (__umul24((uint32_t)jl, (uint32_t)a.sdq.j) + (uint32_t)d0) * (uint32_t)sizeof(T);
    }
  };
  // (a 64-bit base per query tile in scalar registers and the 32-bit byte offset of the lane; every lane of the wave is active here)
  auto store_dq = [&](int jt, const T* base, const DqOut& o) {
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      asm volatile("s_mov_b64 exec, %4\n\tglobal_store_dwordx2 %0, %1, %2 offset:%3\n\ts_mov_b64 exec, -1" : : "v"(o.off), "v"(o.hi[mt]), "s"(base), "n"(64 * mt), "s"(o.live) : "memory");
      if constexpr (MULTI) {
        const T* base_lo = lorow + (int64_t)(32 * jt) * D;
        const uint64_t live_lo = last_pass ? 0ull : o.live;
        asm volatile("" : "+v"(lane_o));
        const int ln = lane_o;
        const uint32_t off_lo = (uint32_t)((ln & 31) * D + 8 * wave + 4 * (ln >> 5)) * (uint32_t)sizeof(T);
        asm volatile("s_mov_b64 exec, %4\n\tglobal_store_dwordx2 %0, %1, %2 offset:%3\n\ts_mov_b64 exec, -1" : : "v"(off_lo), "v"(o.lo[mt]), "s"(base_lo), "n"(64 * mt), "s"(live_lo) : "memory");
      }
    }
  };

  TRI_ROW_MARK(t_p4);
#ifdef TRI_ROW_TIMING
  // one record of 32 words per workgroup (first wave), at the start of what db points to
  uint64_t* const rec = reinterpret_cast<uint64_t*>(a.db) + (int64_t)L * 32;
  if (wave == 0 && lane == 0) {
    const uint64_t t = __builtin_amdgcn_s_memrealtime();
    const uint32_t marks[5] = {t_entry, t_p1, t_p2, t_p3, t_p4};  // 100 MHz
    for (int x = 0; x < 5; ++x) rec[x] = t - ((uint32_t)t - marks[x]);
  }
#endif
  wait_dma_known();
  __syncthreads();

  // ---- query tiles ------------------------------------------------------------------
  // The loop exists in two versions, chosen once per wave: every key of the wave's
  // tiles attended (no mask work) and some keys masked out.  Inside a query tile the key tiles run as a software pipeline: the score
  // and dP MFMAs of tile t+1 are issued before the exponentials of tile t, and the dq
  // MFMAs of tile t-1 (whose dS has been through LDS by then) after them.
  auto query_tiles = [&](auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    int masked_bits = 0;  // bit t set: this lane's key of tile t is masked
    if constexpr (MASKED) {
#pragma unroll
      for (int t = 0; t < KT; ++t) masked_bits |= (kw[t] >> kl & 1u ? 0 : 1) << t;
    }
    // (each version has its own accumulators, from zeroing to the final stores: merging
    // the versions' accumulators where they meet would copy all of them)
    f32x16 dkacc[KT][DM], dvacc[KT][DM];
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
        if constexpr (TWO) {
          dkacc[t][mt] = dvacc[t][mt] = zero16();
        } else {
          E::mfma_acc_zero(dkacc[t][mt]);
          E::mfma_acc_zero(dvacc[t][mt]);
        }
      }
    // One wave per SIMD, or two, leave most of hiding a latency to a wave's own instruction
    // order: the code below is laid out as the schedule it should run in, and scheduling
    // barriers between the pieces keep the compiler from re-ordering it.
    auto SB = [] { __builtin_amdgcn_sched_barrier(0); };
    constexpr int NACC = 2 * PS * DM;  // dv, dk MFMAs of a tile
    constexpr int NDQ = PS * DM;       // dq MFMAs of a tile
    // packed bias of key tile t (t >= KT: tile t - KT of the next query tile) -> the ring slot
    // of that tile's parity, fetched two steps before its use (global memory, through L2).
    // (With an odd KT, tile 0 of the next query tile goes to the slot that tile KT-1 is read
    // from in the same step: its fetch follows the last MFMA that reads bias words.)
    u32x4v bias_ring[2][2] = {};
    auto fetch_bias = [&](int jt, int t) {
      bias_load(jt + t / KT, t % KT, bias_ring[(t % KT) % 2]);
    };
    fetch_bias(0, 0);
    fetch_bias(0, 1);
    uint32_t lw_next = 0u, dw_next = 0u;  // the words of the next query tile
    auto load_words = [&](int jt) {
      const int j = 32 * min(jt, NJ - 1) + perm32(kl);
      lw_next = nl[j];
      if constexpr (!O_STAGE) dw_next = nd[j];
    };
    if constexpr (WORDS_LDS) load_words(0);
    else fetch_words(0, lw_next, dw_next);
    DqCarry carry = {};
    const T* dq_base = dqrow;  // dq of the query tile before the current one (from the second on)
    // dq of a query tile is summed over the waves, and stored, during the first step of the
    // next query tile, which has no vector work of its own.
    int buf = 0;  // jt % 3: the stage of this query tile
#ifdef TRI_ROW_TIMING
    uint32_t tacc[KT + 5] = {};  // shader clocks per step, summed over the query tiles
    const uint32_t t_clk0 = (uint32_t)__builtin_amdgcn_s_memtime(), t_loop0 = (uint32_t)__builtin_amdgcn_s_memrealtime();
    uint32_t tprev = t_clk0;
#endif
    for (int jt = 0; jt < NJ; ++jt) {
      const int buf_fill = buf == 0 ? 2 : buf - 1;  // (jt + 2) % 3: the stage to refill
      DqParts parts;  // (of the query tile before this one)
      DqOut dq_words;
      f32x16 dqacc[DM];  // (the first dq MFMA of a query tile starts it from zero)
      const unsigned char* qt = tri_smem + OFF_ST + buf * STAGE;
      const unsigned char* dot = qt + 32 * ROWB;

      // operand words of this lane's query (lanes 32..63 carry zeros)
      s_off.set_raw(g ? 0u : lw_next);
      if constexpr (!O_STAGE) d_off.v[0] = g ? 0u : dw_next;
      frag qn[DS], don[DS], on[O_STAGE ? DS : 1];
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        qn[s] = ofq.natural(qt, s);
        don[s] = ofq.natural(dot, s);
        if constexpr (O_STAGE) on[s] = ofq.natural(dot + 32 * ROWB, s);
      }
      // delta of the query tile, of which a lane holds half a row, in four sums and their total; the word is kept for the end of
      // the row, by every wave for itself
      float dsum[4];
      auto set_delta = [&](int piece) __attribute__((always_inline)) {
        typedef T pair __attribute__((ext_vector_type(2)));
        if (piece < 2) {
#pragma unroll
          for (int s = piece * DS / 2; s < (piece + 1) * DS / 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; e += 2)
              dsum[e / 2] = pair_dot(pair{on[s][e], on[s][e + 1]}, pair{don[s][e], don[s][e + 1]}, s == 0 ? 0.f : dsum[e / 2]);
        } else {
          const uint32_t word = split_word<T>(-half_sum((dsum[0] + dsum[1]) + (dsum[2] + dsum[3])));
          nd[32 * jt + perm32(kl)] = word;
          d_off.v[0] = word & (uint32_t)((g | (int)(perm32(kl) >= N - 32 * jt)) - 1);
        }
      };
      // Q^T, dO^T (A operands of dk, dv): transposing reads are the slowest LDS reads and the
      // four waves share one LDS pipe, so they are read once per query tile where registers
      // allow and again for every key tile where they do not
      constexpr bool QD_ONCE = D <= 32;
      frag qtr[DM][PS], dotr[DM][PS];
      auto load_qd_tr = [&] {
#pragma unroll
        for (int mt = 0; mt < DM; ++mt)
#pragma unroll
          for (int s2 = 0; s2 < PS; ++s2) {
            qtr[mt][s2] = ofq.transposed_all(qt, s2, mt);
            dotr[mt][s2] = ofq.transposed_all(dot, s2, mt);
          }
      };

      // ---- the state that moves from step to step --------------------------------------
      f32x16 s_cur, p_cur;   // scores and dP of the tile whose P, dS the step computes
      f32x16 s_nxt, p_nxt;   // ... of the tile after it, accumulating
      float p[16], ds[16];
      frag kn[DS];           // K rows of the next tile as B operand
      frag pf[PS], dsf[PS];  // P and dS of the last finished tile as B operands
      frag dst_prev[PS], ktr_prev[DM][PS];
      frag vn[DS];           // V operands of the next tile when they live in LDS
      auto load_kn = [&](int t) {
        const unsigned char* ktile = lds_k + NW * t * 32 * ROWB;
#pragma unroll
        for (int s = 0; s < DS; ++s) kn[s] = ofk.natural(ktile, s);
      };
      load_kn(0);

      // Step t (t = -1 .. KT): the vector work of tile t (P, dS, their conversions) between
      // the MFMAs of its neighbours: dv, dk and dq of tile t-1, scores and dP of tile t+1,
      // in the order of RowSched.  Step -1 only starts tile 0, step KT only finishes tile KT-1.
      auto step = [&](auto tc) __attribute__((always_inline)) {
        constexpr int t = decltype(tc)::value - 1;
        constexpr bool has_prev = t >= 1, has_next = t + 1 < KT, valu = t >= 0 && t < KT;
        constexpr int tn = has_next ? t + 1 : 0, tp = has_prev ? t - 1 : 0;
        using Sch = RowSchedOf<has_prev, has_next, NSB, DS, NACC, NDQ>;
        constexpr int NM = Sch::value.n;
        constexpr int NU = valu ? 16 : 0;  // vector units of four instructions
        // Step KT-2 starts the query tile after next on its way to LDS, right after its last
        // read of bias words: loads return in issue order,
        // so the next wait for bias words is a wait for these loads too, and from there it is
        // the furthest away, at the start of the next query tile.
        constexpr bool refill = t == KT - 2;
        constexpr int refill_at = Sch::value.last_sb;
        SB();
        frag kb = keys_op.plain();
        if constexpr (has_next && MASKED) kb = keys_op.masked_bit(masked_bits, tn);
        SB();
        TRI_ROW_TICK(t + 1);  // (slot 0: from the loop head to step -1; slot k: step k-2)
        // (words from the global planes: those of the next query tile, fetched before the last
        // bias tile of this one so that no wait for them is a wait for everything in flight)
        if constexpr (!WORDS_LDS && t == KT - 1) fetch_words(jt + 1, lw_next, dw_next);
        if constexpr (WORDS_LDS && t == KT) load_words(jt + 1);  // (in front of the barrier: not another trip to LDS behind it)
        if constexpr (valu && !refill) fetch_bias(jt, t + 2);
        SB();
        auto unit = [&](int u) __attribute__((always_inline)) {
          if (u < 8) {
#pragma unroll
            for (int e = 0; e < 2; ++e) p[2 * u + e] = fast_exp2(s_cur[2 * u + e] * c);
          } else if (u < 12) {
#pragma unroll
            for (int e = 0; e < 4; ++e) ds[4 * (u - 8) + e] = p[4 * (u - 8) + e] * p_cur[4 * (u - 8) + e];
          } else if (u < 14) {
            pf[u - 12] = E::pack(&p[KP * (u - 12)]);
          } else {
            dsf[u - 14] = E::pack(&ds[KP * (u - 14)]);
          }
        };
        static_for<NM>([&](auto xc) __attribute__((always_inline)) {
          constexpr int x = decltype(xc)::value;
          constexpr int kind = Sch::value.kind[x], idx = Sch::value.idx[x];
          if constexpr (kind == R_SOFF) {
            s_nxt = E::mfma(s_off.get(), kb, zero16());
          } else if constexpr (kind == R_SB) {
            s_nxt = E::mfma(__builtin_bit_cast(frag, bias_ring[tn % 2][idx / NPART]), bsel[idx / NPART][idx % NPART], s_nxt);
          } else if constexpr (kind == R_SQK) {
            s_nxt = E::mfma(qn[idx], kn[idx], s_nxt);
          } else if constexpr (kind == R_DOFF) {
            p_nxt = E::mfma(__builtin_bit_cast(frag, d_off.v), kb, zero16());
          } else if constexpr (kind == R_DP) {
            if constexpr (tn < VR) p_nxt = E::mfma(don[idx], vf[tn][idx], p_nxt);
            else p_nxt = E::mfma(don[idx], vn[idx], p_nxt);
          } else if constexpr (kind == R_ACC) {
            constexpr int s2 = (idx / 2) / DM, mt = (idx / 2) % DM;
            if constexpr (TWO && idx % 2 == 0) dvacc[tp][mt] = E::mfma(dotr[mt][s2], pf[s2], dvacc[tp][mt]);
            else if constexpr (TWO) dkacc[tp][mt] = E::mfma(qtr[mt][s2], dsf[s2], dkacc[tp][mt]);
            else if constexpr (idx % 2 == 0) E::mfma_acc(dotr[mt][s2], pf[s2], dvacc[tp][mt]);
            else E::mfma_acc(qtr[mt][s2], dsf[s2], dkacc[tp][mt]);
          } else {
            if constexpr (tp == 0 && idx / DM == 0) dqacc[idx % DM] = E::mfma(ktr_prev[idx % DM][idx / DM], dst_prev[idx / DM], zero16());
            else dqacc[idx % DM] = E::mfma(ktr_prev[idx % DM][idx / DM], dst_prev[idx / DM], dqacc[idx % DM]);
          }
          SB();
          if constexpr (O_STAGE && t == -1 && x < 3) set_delta(x);
          // Q^T, dO^T of the query tile are first used by the step after next: their reads go
          // where the LDS pipe has nothing else to do
          if constexpr (QD_ONCE && t == -1 && x == 1) load_qd_tr();
          // dq of the query tile before this one: its parts come from LDS early in this step,
          // which has no vector work of its own, and are summed and stored piece by piece behind
          // the MFMAs that follow (before the first query tile the sum is of stale bytes and is
          // not stored).  No wait for a load that could follow within the time a store takes
          // allows fewer than two operations in flight, so none of them waits for this store
          // (a wait for loads issued after a store is a wait for the store as well).
          if constexpr (t == -1) {
            if constexpr (x == 0) load_partials((jt + 1) & 1, parts);
#pragma unroll
            for (int piece = 0; piece < kSumPieces; ++piece)
              if ((piece + 3 < NM ? piece + 3 : NM - 1) == x) sum_dq_piece(piece, jt - 1, parts, carry, dq_words);
            if constexpr (x == NM - 1) {
              store_dq(jt - 1, dq_base, dq_words);
              dq_base += jt > 0 ? 32 * a.sdq.j : 0;
              if constexpr (MULTI) {
                if (!first_pass) fetch_carry(jt, carry);
              }
            }
          }
          if constexpr (has_prev && x == Sch::value.dq_reads_at) {
            // dS of tile t-1 comes back from LDS with the key index in-lane, with the K
            // rows of that tile transposed beside it
            const unsigned char* ktile = lds_k + NW * tp * 32 * ROWB;
#pragma unroll
            for (int s2 = 0; s2 < PS; ++s2) {
              dst_prev[s2] = ofd.transposed(ds_tile, s2, 0);
#pragma unroll
              for (int mt = 0; mt < DM; ++mt) ktr_prev[mt][s2] = ofk.transposed_all(ktile, s2, mt);
            }
          }
          if constexpr (refill && x == refill_at) {
            issue_stage(buf_fill);
            fetch_bias(jt, t + 2);
          }
          if constexpr (has_next && x == Sch::value.last_sqk && t + 2 < KT) load_kn(t + 2);
          if constexpr (has_next && tn >= VR && x == Sch::value.v_reads_at) {
#pragma unroll
            for (int s = 0; s < DS; ++s) vn[s] = v_lds[((tn - VR) * DS + s) * 64];
          }
#pragma unroll
          for (int u = x * NU / NM; u < (x + 1) * NU / NM; ++u) unit(u);
          SB();
        });
        if constexpr (valu) {
          // dS -> one of the wave's two LDS tiles [key][query]; Q^T, dO^T for the dv, dk
          // MFMAs of this tile, which the next step starts with
          *reinterpret_cast<frag*>(ds_tile + ds_w0) = dsf[0];
          *reinterpret_cast<frag*>(ds_tile + ds_w1) = dsf[1];
          if constexpr (!QD_ONCE) load_qd_tr();
          SB();
        }
        if constexpr (has_next) { s_cur = s_nxt; p_cur = p_nxt; }
      };
      static_for<KT + 2>(step);
      TRI_ROW_TICK(KT + 2);
      store_partials(jt & 1, dqacc);
      TRI_ROW_TICK(KT + 3);
      // The stage of the next query tile was requested a whole query tile ago; since then
      // the wave has issued the loads of the stage after it and of two bias tiles: everything older than those has landed.  A barrier
      // without a fence: a fence would wait for the loads in flight.  It is the only one of
      // the query tile: the partials written before it are read after it, and the buffer they
      // are in is written again two query tiles on, behind the next barrier.
      ring_sync<G2W + 4 + (WORDS_LDS ? 0 : 2)>();
      TRI_ROW_TICK(KT + 4);
      buf = buf == 2 ? 0 : buf + 1;
    }
    {
      DqParts parts;
      DqOut dq_words;
      load_partials((NJ - 1) & 1, parts);
#pragma unroll
      for (int piece = 0; piece < kSumPieces; ++piece) sum_dq_piece(piece, NJ - 1, parts, carry, dq_words);
      store_dq(NJ - 1, dq_base, dq_words);
    }
#ifdef TRI_ROW_TIMING
    const uint32_t t_clk1 = (uint32_t)__builtin_amdgcn_s_memtime(), t_loop1 = (uint32_t)__builtin_amdgcn_s_memrealtime();
#endif

    // the words that the db kernel reads (each thread writes what its own wave has put there)
    if constexpr (O_STAGE) {
#pragma unroll
      for (int x = 0; x < LSE_N; ++x) {
        const int j = x * NW * 64 + tid;
        if (j < N) dplane[j] = nd[j];
      }
    }
    // ---- dk, dv of this wave's keys -------------------------------------------------------
    // (the accumulators were last written by MFMAs inside asm statements, which the compiler
    // does not know to be MFMAs: each is read only after that MFMA has had time to retire)
    T* dkrow = reinterpret_cast<T*>(a.dk) + b * a.sdk.b + h * a.sdk.h + i * a.sdk.i;
    T* dvrow = reinterpret_cast<T*>(a.dv) + b * a.sdv.b + h * a.sdv.h + i * a.sdv.i;
  #pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int key = 32 * (KT0 + NW * t + wave) + kl;
  #pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
#ifndef TRI_MFMA_ACC_BUILTIN
        if constexpr (!TWO) {
          asm volatile("s_nop 15" : "+a"(dkacc[t][mt]));
          asm volatile("s_nop 15" : "+a"(dvacc[t][mt]));
        }
#endif
      }
      store_rows_wide<T, D, DM>(dkrow + (int64_t)key * a.sdk.j, dkacc[t], a.scale, g, key < N);
      store_rows_wide<T, D, DM>(dvrow + (int64_t)key * a.sdv.j, dvacc[t], 1.0f, g, key < N);
    }
#ifdef TRI_ROW_TIMING
    if (wave == 0 && lane == 0) {
      const uint64_t t_end = __builtin_amdgcn_s_memrealtime();
      rec[5] = t_end - ((uint32_t)t_end - t_loop0);
      rec[6] = t_end - ((uint32_t)t_end - t_loop1);
      rec[7] = t_end;
      rec[8] = __builtin_amdgcn_s_getreg(4 | (0 << 6) | (31 << 11));   // HW_ID
      rec[9] = __builtin_amdgcn_s_getreg(20 | (0 << 6) | (31 << 11));  // XCC_ID
      rec[10] = (uint32_t)(t_clk1 - t_clk0);                            // shader clocks of the loop
      for (int x = 0; x < KT + 5; ++x) rec[11 + x] = tacc[x];
      rec[28] = KT;  // what the record is of: key tiles per wave, waves per row, kernel (0: this one, 1: short rows)
      rec[29] = NW;
      rec[30] = 0;
    }
#endif
  };
  bool plain = true;
#pragma unroll
  for (int t = 0; t < KT; ++t) plain = plain && kw[t] == 0xffffffffu;
  if (plain) query_tiles(std::false_type{});
  else query_tiles(std::true_type{});

}

}  // namespace tri
