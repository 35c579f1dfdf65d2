// Backward kernel 3 of 3: db[j, k] = sum over rows i of dS[i, j, k].
//
// Work unit: (batch*head, chunk of pair rows i, block of GJ*WJ*32 queries j, block
// of GK*WK*32 keys k).  The GJ x GK waves of a workgroup each own WJ x WK tiles of
// 32 x 32 and keep their db tiles in fp32 registers while the workgroup walks the
// rows of its chunk, so the reduction over i has one fixed order and needs no
// atomics.  Per row the workgroup stages the Q, dO rows of its queries and the K,
// V rows of its keys in LDS (direct global->LDS loads into a ring of row buffers
// that runs several rows ahead of the compute, swizzled tiles) together with
// the lse and delta operand words left by the dq kernel, and each wave
// recomputes for its tiles
//   S^T = K Q^T + bias - lse, P^T = exp2(c S^T), dP^T = V dO^T - delta, dS^T = P^T dP^T
// with every operand in its natural row-major layout: a lane owns one query
// (column) and 16 keys of each tile.  The additive terms cost the vector ALU nothing:
// the bias tiles (register-resident, fp32, raw-score domain) are the accumulator
// init of every row's score MFMA; -delta (per query) enters through one extra MFMA
// (see rank1_operand); -lse is one number per lane and is the addend of the fma that
// scales the score for exp2.  That leaves two fmas and one exp2 per element.  In the general
// loop a tile with masked keys takes -lse in an extra MFMA that it shares with the key mask (see
// OffsetMask): masked keys get a large negative score there.
//
// Waves that own two key tiles of rows of up to 128 bytes walk the rows, masked or not, as a
// hand-made software pipeline (matrix instructions of one tile between the vector instructions of
// the tile before it, operands a row ahead); see kPipelined below.
//
// All workgroups of one (batch*head, chunk) read the same rows at about the same
// time; the block index is remapped so that they run on one XCD and share its L2.
// When the rows are split into several chunks (to fill the GPU), each chunk writes
// an fp32 partial and a second kernel adds the partials in chunk order.
//
// Replaces _bwd_b of reference src/trifast/triton.py:394-501.
#pragma once
#include <type_traits>

#include "tri_args.hpp"
#include "tri_common.hpp"
#include "tri_f32_plain.hpp"
#include "tri_tile.hpp"

// -DTRI_DB_TIMING builds the kernel as a probe of its pipelined walk
// (benchmark/microbench/db_timeline.py): every wave reads the shader clock around the counted
// wait and the barrier that end a row, and leaves per wave {clocks of the walk, clocks in the
// wait, clocks in the barrier, 100 MHz ticks of the walk} where the db argument points; db
// itself is not written.  -DTRI_DB_TIMING_LOADS=0 also takes the walk's global loads out (the
// rows in LDS are then stale), =2 makes them read one row over and over (the same traffic from
// L2 to LDS, none from memory): what the loads cost the arithmetic beside them.
#if defined(TRI_DB_TIMING) && !defined(TRI_DB_TIMING_LOADS)
#define TRI_DB_TIMING_LOADS 1
#endif

namespace tri {

// LDS bytes of one stage (one pair row) of the kernel below
constexpr int bwd_b_stage_bytes(int BJ, int BKB, int ROWB) { return 2 * (BJ * 4 + 256) + (2 * BJ + 2 * BKB) * ROWB; }
// and of its fp32 version
constexpr int bwd_b_split_stage_bytes(int BJ, int BKB, int D) { return (D > 64 ? 1 : 2) * (BJ + BKB) * lds_row_bytes(D, 4); }

// The workgroup's part of the problem.
struct DbBlock {
  int bh, chunk, j, k;  // batch * head, chunk of pair rows, first query and key
  bool live;
};
TRI_DEV DbBlock db_block(const BwdArgs& a, int BJ, int BKB) {
  // Linear block id L = 8 * slot + xcd (workgroups go to the 8 XCDs round-robin).
  // Every XCD walks its own sequence of (batch*head, chunk) groups; the launcher
  // pads the group count to a multiple of 8.
  // With fewer than 8 groups each group gets 8 / groups XCDs (whole number) and deals its
  // blocks to them in turn, so that no XCD stays idle: the rows are then fetched once per XCD
  // of the group.
  const int per_group = gridDim.x * gridDim.y;
  const int L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const int slot = L >> 3;
  const int ngroups = a.BH * a.nchunks;
  const int share = ngroups >= 8 ? 1 : 8 / ngroups;  // XCDs per group
  const int group = share == 1 ? 8 * (slot / per_group) + (L & 7) : (L & 7) / share;
  const int within = share == 1 ? slot % per_group : slot * share + (L & 7) % share;
  return DbBlock{group % a.BH, group / a.BH, (int)(within % gridDim.x) * BJ, (int)(within / gridDim.x) * BKB, group < ngroups && within < per_group};
}

// db tiles of a wave -> db, or the partial sums of its chunk
template <typename T, int WJ, int WK>
TRI_DEV void store_db(const BwdArgs& a, const f32x16 (&dbacc)[WJ][WK], int bh, int chunk, int j_wave, int k_wave, int jl, int g) {
  using E = Elem<T>;
  const int N = a.N, b = bh / a.H, h = bh % a.H;
  // a single chunk writes db itself; several chunks write fp32 partials.  The lane
  // owns query j; its 16 values are two runs of 8 consecutive keys.
  const bool direct = a.nchunks == 1;
  T* db_bh = reinterpret_cast<T*>(a.db) + b * a.sdb_b + h * a.sdb_h;
  float* part = a.dbpart + ((int64_t)chunk * a.BH + bh) * N * N;
  const bool vec_store = (N % 8) == 0;
  // 16-byte stores of 8 keys need db contiguous along k with rows that stay aligned
  const bool db_vec = a.sdb_k == 1 && ((a.sdb_j | a.sdb_h | a.sdb_b) % 8) == 0;
#pragma unroll
  for (int tj = 0; tj < WJ; ++tj) {
    const int j = j_wave + 32 * tj + jl;
    if (j >= N) continue;
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int key0 = k_wave + 32 * tk + 16 * r + 8 * g;
        if (!direct) {
          float* dst = part + (int64_t)j * N + key0;
          if (vec_store && key0 + 8 <= N) {
#pragma unroll
            for (int e4 = 0; e4 < 2; ++e4) {
              f32x4 ov;
#pragma unroll
              for (int e = 0; e < 4; ++e) ov[e] = dbacc[tj][tk][8 * r + 4 * e4 + e];
              *reinterpret_cast<f32x4*>(dst + 4 * e4) = ov;
            }
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (key0 + e < N) dst[e] = dbacc[tj][tk][8 * r + e];
          }
          continue;
        }
        T* dst = db_bh + j * a.sdb_j + key0 * a.sdb_k;
        if (db_vec && key0 + 8 <= N) {
          if constexpr (sizeof(T) == 2) {
            typename E::vec ov;
#pragma unroll
            for (int e = 0; e < 8; ++e) ov[e] = (T)dbacc[tj][tk][8 * r + e];
            *reinterpret_cast<typename E::vec*>(dst) = ov;
          } else {
#pragma unroll
            for (int e4 = 0; e4 < 2; ++e4) {
              f32x4 ov;
#pragma unroll
              for (int e = 0; e < 4; ++e) ov[e] = dbacc[tj][tk][8 * r + 4 * e4 + e];
              *reinterpret_cast<f32x4*>(dst + 4 * e4) = ov;
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (key0 + e < N) dst[e * a.sdb_k] = (T)dbacc[tj][tk][8 * r + e];
        }
      }
    }
  }
}

template <typename T, int D, int GJ, int GK, int WJ, int WK, int NBUF>
__global__ __launch_bounds__(GJ * GK * 64) void tri_bwd_b_kernel(const BwdArgs a) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using Tile = LdsTile<T, D>;
  constexpr int KP = E::KP;
  constexpr int DS = D / (2 * KP);
  constexpr int NW = GJ * GK;
  constexpr int BJ = GJ * WJ * 32, BKB = GK * WK * 32;  // queries / keys per workgroup
  constexpr int ROWB = Tile::ROWB;
  // one stage: lse2[BJ] | 64 keep words | -delta[BJ] | 64 spare words | Q rows | dO rows |
  // K rows | V rows.  The small arrays come first so that their offsets in every ring
  // buffer fit the 16-bit immediate of an LDS read.  (The general loop takes the row's flag and
  // keep words by scalar loads instead: it branches on them.)
  constexpr int OFF_LSE = 0, OFF_KW = OFF_LSE + BJ * 4, OFF_DELTA = OFF_KW + 256;
  constexpr int OFF_Q = OFF_DELTA + BJ * 4 + 256, OFF_DO = OFF_Q + BJ * ROWB, OFF_K = OFF_DO + BJ * ROWB, OFF_V = OFF_K + BKB * ROWB;
  constexpr int STAGE = OFF_V + BKB * ROWB;
  static_assert(STAGE == bwd_b_stage_bytes(BJ, BKB, ROWB), "the launcher sizes LDS with bwd_b_stage_bytes");

  extern __shared__ __attribute__((aligned(16))) unsigned char tri_smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int jl = lane & 31, g = lane >> 5;
  const int N = a.N;

  const DbBlock blk = db_block(a, BJ, BKB);
  if (!blk.live) return;
  const int bh = blk.bh, chunk = blk.chunk, j_blk = blk.j, k_blk = blk.k;
  const int b = bh / a.H, h = bh % a.H;
  const int wj = wave % GJ, wk = wave / GJ;
  const int j_wave = j_blk + wj * (WJ * 32), k_wave = k_blk + wk * (WK * 32);
  // the rows in front of the first fully masked one take the loop of their own below
  constexpr bool kPipelined = WJ == 1 && WK == 2 && NBUF >= 2 && D <= 64;
  // What the rows of the chunk are like: every thread looks at its share of them, the result goes
  // through words of LDS, which is not yet in use (scan_words).
  //   * Where the run of fully masked rows at the end of the row range starts (padding; looked for only where
  //     the last row is fully masked: a scan on every launch cost 2 % at n = 704, 5 rounds of 88 rows).
  //     A chunk is a share of the rows in front and a share of the run: rows of the run take about
  //     half the time of the others.
  //   * (pipelined walk) The rows from the first to the last with an attended key of this block: the others add
  //     nothing and are left out (n = 1024, h = 4, d = 32, four parts that attend to themselves: 0.81 -> 0.26 ms; before
  //     the walk took masked rows 0.75, in the 16-wave block 0.69).
  //     Of those rows, the first fully masked one; whether any other masks a key of the block; which key tiles of the
  //     block have an attended key in any of them, and which have none in some.
  uint32_t* scan_words = reinterpret_cast<uint32_t*>(tri_smem);
  if (tid == 0) {
    scan_words[0] = 0;
    scan_words[1] = (uint32_t)N;
    scan_words[2] = 0;            // key tiles with an attended key in some row; from bit 8 on those with a masked one; from bit 16
                                  // on those without an attended one in some row
    scan_words[3] = (uint32_t)N;  // the first row with an attended key of the block, the row past the last, how many there are
    scan_words[4] = scan_words[5] = 0;
  }
  __syncthreads();
  const uint32_t* flags = a.rowflag + (int64_t)b * N;
  auto share_of = [&](int rows, int at) { return __builtin_amdgcn_readfirstlane((int)((uint32_t)rows * (uint32_t)at / (uint32_t)a.nchunks)); };
  // (keys past the end of the row feed entries that are never stored: they do not count as masked)
  auto past_end = [&](int word) { return word == a.nwords - 1 && (N & 31) != 0 ? 0xffffffffu << (N & 31) : word >= a.nwords ? 0xffffffffu : 0u; };
  int i_begin = share_of(N, chunk), i_end = share_of(N, chunk + 1), run_begin = N;
  if (uniform_word(a.rowflag, (int64_t)b * N + N - 1) != 0) {
    uint32_t last_other = 0;
    for (int i = tid; i < N; i += NW * 64)
      if (flags[i] == 0) last_other = (uint32_t)i + 1;
    if (last_other) atomicMax(scan_words, last_other);
    __syncthreads();
    run_begin = __builtin_amdgcn_readfirstlane((int)scan_words[0]);
    i_begin = share_of(run_begin, chunk);
    i_end = share_of(run_begin, chunk + 1);
  }
  if constexpr (kPipelined) {
    // (a wave takes 64 rows side by side: what they are like together is a few scalar instructions)
    uint32_t tiles = 0;
    int first = N, last = 0, count = 0, first_flagged = N;
    for (int i0 = i_begin + wave * 64; i0 < i_end; i0 += NW * 64) {
      const int i = i0 + lane;
      const bool flagged = i < i_end && flags[i] != 0;
      uint32_t live = 0, rest = 0;
      if (i < i_end && !flagged) {
        const uint32_t* kw = a.keep + ((int64_t)b * N + i) * a.nwords;
#pragma unroll
        for (int w = 0; w < BKB / 32; ++w) {
          const uint32_t x = k_blk / 32 + w < a.nwords ? kw[k_blk / 32 + w] : 0u;
          const uint32_t past = past_end(k_blk / 32 + w);
          live |= x != 0 ? 1u << w : 0u;
          rest |= (x == 0 && past != 0xffffffffu ? 0x10000u << w : 0u) | ((x | past) != 0xffffffffu ? 0x100u << w : 0u);
        }
      }
      const uint64_t fl = __ballot(flagged), lv = __ballot(flagged || live != 0);
      if (fl != 0) {
        first_flagged = min(first_flagged, i0 + __builtin_ctzll(fl));
        tiles |= 0xffu;
      }
      if (lv != 0) {
        first = min(first, i0 + __builtin_ctzll(lv));
        last = i0 + 64 - __builtin_clzll(lv);
        count += __builtin_popcountll(lv);
      }
      const uint32_t t = live != 0 ? live | rest : 0u;
#pragma unroll
      for (int w = 0; w < BKB / 32; ++w)
#pragma unroll
        for (int f = 0; f < 3; ++f) tiles |= __ballot((t >> (8 * f + w) & 1u) != 0) != 0 ? 1u << (8 * f + w) : 0u;
    }
    if (lane == 0 && count != 0) {
      atomicMin(scan_words + 1, (uint32_t)first_flagged);
      atomicOr(scan_words + 2, tiles);
      atomicMin(scan_words + 3, (uint32_t)first);
      atomicMax(scan_words + 4, (uint32_t)last);
      atomicAdd(scan_words + 5, (uint32_t)count);
    }
  }
  __syncthreads();
  // (pinned to scalar registers: the branches of the walk must be real ones, see compute_row)
  i_begin = __builtin_amdgcn_readfirstlane(i_begin);
  run_begin = __builtin_amdgcn_readfirstlane(run_begin);
  uint32_t block_tiles = 0xffu;
  if constexpr (kPipelined) {
    block_tiles = __builtin_amdgcn_readfirstlane(scan_words[2]);
    const int count = __builtin_amdgcn_readfirstlane((int)scan_words[5]);
    if (count != 0) {
      i_begin = __builtin_amdgcn_readfirstlane((int)scan_words[3]);
      i_end = __builtin_amdgcn_readfirstlane((int)scan_words[4]);
      if (count != i_end - i_begin) block_tiles |= 0xffff00u;  // rows without an attended key among them
    }
  }
  int nrows = __builtin_amdgcn_readfirstlane(i_end) - i_begin;
  const int tail_begin = run_begin + share_of(N - run_begin, chunk), tail_end = run_begin + share_of(N - run_begin, chunk + 1);
  // rows that take the pipelined walk, and the block's key tiles (see scan_words)
  int nwalk = kPipelined ? __builtin_amdgcn_readfirstlane(min((int)scan_words[1] - i_begin, nrows)) : 0;
  if ((block_tiles & 0xffu) == 0) nrows = nwalk = 0;  // no attended key in any row: dS = 0
  __syncthreads();

  const T* qbase = reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h;
  const T* kbase = reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h;
  const T* vbase = reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h;
  const T* dobase = reinterpret_cast<const T*>(a.dout) + b * a.sdo.b + h * a.sdo.h;
  const T* pack_bh = reinterpret_cast<const T*>(a.packq) + (int64_t)bh * a.NP * a.NP * 1024;
  const float* lse2_bh = reinterpret_cast<const float*>(a.lse2) + (int64_t)bh * N * N;    // 32-bit words, moved as floats
  const float* delta_bh = reinterpret_cast<const float*>(a.delta) + (int64_t)bh * N * N;

  // bias tiles in the raw-score domain: accumulator init of every row's score MFMA.  (Each loop over
  // the rows fetches its own: tiles that are live across the choice between the loops end up in scratch
  // memory.  The tag keeps the compiler from making the fetches one again in front of the choice.)
  auto load_bias = [&](f32x16 (&biasr)[WJ][WK], auto tag) __attribute__((always_inline)) {
    int lane_now = lane;
    asm volatile("; bias of loop %1" : "+v"(lane_now) : "n"(decltype(tag)::value));
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj)
#pragma unroll
      for (int tk = 0; tk < WK; ++tk)
        biasr[tj][tk] = bias_tile<T>(pack_bh, a.NP, min((j_wave >> 5) + tj, a.NP - 1), min((k_wave >> 5) + tk, a.NP - 1), lane_now, a.sqrt_d, 0.f);
  };

  f32x16 dbacc[WJ][WK];
#pragma unroll
  for (int tj = 0; tj < WJ; ++tj)
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) dbacc[tj][tk] = zero16();

  // The loads of one row, as two lists of wave-sized items: 1 KiB pieces of the Q, dO, K,
  // V tiles (16 bytes per lane), and 64-float pieces of lse2 and -delta (4 bytes per lane).  Wave w takes items w, w + NW, ...
  // of each list; every wave issues exactly XW wide and XF narrow loads per row, in that
  // order (a wave that runs out repeats the last item of the list, which rewrites the same
  // bytes), so the width of a load is known at compile time and "all but the newest K rows
  // have landed" is one s_waitcnt vmcnt(K * XN) for every wave.  Queries and keys past
  // the end are clamped (they feed db entries that are never stored).
  constexpr int CPR = Tile::CPR;
  constexpr int GQ = BJ * CPR / 64, GKK = BKB * CPR / 64, GF = BJ / 64;
  constexpr int TOTW = 2 * GQ + 2 * GKK, TOTF = 2 * GF + (kPipelined ? 1 : 0);
  constexpr int XW = (TOTW + NW - 1) / NW, XF = (TOTF + NW - 1) / NW;
  constexpr int XN = XW + XF;
  static_assert(BJ * CPR % 64 == 0 && BKB * CPR % 64 == 0 && BJ % 64 == 0, "whole wave loads only");
  auto uniform64 = [](int64_t x) -> int64_t {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x), hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
  };
  // An item's source is a 64-bit base (wave-uniform, scalar registers, stepped from one pair
  // row to the next with scalar adds) plus a 32-bit byte offset per lane that never changes.
  // Where every wave takes the same number of items of each tensor, the items of a tensor share
  // one base, and their places in LDS are the wave's share plus constants.
  constexpr bool kShared = GQ % NW == 0 && GKK % NW == 0;
  constexpr int NBASE = kShared ? 4 + XF : XN;
  auto base_of = [](int x) constexpr {
    if (!kShared) return x;
    if (x >= XW) return 4 + x - XW;
    const int it = x * NW;
    return it < GQ ? 0 : it < 2 * GQ ? 1 : it < 2 * GQ + GKK ? 2 : 3;
  };
  const char* item_base[NBASE];
  int64_t item_step[NBASE];   // bytes from one pair row to the next (wave-uniform)
  uint32_t item_voff[XN];
  int item_lds[XN];           // destination offset inside a stage (wave-uniform)
  // (items 0 .. XW-1 move 16 bytes per lane, items XW .. XN-1 4 bytes)
  {
    const int es = (int)sizeof(T);
    auto tile_item = [&](int x, int gi, const T* base, int64_t srow, int64_t si, int blk, int off) {
      const int p = gi * 64 + lane;
      const int r = p / CPR, cc = (p % CPR) ^ Tile::swz(r);
      item_base[base_of(x)] = reinterpret_cast<const char*>(uniform64((int64_t)(uintptr_t)(base + (int64_t)blk * srow + (int64_t)i_begin * si)));
      // (row strides are below 2^24 bytes)
      item_voff[x] = __umul24((uint32_t)min(r, N - 1 - blk), (uint32_t)srow * (uint32_t)es) + (uint32_t)(cc * 16);
      item_step[base_of(x)] = uniform64(si * es);
      item_lds[x] = off + gi * 1024;
    };
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      if (kShared && x < XW) {
        const int first = x * NW;  // (a constant: so is the tensor)
        if (first < GQ) tile_item(x, first + wave, qbase, a.sq.j, a.sq.i, j_blk, OFF_Q);
        else if (first < 2 * GQ) tile_item(x, first - GQ + wave, dobase, a.sdo.j, a.sdo.i, j_blk, OFF_DO);
        else if (first < 2 * GQ + GKK) tile_item(x, first - 2 * GQ + wave, kbase, a.sk.j, a.sk.i, k_blk, OFF_K);
        else tile_item(x, first - 2 * GQ - GKK + wave, vbase, a.sv.j, a.sv.i, k_blk, OFF_V);
        continue;
      }
      // position in the flat order Q | dO | K | V | lse2 | delta | keep words
      const int it = x < XW ? __builtin_amdgcn_readfirstlane(min(x * NW + wave, TOTW - 1))
                            : TOTW + __builtin_amdgcn_readfirstlane(min((x - XW) * NW + wave, TOTF - 1));
      if (it < GQ) {
        tile_item(x, it, qbase, a.sq.j, a.sq.i, j_blk, OFF_Q);
      } else if (it < 2 * GQ) {
        tile_item(x, it - GQ, dobase, a.sdo.j, a.sdo.i, j_blk, OFF_DO);
      } else if (it < 2 * GQ + GKK) {
        tile_item(x, it - 2 * GQ, kbase, a.sk.j, a.sk.i, k_blk, OFF_K);
      } else if (it < 2 * GQ + 2 * GKK) {
        tile_item(x, it - 2 * GQ - GKK, vbase, a.sv.j, a.sv.i, k_blk, OFF_V);
      } else if (kPipelined && it == TOTW + TOTF - 1) {
        item_base[base_of(x)] = reinterpret_cast<const char*>(uniform64((int64_t)(uintptr_t)(a.keep + ((int64_t)b * N + i_begin) * a.nwords)));
        item_voff[x] = (uint32_t)(min(k_blk / 32 + lane, a.nwords - 1) * 4);
        item_step[base_of(x)] = uniform64((int64_t)a.nwords * 4);
        item_lds[x] = OFF_KW;
      } else {
        const int f = it - 2 * GQ - 2 * GKK;
        const int gi = f % GF;
        const float* base = (f < GF) ? lse2_bh : delta_bh;
        const int j0 = min(j_blk + gi * 64, N - 1);
        item_base[base_of(x)] = reinterpret_cast<const char*>(uniform64((int64_t)(uintptr_t)(base + (int64_t)i_begin * N + j0)));
        item_voff[x] = (uint32_t)(min(lane, N - 1 - j0) * 4);
        item_step[base_of(x)] = uniform64((int64_t)N * 4);
        item_lds[x] = ((f < GF) ? OFF_LSE : OFF_DELTA) + gi * 256;
      }
    }
  }
  // all ones if x > 0, else zero, as a 64-bit scalar (written out: the compiler would keep the
  // condition as a lane mask and turn it into a number with vector instructions in every row)
  auto ones_while_positive = [](int x) -> int64_t {
    int64_t m;
    asm volatile("s_cmp_gt_i32 %1, 0\n\ts_cselect_b64 %0, -1, 0" : "=s"(m) : "s"(__builtin_amdgcn_readfirstlane(x)) : "scc");
    return m;
  };
  // issue the loads of the next row into stage buffer `buf`; past the last row of
  // the walk the bases stop and the last row is loaded again (never used)
  int rows_issued = 0, row_end = nrows;
  auto issue_row = [&](int buf) {
    const uint32_t st = (uint32_t)(uintptr_t)(TRI_L3 unsigned char*)(tri_smem + buf * STAGE);
    const int64_t advance = ones_while_positive(row_end - 1 - rows_issued);
    ++rows_issued;
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const uint32_t dst = __builtin_amdgcn_readfirstlane(st + (uint32_t)item_lds[x]);
      if (x < XW) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(item_voff[x]), "s"(item_base[base_of(x)]) : "memory", "m0");
      else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(dst), "v"(item_voff[x]), "s"(item_base[base_of(x)]) : "memory", "m0");
    }
#pragma unroll
    for (int x = 0; x < NBASE; ++x) item_base[x] += advance & item_step[x];
  };
  // the same, one item at a time (for loops that deal the loads of a row between other work);
  // next_row_advance() once per row, before its items
  auto next_row_advance = [&]() __attribute__((always_inline)) -> int64_t {
#if defined(TRI_DB_TIMING) && TRI_DB_TIMING_LOADS == 2
    const int64_t advance = ones_while_positive(0);
#else
    const int64_t advance = ones_while_positive(row_end - 1 - rows_issued);
#endif
    ++rows_issued;
    return advance;
  };
  auto issue_item = [&](int stage_off, auto x_tag, int64_t advance) __attribute__((always_inline)) {
    constexpr int x = decltype(x_tag)::value;
    const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(TRI_L3 unsigned char*)(tri_smem + stage_off) + (uint32_t)item_lds[x]);
    constexpr int bx = base_of(x);
    if constexpr (x < XW) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(item_voff[x]), "s"(item_base[bx]) : "memory", "m0");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(dst), "v"(item_voff[x]), "s"(item_base[bx]) : "memory", "m0");
    if constexpr (x + 1 == XN || base_of(x + 1) != bx) item_base[bx] += advance & item_step[bx];
  };
  // wait until at most the newest `K` rows of this wave's loads are in flight and
  // every LDS read has returned, then meet the other waves
  auto sync_rows = [&](auto k_tag) {
    constexpr int K = decltype(k_tag)::value * XN;
    static_assert(K <= 63, "vmcnt has 6 bits");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(K) : "memory");
  };

  // lane-constant LDS offsets: K, V rows as A operands (tile row m stands for key
  // perm32(m)); Q, dO rows as B operands (the lane's own query)
  OperandOffsets<T, D> ofk, ofq;
  ofk.init(perm32(jl), lane);
  ofq.init(jl, lane);
  // the wave's own tiles inside the workgroup's rows: folded into the offsets once
  ofk.shift(wk * WK * 32 * ROWB);
  ofq.shift(wj * WJ * 32 * ROWB);
  // (absolute LDS addresses from here on: the block's address is folded in once)
  ofk.make_absolute(tri_smem);
  ofq.make_absolute(tri_smem);
  ofk.pin();
  ofq.pin();
  // this lane's query in the lse / delta words, as an absolute LDS address (both halves of
  // the wave read the word of their query: lanes 32..63 zero it where it becomes a rank-1
  // operand, and use it as it is where -lse enters as a per-lane term of the exponent)
  int scalar_off = ((wj * WJ) * 32 + jl) * 4 + (int)(uintptr_t)(TRI_L3 const unsigned char*)tri_smem;
  asm volatile("" : "+v"(scalar_off));
  // LDS reads take a 16-bit immediate offset: for ring buffers past the first 64 KiB a
  // second set of lane offsets, moved up by two stages, keeps the buffer's offset an
  // immediate (the reads of those buffers would otherwise each need an address add).  The
  // pipelined walk of 128-byte rows has no registers for a second set: its offsets move from row to row.
  constexpr int kHighFrom = 2;
  constexpr bool kMoving = kPipelined && D > 32;
  constexpr bool kHighSet = NBUF > 2 && !kMoving;
  constexpr int HIGH = kHighSet ? kHighFrom * STAGE : 0;
  OperandOffsets<T, D> ofk_hi = ofk, ofq_hi = ofq;
  int scalar_off_hi = scalar_off;
  if constexpr (kHighSet) {
    ofk_hi.shift(HIGH);
    ofq_hi.shift(HIGH);
    ofk_hi.pin();
    ofq_hi.pin();
    scalar_off_hi += HIGH;
    asm volatile("" : "+v"(scalar_off_hi));
  }
  const frag ones = resident_ones<T>();
  // -lse per query and the key mask share one MFMA (see OffsetMask), -delta has its own
  typename OffsetMask<T>::Queries lrank[WJ];
  Rank1<T> drank[WJ];
  typename OffsetMask<T>::Keys kop;
  // (set up by the loops that use them: the walk has no registers for values that wait for the general loop)
  auto init_operands = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) { lrank[tj].init(0u, g); drank[tj].init(); }
    kop.init(perm32(jl), g);
  };

  const float c = a.c;
  // (an integer that the compiler cannot see through: a boolean would be kept as a lane mask
  // and negated with vector instructions in every row)
  int wave_live = __builtin_amdgcn_readfirstlane((int)(j_wave < N && k_wave < N));
  asm volatile("" : "+s"(wave_live));

  // The row's flag and the keep words of the wave's key tiles are the same for every lane:
  // they are read from global memory with scalar loads, one row ahead of their use (rows
  // past the end of the chunk repeat the last one and are not used).
  struct RowMeta {
    uint32_t flag;
    uint32_t keep[WK];
  };
  typedef const __attribute__((address_space(4))) uint32_t* const_words;
  const int64_t keep_step = uniform64((int64_t)a.nwords * 4);
  const_words flag_word = (const_words)(uintptr_t)(a.rowflag + (int64_t)b * N + i_begin);
  // (a key tile past the last word of the row has no attended key: its word is never read)
  const_words keep_word = (const_words)(uintptr_t)(a.keep + ((int64_t)b * N + i_begin) * a.nwords + min(k_wave / 32, a.nwords - 1));
  int word_at[WK];         // offset of tile tk's word from keep_word (clamped to the row)
  uint32_t word_mask[WK];  // zero for a tile past the last word
#pragma unroll
  for (int tk = 0; tk < WK; ++tk) {
    word_at[tk] = __builtin_amdgcn_readfirstlane(min(k_wave / 32 + tk, a.nwords - 1) - min(k_wave / 32, a.nwords - 1));
    word_mask[tk] = __builtin_amdgcn_readfirstlane(k_wave / 32 + tk < a.nwords ? 0xffffffffu : 0u);
  }
  int meta_rows = 0;
  // the words of the next row (the first call gives those of row 0)
  auto load_meta = [&]() -> RowMeta {
    RowMeta m;
    m.flag = *flag_word;
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) m.keep[tk] = keep_word[word_at[tk]] & word_mask[tk];
    const int64_t advance = ones_while_positive(row_end - 1 - meta_rows);
    ++meta_rows;
    flag_word = (const_words)((uintptr_t)flag_word + (uintptr_t)(advance & 4));
    keep_word = (const_words)((uintptr_t)keep_word + (uintptr_t)(advance & keep_step));
    return m;
  };

  auto compute_row = [&](int buf, const RowMeta& meta, const f32x16 (&biasr)[WJ][WK]) __attribute__((always_inline)) {
    const bool high = kHighSet && buf >= kHighFrom;  // (a constant once the ring loop is unrolled)
    const int sl = buf * STAGE - (high ? HIGH : 0);  // offset of the buffer for reads through the lane offsets
    const OperandOffsets<T, D>& oq = high ? ofq_hi : ofq;
    const OperandOffsets<T, D>& ok = high ? ofk_hi : ofk;
    const int soff = high ? scalar_off_hi : scalar_off;
    // (wave-uniform values are pinned to scalar registers so that the branches on
    // them are real branches and not lane masks)
    const bool flagged = meta.flag != 0;
    frag qf[WJ][DS], dof[WJ][DS], kf[WK][DS], vf[WK][DS];
    frag lf[WJ], df[WJ];  // per-query terms -lse*sqrt(d) and -delta as rank-1 MFMA operands
    float nl2[WJ];         // -lse of this lane's query in the exponent's unit
    uint32_t lw[WJ], dw[WJ];
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) {
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        qf[tj][s] = oq.natural_at(sl + OFF_Q + tj * 32 * ROWB, s);
        dof[tj][s] = oq.natural_at(sl + OFF_DO + tj * 32 * ROWB, s);
      }
      lw[tj] = *reinterpret_cast<TRI_L3 const uint32_t*>((uintptr_t)(uint32_t)(sl + OFF_LSE + tj * 128 + soff));
      dw[tj] = *reinterpret_cast<TRI_L3 const uint32_t*>((uintptr_t)(uint32_t)(sl + OFF_DELTA + tj * 128 + soff));
    }
#pragma unroll
    for (int tk = 0; tk < WK; ++tk)
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        kf[tk][s] = ok.natural_at(sl + OFF_K + tk * 32 * ROWB, s);
        vf[tk][s] = ok.natural_at(sl + OFF_V + tk * 32 * ROWB, s);
      }
    // every LDS read of the row is issued before the first branch on the row's keep words
    // (read where they are used, they would return in several waited-for batches)
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) {
#pragma unroll
      for (int s = 0; s < DS; ++s) asm volatile("" : "+v"(qf[tj][s]), "+v"(dof[tj][s]));
      asm volatile("" : "+v"(lw[tj]), "+v"(dw[tj]));
    }
#pragma unroll
    for (int tk = 0; tk < WK; ++tk)
#pragma unroll
      for (int s = 0; s < DS; ++s) asm volatile("" : "+v"(kf[tk][s]), "+v"(vf[tk][s]));
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) {
      lrank[tj].set_raw(g ? 0u : lw[tj]);
      lf[tj] = lrank[tj].get();
      df[tj] = drank[tj].set(g ? 0u : dw[tj]);
      nl2[tj] = split_value<T>(lw[tj]) * c;
    }
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) {
      const uint32_t keepw = meta.keep[tk];
      if (keepw == 0) continue;  // no attended key in this tile: dS = 0
#pragma unroll
      for (int tj = 0; tj < WJ; ++tj) {
        f32x16 s;
        float addend = 0.f;
        // Each case ends in the MFMA that defines s from the bias tile in place (a
        // select between accumulator inits would copy 16 registers).
        if (!flagged) {
          if (keepw == 0xffffffffu) {
            // no masked key in the tile: a lane owns one query, so -lse is one number per
            // lane and rides on the multiply of the exponent (an fma) instead of an MFMA
            s = E::mfma(kf[tk][0], qf[tj][0], biasr[tj][tk]);
#pragma unroll
            for (int sd = 1; sd < DS; ++sd) s = E::mfma(kf[tk][sd], qf[tj][sd], s);
            addend = nl2[tj];
          } else {
            s = E::mfma(kop.masked_copy(keepw), lf[tj], biasr[tj][tk]);  // masked keys: large negative score
#pragma unroll
            for (int sd = 0; sd < DS; ++sd) s = E::mfma(kf[tk][sd], qf[tj][sd], s);
          }
        } else {
          // rare: a fully masked row ignores q.k and the bias
          asm volatile("" ::);
          s = E::mfma(kop.masked_copy(keepw), lf[tj], zero16());
        }
        f32x16 dp = E::mfma(ones, df[tj], zero16());
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) dp = E::mfma(vf[tk][sd], dof[tj][sd], dp);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float p = fast_exp2(__builtin_fmaf(s[v], c, addend));
          dbacc[tj][tk][v] = __builtin_fmaf(p, dp[v], dbacc[tj][tk][v]);
        }
      }
    }
  };

  // a row of the trailing run of fully masked ones (see below): dO V^T - delta on top of the accumulator itself
  auto add_uniform_row = [&](int buf) __attribute__((always_inline)) {
    const bool high = kHighSet && buf >= kHighFrom;
    const int sl = buf * STAGE - (high ? HIGH : 0);
    const OperandOffsets<T, D>& oq = high ? ofq_hi : ofq;
    const OperandOffsets<T, D>& ok = high ? ofk_hi : ofk;
    const int soff = high ? scalar_off_hi : scalar_off;
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) {
      const uint32_t dw = *reinterpret_cast<TRI_L3 const uint32_t*>((uintptr_t)(uint32_t)(sl + OFF_DELTA + tj * 128 + soff));
      const frag df = drank[tj].set(g ? 0u : dw);
#pragma unroll
      for (int tk = 0; tk < WK; ++tk) {
        dbacc[tj][tk] = E::mfma(ones, df, dbacc[tj][tk]);
#pragma unroll
        for (int sd = 0; sd < DS; ++sd)
          dbacc[tj][tk] = E::mfma(ok.natural_at(sl + OFF_V + tk * 32 * ROWB, sd), oq.natural_at(sl + OFF_DO + tj * 32 * ROWB, sd), dbacc[tj][tk]);
      }
    }
  };
  // move the loads and the row words to row `row`, with nothing in flight, for a walk up to row `end`
  auto seek = [&](int row, int end) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const int last = max(row_end - 1, 0), at = min(rows_issued, last), meta_at = min(meta_rows, last);
#pragma unroll
    for (int x = 0; x < NBASE; ++x) item_base[x] += (int64_t)(row - at) * item_step[x];
    flag_word = (const_words)((uintptr_t)flag_word + (uintptr_t)((int64_t)(row - meta_at) * 4));
    keep_word = (const_words)((uintptr_t)keep_word + (uintptr_t)((int64_t)(row - meta_at) * keep_step));
    rows_issued = meta_rows = row;
    row_end = end;
  };

  // the rows from `first_row` to row_end (the loads and the row words stand at the first)
  auto walk_rows = [&](int first_row, auto uniform_tag) __attribute__((always_inline)) {
  constexpr bool UNIFORM = decltype(uniform_tag)::value;
  init_operands();
  f32x16 biasr[WJ][WK];
  if constexpr (!UNIFORM) {
    load_bias(biasr, std::integral_constant<int, 2>{});
    wait_dma_known();  // (or the first use in every row would wait for everything in flight)
  }
  if constexpr (NBUF >= 2) {
    // Ring of NBUF row buffers: the loads run NBUF-1 rows ahead of the compute, which
    // hides the memory latency behind several rows of work.  Row q lives in buffer
    // q % NBUF; the buffer that row q + NBUF - 1 goes to was last read for row q - 1,
    // which every wave finished before the barrier that ended that row.
    constexpr int P = NBUF - 1;
#pragma unroll
    for (int u = 0; u < P; ++u) issue_row(u);
    RowMeta meta = load_meta();
    sync_rows(std::integral_constant<int, P - 1>{});  // row 0 has landed
    for (int r = first_row; r < row_end; r += NBUF) {
#pragma unroll
      for (int u = 0; u < NBUF; ++u) {
        if (r + u < row_end) {
          issue_row((u + P) % NBUF);
          const RowMeta next = load_meta();
          if (wave_live != 0) {
            if constexpr (UNIFORM) add_uniform_row(u);
            else compute_row(u, meta, biasr);
          }
          sync_rows(std::integral_constant<int, P - 1>{});  // the next row has landed
          meta = next;
        }
      }
    }
  } else {
    // one stage only (two do not fit in LDS): load, then compute
    for (int ir = first_row; ir < row_end; ++ir) {
      issue_row(0);
      const RowMeta meta = load_meta();
      sync_rows(std::integral_constant<int, 0>{});
      if (wave_live != 0) {
        if constexpr (UNIFORM) add_uniform_row(0);
        else compute_row(0, meta, biasr);
      }
      sync_rows(std::integral_constant<int, 0>{});
    }
  }
  };
  // Waves that own two key tiles (16-bit types, d <= 64) walk the rows in front of the chunk's first
  // fully masked one software-pipelined: a wave's matrix instructions of one tile are issued
  // between the exponentials and multiply-adds of the tile before it (the second tile of a row
  // overlaps the first, the first tile of the next row overlaps the second), so neither pipe
  // waits for the other although only one or two waves share a SIMD.  The score chain of a tile
  // runs before its dP chain, and every operand is read from LDS into the register that the
  // product before it has freed, several products ahead of its use: V where K was, the next tile's K
  // where V was, the next row's Q and dO where this row's were.  (Two sets of operands took 243 registers
  // at d = 32 and left none for a mask; d = 64 does not fit two.)  -lse is the addend of the
  // exponent's fma in every row; where rows have masked keys in this block each tile takes one more
  // product, which adds the mask element to the scores of the masked keys (keys operand against ones), and leaves
  // out tiles without an attended key (see phase).
  // Alone, back to back on one card against the walk with two operand sets, which took unmasked rows of up to
  // 64 bytes only: h = 4, d = 32 n = 1024 0.96 -> 0.91 ms; 2048 with 5 % masked 9.6 (16 waves: 8.9) -> 8.5;
  // h = 8, d = 64 n = 768 1.80 -> 1.53, half of the keys masked 1.84 -> 1.60, with pair rows 98 KiB apart 1.85 ->
  // 1.78.  (Within a training step the large ones gain little of it: the chip then lowers its clock, 2.0 GHz at
  // n = 1024.)  With its loads taken out the d = 64 walk takes 1.10 ms: two row buffers of 64 KiB are
  // all that fits, and a compute unit takes in 64 bytes per clock.
  // The trailing fully masked rows come first: with P = 1 / n everywhere their part is
  // sum_i (dO_i V_i^T - delta_i) / n, matrix products into the accumulator and one multiply at the
  // end instead of an exponential and two multiply-adds per element and row (n = 1000 with 800 valid
  // rows, h = 4, d = 32: 1006 -> 930 us).
  if (tail_end > tail_begin) {
    seek(tail_begin - i_begin, tail_end - i_begin);
    walk_rows(tail_begin - i_begin, std::true_type{});
    const float inv = 1.0f / (float)N;
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj)
#pragma unroll
      for (int tk = 0; tk < WK; ++tk)
#pragma unroll
        for (int v = 0; v < 16; ++v) dbacc[tj][tk][v] *= inv;
    seek(0, nrows);
  }
  if constexpr (kPipelined) {
    if (nwalk < 2 * NBUF) nwalk = 0;  // too few to fill the pipeline
    static_assert(BKB / 32 <= 8, "eight key tiles per field of the block's words");
    const uint32_t wave_tiles = __builtin_amdgcn_readfirstlane(block_tiles >> (wk * WK));
    // masked_tag: 0 every key is attended, 1 some are masked, 2 some tile of the wave has no attended key in some row
    auto walk = [&](auto masked_tag, auto busy_tag) __attribute__((always_inline)) {
      constexpr bool MASKED = decltype(masked_tag)::value != 0, DEAD = decltype(masked_tag)::value == 2;
      // (a wave without queries or attended keys takes part in the loads and barriers only)
      constexpr bool BUSY = decltype(busy_tag)::value;
      typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
      f32x16 biasr[WJ][WK];
      if constexpr (BUSY) {
        load_bias(biasr, masked_tag);
        wait_dma_known();
      }
      // the tile in flight and the tile being consumed: scores and dP
      f32x16 sc[2], dpc[2];
      // Operands of the tile whose matrix instructions run: its K, then, step by step as the score chain has
      // used them, its V in the same registers; Q and dO of the row; -delta of the lane's query as a
      // rank-1 operand, -lse in the exponent's unit.
      frag kv[DS], qf[DS], dof[DS], df;
      float nl2, nl2_next;
      uint32_t lw, dw;
      drank[0].init();
      // the keep words of the wave's two key tiles (this lane's key is bit perm32(jl))
      uint32_t kw[WK] = {}, kw_next[WK] = {}, past[WK] = {};
      const uint32_t key_bit = 1u << perm32(jl);
      int keep_off = wk * WK * 4 + (int)(uintptr_t)(TRI_L3 const unsigned char*)tri_smem, keep_off_hi = keep_off + HIGH;
      if constexpr (MASKED) {
        asm volatile("" : "+v"(keep_off), "+v"(keep_off_hi));
#pragma unroll
        for (int tk = 0; tk < WK; ++tk) past[tk] = __builtin_amdgcn_readfirstlane(past_end(k_wave / 32 + tk));
      }
      // (kMoving: the lane offsets stand at the buffer that is read)
      auto step_stages = [&](int bytes) __attribute__((always_inline)) {
        ofk.shift(bytes);
        ofq.shift(bytes);
        ofk.pin();
        ofq.pin();
        scalar_off += bytes;
        keep_off += bytes;
        asm volatile("" : "+v"(scalar_off), "+v"(keep_off));
      };
      // operand `sd` of the rows at `off` in row buffer `buf`
      auto read_keys = [&](int buf, int off, int sd) __attribute__((always_inline)) {
        const bool high = kHighSet && buf >= kHighFrom;
        return (high ? ofk_hi : ofk).natural_at((kMoving ? 0 : buf * STAGE) - (high ? HIGH : 0) + off, sd);
      };
      auto read_queries = [&](int buf, int off, int sd) __attribute__((always_inline)) {
        const bool high = kHighSet && buf >= kHighFrom;
        return (high ? ofq_hi : ofq).natural_at((kMoving ? 0 : buf * STAGE) - (high ? HIGH : 0) + off, sd);
      };
      auto read_words = [&](int buf) __attribute__((always_inline)) {
        const bool high = kHighSet && buf >= kHighFrom;
        const int at = (kMoving ? 0 : buf * STAGE) - (high ? HIGH : 0);
        const int words = at + (high ? scalar_off_hi : scalar_off), keeps = at + (high ? keep_off_hi : keep_off) + OFF_KW;
        lw = *reinterpret_cast<TRI_L3 const uint32_t*>((uintptr_t)(uint32_t)(words + OFF_LSE));
        dw = *reinterpret_cast<TRI_L3 const uint32_t*>((uintptr_t)(uint32_t)(words + OFF_DELTA));
        if constexpr (MASKED) {
#pragma unroll
          for (int tk = 0; tk < WK; ++tk) kw_next[tk] = *reinterpret_cast<TRI_L3 const uint32_t*>((uintptr_t)(uint32_t)(keeps + 4 * tk));
        }
      };
      auto mask_operand = [&](uint32_t keepw, int tk) __attribute__((always_inline)) {
        u32x4v t = {0u, ((keepw | past[tk]) & key_bit) ? 0u : OffsetMask<T>::mask_dword(), 0u, 0u};
        return __builtin_bit_cast(frag, t);
      };
      constexpr int M = MASKED ? 1 : 0;
      constexpr int NM = 2 * DS + 1 + M;  // matrix instructions of a tile
      // the elements of the tile before that are dealt to slot X: [dealt(X), dealt(X + 1))
      auto dealt = [](int X) constexpr { return 16 * X / NM; };
      // The matrix instructions of key tile TN (scores from the bias tile, dP from -delta) go into sn / dpn, dealt
      // between the elementwise work of the tile before it, whose scores s and dP are complete: db +=
      // exp2(c s - lse) dP.  `cur`, `next`: row buffers of the tile and of the tile after it; `turn` comes
      // between the two chains.
      auto phase = [&](auto tn_tag, int cur, int next, uint32_t keepw, uint32_t attended, f32x16& sn, f32x16& dpn, f32x16& s, f32x16& dp,
                       float addend, auto&& turn, auto&& between) __attribute__((always_inline)) {
        constexpr int TN = decltype(tn_tag)::value, TC = 1 - TN;
        // A tile without an attended key (`attended`: the keep word of the tile before) adds nothing: dS = 0 whatever its K and V
        // rows and its bias hold.  Where they are infinite or NaN, as padding may be, zero probabilities
        // times their dP are not zero.  Its elementwise work is skipped, a branch per step, in a loop of its own for waves
        // with such a tile (n = 1024, d = 32, four parts that attend to themselves with all rows walked: 0.81 ms, 1.19 done on
        // zeros; with the branches in every masked loop n = 2048 with 5 % masked 8.24 -> 8.5 ms from a cool chip).  In rows of
        // 128 bytes a second masked loop leaves the compiler spilling in the first: there the work is done on zeros, one
        // branch per tile in the one loop (n = 768, h = 8 with half of the keys masked: 1.61 ms, as without it).
        uint32_t adds = 1u;
        if constexpr (DEAD) adds = __builtin_amdgcn_readfirstlane(attended);
        if constexpr (DEAD && kMoving) {
          if (adds == 0) {
            asm volatile("" ::);
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = dp[v] = 0.f;
            addend = 0.f;
          }
        }
        frag mk;
        if constexpr (MASKED) mk = mask_operand(keepw, TN);
        static_for<NM>([&](auto xc) __attribute__((always_inline)) {
          constexpr int X = decltype(xc)::value;
          if constexpr (X < M) {
            sn = E::mfma(mk, ones, biasr[0][TN]);
          } else if constexpr (X < M + DS) {
            constexpr int sd = X - M;
            sn = E::mfma(kv[sd], qf[sd], X == 0 ? biasr[0][TN] : sn);
            kv[sd] = read_keys(cur, OFF_V + TN * 32 * ROWB, sd);
            if constexpr (TN == 0) dof[sd] = read_queries(cur, OFF_DO, sd);
          } else if constexpr (X == M + DS) {
            dpn = E::mfma(ones, df, zero16());
          } else {
            constexpr int sd = X - M - DS - 1;
            dpn = E::mfma(kv[sd], dof[sd], dpn);
            kv[sd] = read_keys(next, OFF_K + TC * 32 * ROWB, sd);
            if constexpr (TN == 1) {
              qf[sd] = read_queries(next, OFF_Q, sd);
              if constexpr (sd == 0) read_words(next);
            }
          }
          between(std::integral_constant<int, X>{});
          auto add = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int v = dealt(X); v < dealt(X + 1); ++v) {
              const float p = fast_exp2(__builtin_fmaf(s[v], c, addend));
              dbacc[0][TC][v] = __builtin_fmaf(p, dp[v], dbacc[0][TC][v]);
            }
          };
          if constexpr (!DEAD || kMoving) add();
          else if (adds != 0) add();
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (X == M + DS) {
            turn();
            __builtin_amdgcn_sched_barrier(0);
          }
        });
      };
      auto take_words = [&]() __attribute__((always_inline)) {
        nl2_next = split_value<T>(lw) * c;
        df = drank[0].set(g ? 0u : dw);
      };
#pragma unroll
      for (int u = 0; u < NBUF; ++u) issue_row(u);
      sync_rows(std::integral_constant<int, NBUF - 1>{});  // row 0 has landed
      if constexpr (BUSY) {
        // the first tile of the first row has nothing to overlap with
        read_words(0);
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) {
          qf[sd] = read_queries(0, OFF_Q, sd);
          dof[sd] = read_queries(0, OFF_DO, sd);
          kv[sd] = read_keys(0, OFF_K, sd);
        }
        take_words();
        nl2 = nl2_next;
#pragma unroll
        for (int tk = 0; tk < WK; ++tk) kw[tk] = kw_next[tk];
        sc[0] = biasr[0][0];
        if constexpr (MASKED) sc[0] = E::mfma(mask_operand(kw[0], 0), ones, sc[0]);
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) {
          sc[0] = E::mfma(kv[sd], qf[sd], sc[0]);
          kv[sd] = read_keys(0, OFF_V, sd);
        }
        dpc[0] = E::mfma(ones, df, zero16());
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) {
          dpc[0] = E::mfma(kv[sd], dof[sd], dpc[0]);
          kv[sd] = read_keys(0, OFF_K + 32 * ROWB, sd);
        }
      }
#ifdef TRI_DB_TIMING
      uint64_t t_wait = 0, t_barrier = 0;
      const uint64_t t_clk0 = __builtin_amdgcn_s_memtime(), t_real0 = __builtin_amdgcn_s_memrealtime();
#endif
      // Row r, in buffer `cur` (offset stage_off): its second tile beside the elementwise work of its first, and the
      // first tile of the next row beside that of its second.  Between the two chains of the second
      // tile every wave is done with the row's buffer (V of that tile was the last it had to read): the
      // next row's rows have landed there, and the loads of row r + NBUF go into the buffer, dealt
      // over the slots up to the end of the row (a burst of them would hold up the wave's other
      // instructions until the memory pipeline has taken them all).
      constexpr int kEarly = 2;
      auto row = [&](int stage_off, int cur, int next, int step) __attribute__((always_inline)) {
        const int64_t advance = next_row_advance();
        auto deal_loads = [&](auto slot_tag) __attribute__((always_inline)) {
          constexpr int slot = decltype(slot_tag)::value;  // 0 .. DS - 1: rest of the second tile; then the first tile
          static_for<XN>([&](auto xt) __attribute__((always_inline)) {
            constexpr int x = decltype(xt)::value;
#if !defined(TRI_DB_TIMING) || TRI_DB_TIMING_LOADS != 0
            if constexpr (slot == (x * (NBUF == 2 ? kEarly : DS + NM)) / XN) issue_item(stage_off, xt, advance);
#endif
          });
        };
        auto turn = [&]() __attribute__((always_inline)) {
#ifdef TRI_DB_TIMING
          const uint64_t m0 = __builtin_amdgcn_s_memtime();
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"((NBUF - 2) * XN) : "memory");
          const uint64_t m1 = __builtin_amdgcn_s_memtime();
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          const uint64_t m2 = __builtin_amdgcn_s_memtime();
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          t_wait += m1 - m0;
          t_barrier += m2 - m1;
#else
          sync_rows(std::integral_constant<int, NBUF - 2>{});
#endif
          if constexpr (kMoving && BUSY) step_stages(step);
        };
        if constexpr (BUSY) {
          // (used and defined in every row: the compiler's allocator otherwise parks what the loop only reads in
          // scratch memory, with registers to spare, and a reload from there waits for every load in flight)
          asm volatile("" : "+v"(biasr[0][0]), "+v"(biasr[0][1]));
          phase(std::integral_constant<int, 1>{}, cur, next, kw[1], kw[0], sc[1], dpc[1], sc[0], dpc[0], nl2, turn, [&](auto slot) __attribute__((always_inline)) {
            constexpr int after = decltype(slot)::value - (M + DS + 1);
            if constexpr (after >= 0) deal_loads(std::integral_constant<int, after>{});
          });
          take_words();
          phase(std::integral_constant<int, 0>{}, next, next, kw_next[0], kw[1], sc[0], dpc[0], sc[1], dpc[1], nl2, [] {}, [&](auto slot) __attribute__((always_inline)) {
            deal_loads(std::integral_constant<int, DS + decltype(slot)::value>{});
          });
          nl2 = nl2_next;
          kw[0] = kw_next[0];
          kw[1] = kw_next[1];
        } else {
          turn();
          static_for<DS + NM>(deal_loads);
        }
      };
      if constexpr (kMoving) {
        int at = 0;  // offset of row r's buffer
#pragma unroll 1
        for (int r = 0; r < nwalk; ++r) {
          const int step = at == (NBUF - 1) * STAGE ? -(NBUF - 1) * STAGE : STAGE;
          row(at, 0, 0, step);
          at += step;
        }
        if constexpr (BUSY) step_stages(-at);  // (back to the first buffer)
      } else {
        for (int r = 0; r < nwalk; r += NBUF) {
          static_for<NBUF>([&](auto uc) __attribute__((always_inline)) {
            constexpr int u = decltype(uc)::value;
            if (r + u < nwalk) row(u * STAGE, u, (u + 1) % NBUF, 0);
          });
        }
      }
#ifdef TRI_DB_TIMING
      {
        const uint64_t t_clk1 = __builtin_amdgcn_s_memtime(), t_real1 = __builtin_amdgcn_s_memrealtime();
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        // (the sums are not stored here, and without a use the compiler leaves their arithmetic out)
#pragma unroll
        for (int tk = 0; tk < WK; ++tk)
#pragma unroll
          for (int v = 0; v < 16; ++v) asm volatile("" : : "v"(dbacc[0][tk][v]));
        if (lane == 0) {
          const int64_t L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
          uint64_t* rec = reinterpret_cast<uint64_t*>(a.db) + (L * NW + wave) * 4;
          rec[0] = t_clk1 - t_clk0;
          rec[1] = t_wait;
          rec[2] = t_barrier;
          rec[3] = t_real1 - t_real0;
        }
        return;
      }
#endif
    };
    if (nwalk > 0) {
      constexpr uint32_t kMine = (1u << WK) - 1;
      const bool busy = wave_live != 0 && (wave_tiles & kMine) != 0, masked = (block_tiles & 0xff00u) != 0;
      const bool dead = kMoving || (wave_tiles >> 16 & kMine) != 0;
      if (!busy) walk(std::integral_constant<int, 0>{}, std::false_type{});
      else if (!masked) walk(std::integral_constant<int, 0>{}, std::true_type{});
      else if (dead) walk(std::integral_constant<int, 2>{}, std::true_type{});
      else if constexpr (!kMoving) walk(std::integral_constant<int, 1>{}, std::true_type{});
#ifdef TRI_DB_TIMING
      return;
#endif
      if (nwalk < row_end) {
        // hand over: nothing in flight, the loads and the row words moved to row nwalk
        seek(nwalk, row_end);
      }
    }
    if (nwalk < row_end) walk_rows(nwalk, std::false_type{});
  } else if (row_end > 0) {
    walk_rows(0, std::false_type{});
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the spare rows loaded past the end
  if (wave_live == 0) return;

  store_db<T, WJ, WK>(a, dbacc, bh, chunk, j_wave, k_wave, jl, g);
}

// The same for fp32, whose rows pass through registers on their way to LDS, where they lie as
// three bf16 parts (see SplitStream): the next row is loaded before the current one is computed
// and written after it, into the other buffer where two fit.  What bounds it is the 24 matrix
// instructions per tile and row (d = 32: 768 clocks, half of the kernel) and the splitting beside
// them, which a larger block pays for fewer rows per tile: at n = 512, h = 4 0.51 ms with 128 x 128
// and one buffer, 0.60 with 64 x 128 and two (0.78 through the fp32 matrix pipe); at n = 250 0.16
// and 0.11, where the larger blocks are too few.
template <int D, int GJ, int GK, int WJ, int WK, int NBUF>
__global__ __launch_bounds__(GJ * GK * 64) void tri_bwd_b_split_kernel(const BwdArgs a) {
  using T = float;
  using E = Elem<float>;
  using frag = E::frag;
  using Off = OperandOffsets<float, D>;
  constexpr int DS = Off::DS, NW = GJ * GK;
  constexpr int BJ = GJ * WJ * 32, BKB = GK * WK * 32;
  constexpr int ROWB = lds_row_bytes(D, 4);
  // The widest rows leave LDS room for two of the four tensors at a time: Q, K, then dO, V.
  constexpr bool PHASED = D > 64;
  static_assert(!PHASED || (NBUF == 1 && WJ * WK == 1), "one tile per wave and one buffer");
  constexpr int OFF_Q = 0, OFF_K = OFF_Q + BJ * ROWB, OFF_DO = PHASED ? OFF_Q : OFF_K + BKB * ROWB, OFF_V = OFF_DO + BJ * ROWB;
  constexpr int STAGE = OFF_V + BKB * ROWB;
  static_assert(STAGE == bwd_b_split_stage_bytes(BJ, BKB, D), "the launcher sizes LDS with bwd_b_split_stage_bytes");
  extern __shared__ __attribute__((aligned(16))) unsigned char tri_smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int jl = lane & 31, g = lane >> 5;
  const int N = a.N;
  const DbBlock blk = db_block(a, BJ, BKB);
  if (!blk.live) return;
  const int bh = blk.bh, b = bh / a.H, h = bh % a.H;
  const int wj = wave % GJ, wk = wave / GJ;
  const int j_wave = blk.j + wj * (WJ * 32), k_wave = blk.k + wk * (WK * 32);
  const int i_begin = blk.chunk * a.rows_per_chunk;
  const int i_end = min(N, i_begin + a.rows_per_chunk);
  const bool wave_live = j_wave < N && k_wave < N;

  const T* qbase = reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h;
  const T* kbase = reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h;
  const T* vbase = reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h;
  const T* dobase = reinterpret_cast<const T*>(a.dout) + b * a.sdo.b + h * a.sdo.h;
  const T* pack_bh = reinterpret_cast<const T*>(a.packq) + (int64_t)bh * a.NP * a.NP * 1024;

  f32x16 biasr[WJ][WK], dbacc[WJ][WK];
#pragma unroll
  for (int tj = 0; tj < WJ; ++tj)
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) {
      biasr[tj][tk] = bias_tile<T>(pack_bh, a.NP, min((j_wave >> 5) + tj, a.NP - 1), min((k_wave >> 5) + tk, a.NP - 1), lane, a.sqrt_d, 0.f);
      dbacc[tj][tk] = zero16();
    }

  // queries and keys past the end repeat the last one (they feed db entries that are never stored)
  SplitStream<D, BJ, NW> qs, dos;
  SplitStream<D, BKB, NW> ks, vs;
  qs.init([&](int r) { return qbase + (int64_t)min(blk.j + r, N - 1) * a.sq.j; }, wave, lane);
  dos.init([&](int r) { return dobase + (int64_t)min(blk.j + r, N - 1) * a.sdo.j; }, wave, lane);
  ks.init([&](int r) { return kbase + (int64_t)min(blk.k + r, N - 1) * a.sk.j; }, wave, lane);
  vs.init([&](int r) { return vbase + (int64_t)min(blk.k + r, N - 1) * a.sv.j; }, wave, lane);
  // the per-query words of this lane's queries travel in registers
  float lw[WJ], dw[WJ], lw_next[WJ], dw_next[WJ];
  const int64_t words = (int64_t)bh * N * N;
  auto load_words = [&](int i) {
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) {
      const int64_t at = words + (int64_t)i * N + min(j_wave + 32 * tj + jl, N - 1);
      lw_next[tj] = reinterpret_cast<const float*>(a.lse2)[at];
      dw_next[tj] = reinterpret_cast<const float*>(a.delta)[at];
    }
  };
  auto take_words = [&] {
#pragma unroll
    for (int tj = 0; tj < WJ; ++tj) {
      lw[tj] = lw_next[tj];
      dw[tj] = dw_next[tj];
    }
  };
  auto load_qk = [&](int i) { qs.load(i * a.sq.i); ks.load(i * a.sk.i); };
  auto load_dov = [&](int i) { dos.load(i * a.sdo.i); vs.load(i * a.sv.i); };
  auto store_qk = [&](unsigned char* st) { qs.store(st + OFF_Q); ks.store(st + OFF_K); };
  auto store_dov = [&](unsigned char* st) { dos.store(st + OFF_DO); vs.store(st + OFF_V); };

  Off ofk, ofq;
  ofk.init(perm32(jl), lane);
  ofq.init(jl, lane);
  ofk.shift(wk * WK * 32 * ROWB);
  ofq.shift(wj * WJ * 32 * ROWB);
  const E::ofrag ones = resident_ones<T>();
  typename OffsetMask<T>::Queries lrank;
  Rank1<T> drank;
  lrank.init(0u, g);
  drank.init();
  typename OffsetMask<T>::Keys kop;
  kop.init(perm32(jl), g);
  const float c = a.c;

  struct RowMeta {
    bool flagged;
    uint32_t keep[WK];
  };
  auto row_meta = [&](int i) {
    RowMeta m;
    m.flagged = uniform_word(a.rowflag, b * N + i) != 0;
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) {
      const int w = (k_wave >> 5) + tk;
      m.keep[tk] = w < a.nwords ? uniform_word(a.keep + ((int64_t)b * N + i) * a.nwords, w) : 0u;
    }
    return m;
  };
  // scores of tile (tj, tk), with -lse on the fma of the exponent (addend) or, where keys are
  // masked, in one product with the key mask, as in the kernel above
  auto scores = [&](const RowMeta& m, const unsigned char* st, int tj, int tk, const frag* qf, float& addend) __attribute__((always_inline)) -> f32x16 {
    const uint32_t keepw = m.keep[tk];
    const unsigned char* kt = st + OFF_K + tk * 32 * ROWB;
    f32x16 s;
    addend = 0.f;
    if (!m.flagged && keepw == 0xffffffffu) {
      s = E::mfma(ofk.natural(kt, 0), qf[0], biasr[tj][tk]);
#pragma unroll
      for (int sd = 1; sd < DS; ++sd) s = E::mfma(ofk.natural(kt, sd), qf[sd], s);
      addend = lw[tj] * c;
    } else {
      asm volatile("" ::);
      lrank.set_raw(g ? 0u : __builtin_bit_cast(uint32_t, lw[tj]));
      if (!m.flagged) {
        s = E::mfma(kop.masked_copy(keepw), lrank.get(), biasr[tj][tk]);
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) s = E::mfma(ofk.natural(kt, sd), qf[sd], s);
      } else {
        // a fully masked row ignores q.k and the bias
        s = E::mfma(kop.masked_copy(keepw), lrank.get(), zero16());
      }
    }
    return s;
  };
  // db += exp2(c s - lse) (dO V^T - delta)
  auto add_tile = [&](const unsigned char* st, int tj, int tk, const frag* dof, const f32x16& s, float addend) __attribute__((always_inline)) {
    const unsigned char* vt = st + OFF_V + tk * 32 * ROWB;
    f32x16 dp = E::mfma(ones, drank.set(g ? 0u : __builtin_bit_cast(uint32_t, dw[tj])), zero16());
#pragma unroll
    for (int sd = 0; sd < DS; ++sd) dp = E::mfma(ofk.natural(vt, sd), dof[sd], dp);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float p = fast_exp2(__builtin_fmaf(s[v], c, addend));
      dbacc[tj][tk][v] = __builtin_fmaf(p, dp[v], dbacc[tj][tk][v]);
    }
  };

  load_qk(i_begin);
  load_words(i_begin);
  if constexpr (PHASED) {
    unsigned char* st = tri_smem;
    store_qk(st);
    __syncthreads();
    for (int i = i_begin; i < i_end; ++i) {
      load_dov(i);
      take_words();
      const RowMeta m = row_meta(i);
      const bool on = wave_live && m.keep[0] != 0;
      f32x16 s = zero16();
      float addend = 0.f;
      if (on) {
        frag qf[DS];
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) qf[sd] = ofq.natural(st + OFF_Q, sd);
        s = scores(m, st, 0, 0, qf, addend);
      }
      __syncthreads();  // (every wave has read Q, K)
      store_dov(st);
      __syncthreads();
      if (i + 1 < i_end) {
        load_qk(i + 1);
        load_words(i + 1);
      }
      if (on) {
        frag dof[DS];
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) dof[sd] = ofq.natural(st + OFF_DO, sd);
        add_tile(st, 0, 0, dof, s, addend);
      }
      __syncthreads();
      if (i + 1 < i_end) store_qk(st);
      __syncthreads();
    }
  } else {
    load_dov(i_begin);
    store_qk(tri_smem);
    store_dov(tri_smem);
    __syncthreads();
    for (int i = i_begin; i < i_end; ++i) {
      const int buf = NBUF == 2 ? (i - i_begin) & 1 : 0;
      const unsigned char* st = tri_smem + buf * STAGE;
      take_words();
      if (i + 1 < i_end) {
        load_qk(i + 1);
        load_dov(i + 1);
        load_words(i + 1);
      }
      if (wave_live) {
        const RowMeta m = row_meta(i);
#pragma unroll
        for (int tj = 0; tj < WJ; ++tj) {
          frag qf[DS], dof[DS];
#pragma unroll
          for (int sd = 0; sd < DS; ++sd) {
            qf[sd] = ofq.natural(st + OFF_Q + tj * 32 * ROWB, sd);
            dof[sd] = ofq.natural(st + OFF_DO + tj * 32 * ROWB, sd);
          }
#pragma unroll
          for (int tk = 0; tk < WK; ++tk) {
            if (m.keep[tk] == 0) continue;  // no attended key in this tile: dS = 0
            float addend;
            const f32x16 s = scores(m, st, tj, tk, qf, addend);
            add_tile(st, tj, tk, dof, s, addend);
          }
        }
      }
      if (NBUF == 1) __syncthreads();  // (every wave has read the row)
      if (i + 1 < i_end) {
        unsigned char* next = tri_smem + (NBUF == 2 ? buf ^ 1 : 0) * STAGE;
        store_qk(next);
        store_dov(next);
      }
      __syncthreads();
    }
  }
  if (!wave_live) return;
  store_db<T, WJ, WK>(a, dbacc, bh, blk.chunk, j_wave, k_wave, jl, g);
  float check = 0.f;
#pragma unroll
  for (int tj = 0; tj < WJ; ++tj)
#pragma unroll
    for (int tk = 0; tk < WK; ++tk) check = finite_check<16>(dbacc[tj][tk], check);
  // (called or inlined: at d = 64, n = 500 1720 against 1740 us, at d = 32, n = 512 490 against 486, and 136
  // bytes of scratch less)
  if (__any(!(check == 0.f))) {
    if constexpr (D >= 64) plain_db<D, WJ * 32, WK * 32>(arg_words(), bh, blk.chunk, j_wave, k_wave, i_begin, i_end, fresh_lane());
    else plain_db_block<D, WJ * 32, WK * 32>(read_args<BwdArgs>(arg_words()), bh, blk.chunk, j_wave, k_wave, i_begin, i_end, fresh_lane());
  }
}

// db = sum over chunks of the fp32 partials, in chunk order.  The chunks' loads are in flight
// together (read one after the other, 16 chunks took 6.8 us at n = 64).  Where db's queries are
// contiguous (a transposed layout) a workgroup turns its 32 x 32 tile around in LDS.
template <typename T>
__global__ __launch_bounds__(256) void tri_bwd_b_reduce_kernel(const BwdArgs a, int64_t count) {
  const int N = a.N, tiles = (N + 31) / 32;
  const int tile = blockIdx.x % (tiles * tiles), bh = blockIdx.x / (tiles * tiles);
  const int j0 = tile / tiles * 32, k0 = tile % tiles * 32, tk = threadIdx.x & 31, tj = threadIdx.x >> 5;
  T* db = reinterpret_cast<T*>(a.db) + (bh / a.H) * a.sdb_b + (bh % a.H) * a.sdb_h;
  const bool turn = a.sdb_j == 1 && a.sdb_k != 1;
  __shared__ float turned[32][33];
  float acc[4];
  const float* p[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int j = min(j0 + tj + 8 * x, N - 1), k = min(k0 + tk, N - 1);
    p[x] = a.dbpart + ((int64_t)bh * N + j) * N + k;
    acc[x] = *p[x];
  }
  int ch = 1;
  for (; ch + 4 <= a.nchunks; ch += 4) {
    float y[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int x = 0; x < 4; ++x) y[u][x] = p[x][(ch + u) * count];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x] += y[u][x];
  }
  for (; ch < a.nchunks; ++ch)
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x] += p[x][ch * count];
  if (turn) {
#pragma unroll
    for (int x = 0; x < 4; ++x) turned[tj + 8 * x][tk] = acc[x];
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int j = j0 + tk, k = k0 + tj + 8 * x;
      if (j < N && k < N) db[j + k * a.sdb_k] = (T)turned[tk][tj + 8 * x];
    }
  } else {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int j = j0 + tj + 8 * x, k = k0 + tk;
      if (j < N && k < N) db[j * a.sdb_j + k * a.sdb_k] = (T)acc[x];
    }
  }
}

}  // namespace tri
