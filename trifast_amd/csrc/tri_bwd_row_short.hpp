// Row-resident backward of short rows: dq, dk and dv of one pair row of up to 512 keys (head dims 16 and 32) by ONE or TWO
// waves, from one computation of the scores and of dP.  The arithmetic is that of tri_bwd_row.hpp (see there: the index
// permutation, the bias and the per-query terms through the matrix pipe, dS through LDS); what differs is who does it and when.
//
// Four waves per row, which longer rows need to hold their dk and dv, cost a short row more than its arithmetic: at n = 512 a
// query tile took 4.3 thousand clocks of which 2.0 are its MFMAs, because every query tile starts and ends the pipeline of its
// few key tiles per wave, is summed from the parts of all waves behind a barrier, and the start and the end of a row (K, V, o and do arrive;
// dk and dv leave) had the compute unit to themselves.  Here
// * a wave holds up to eight key tiles, as at n = 1024: rows of up to 256 keys are one wave's (four rows share a compute unit, nothing
//   is exchanged, no barrier; tri_bwd_row_rule.hpp says which launches spread them over more), rows of up to 512 two waves' (two rows share it).  Rows of a compute unit run apart, so one's loads and stores
//   go on beside the other's arithmetic.
// * the (query tile, key tile) pairs of a wave are one software pipeline that does not end with a query tile: a step holds the
//   exponentials of its pair, the score and dP MFMAs of the pair after it and the dv, dk and dq MFMAs of the pair before it, the next
//   query tile's first pair included.
// * a stage of the query stream carries the o rows beside Q and dO, and delta = rowsum(o * do) of a query tile is formed when it is
//   first needed: the prologue waits for K and V alone (n = 256: 12.2 -> 7.5 us of a row, 512: 14.9 -> 8).
// * nothing in a step branches: the compiler sinks what stands in front of a branch behind it, out of the schedule (a step with one took
//   1.8 instead of 0.9 thousand clocks).  Lanes are masked with exec inside asm statements, pointers advance by masked steps.
//
// bf16, h = 4, d = 32, the dq + dk + dv kernel alone, against the four- and eight-wave forms before it on one card: n = 200 41.1 ->
// 36.0 us, 256 51.2 -> 45.3, 300 115 -> 94, 384 170 -> 142, 449 (interleaved heads) 319 -> 279, 512 343 -> 297, 512 with padding from 397
// on 309 -> 287.  With eight heads at n = 256, two rounds of rows per SIMD, 98 -> 98: the start and end of a row are not hidden there.
//
// What bounds it: instruction issue, as in tri_bwd_row.hpp: a step with both neighbours takes about 740 clocks for 14 to 16 MFMAs (448 to 512
// clocks of matrix pipe), 64 vector instructions of its pair and 50 others (two waves, beside another row's on the same LDS: 820 to 880); the four
// steps that carry the query tile's own work (operands of the next one, its delta, the requests and stores) 50 to 850 more.
#pragma once
#include "tri_bwd_row.hpp"

namespace tri {

constexpr int kShortRowKeys = 512;
constexpr int bwd_short_red_bytes(int NW) { return 4 * (NW - 1) * 1024; }   // dq parts of a query tile for the other wave
constexpr int bwd_short_own_bytes(int NW) { return NW > 1 ? 4 * 1024 : 0; }  // ... and those a wave sums itself
constexpr int bwd_short_stage_bytes(int D, int es) { return 3 * 32 * D * es; }
// Key tiles per wave whose V operands live in LDS instead of registers (eight tiles: as many as LDS has room for)
constexpr int bwd_short_v_lds_tiles(int D, int KT) { return KT * (D / 16) < 16 ? 0 : KT - 3; }
constexpr int bwd_short_lds_bytes(int D, int es, int KT, int NW) {
  const int row = NW * KT * 32 * D * es + 2 * bwd_short_stage_bytes(D, es) + NW * 2048 + 2 * bwd_short_red_bytes(NW) + bwd_short_own_bytes(NW) +
                  NW * bwd_short_v_lds_tiles(D, KT) * (D / 16) * 1024;
  return row > bwd_uniform_lds_bytes(D, es, NW) ? row : bwd_uniform_lds_bytes(D, es, NW);  // (a fully masked row's)
}

template <typename T, int D, int KT, int NW>
__global__ __launch_bounds__(NW * 64, 1) void tri_bwd_row_short_kernel(const BwdArgs a) {
  static_assert(D <= 32 && (NW == 1 || NW == 2) && KT >= 2 && KT <= 8, "the schedule and the registers below");
  static_assert(sizeof(T) == 2, "16-bit inputs only (the transposing LDS reads)");
  using E = Elem<T>;
  using frag = typename E::frag;
  using Tile = LdsTile<T, D>;
  using DsTile = LdsTile<T, 32, 2>;  // the wave's dS tile: 16-byte stores of whole rows, transposed reads
  constexpr int KP = E::KP;
  constexpr int DS = D / (2 * KP);
  constexpr int PS = 2;
  constexpr int ROWB = Tile::ROWB;
  constexpr int KEYS = NW * KT * 32;  // keys the workgroup can hold
  constexpr int STAGE = bwd_short_stage_bytes(D, (int)sizeof(T));  // Q tile | dO tile | o tile
  constexpr int OFF_ST = KEYS * ROWB;  // (the K row comes first)
  constexpr int OFF_DS = OFF_ST + 2 * STAGE;  // two stages: in use; ready or in flight
  constexpr int OFF_RED = OFF_DS + NW * 2048;
  constexpr int RED_BYTES = bwd_short_red_bytes(NW);
  constexpr int OFF_OWN = OFF_RED + 2 * RED_BYTES;
  constexpr int OFF_V = OFF_OWN + bwd_short_own_bytes(NW);
  constexpr int VL = bwd_short_v_lds_tiles(D, KT);  // this wave's last VL key tiles keep V in LDS
  constexpr int VR = KT - VL;
  static_assert(OFF_V + NW * VL * DS * 1024 <= bwd_short_lds_bytes(D, (int)sizeof(T), KT, NW), "the launcher sizes LDS with bwd_short_lds_bytes");
  static_assert(bwd_short_lds_bytes(D, (int)sizeof(T), KT, NW) <= 160 * 1024 / (4 / NW), "a wave for every SIMD of the compute unit");
  extern __shared__ __attribute__((aligned(16))) unsigned char tri_smem[];

  TRI_ROW_MARK(t_entry);
  stagger_rows(blockIdx.x, 4 / NW, a.BH, a.N, D);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = NW > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) : 0;
  // The lane id for addresses inside the loop: opaque wherever it is used, so that nothing derived from it is hoisted out of the loop
  // and kept in registers (it would be spilled, and a reload from scratch waits for every load in flight).
  int lane_o = lane;
  const int kl = lane & 31, g = lane >> 5;
  const int N = a.N;
  const int NJ = a.nwords;  // 32-tiles of the row (queries and keys); this wave's key tiles: wave, wave + NW, ... (past the end: empty)

  // (rows to XCDs as in tri_bwd_row_kernel)
  const int share = bwd_row_xcd_share(a.BH), per_head = (N + share - 1) / share;
  const int L = blockIdx.x, slot = L >> 3;
  const int bh = slot / per_head * (8 / share) + (L & 7) / share, i = slot % per_head * share + (L & 7) % share;
  if (bh >= a.BH || i >= N) return;
  const int b = bh / a.H, h = bh % a.H;

  const T* qrow = reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h + i * a.sq.i;
  const T* krow = reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h + i * a.sk.i;
  const T* vrow = reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h + i * a.sv.i;
  const T* dorow = reinterpret_cast<const T*>(a.dout) + b * a.sdo.b + h * a.sdo.h + i * a.sdo.i;
  const T* orow = reinterpret_cast<const T*>(a.o) + ((int64_t)bh * N + i) * N * D;
  const float* const lserow = a.lse + ((int64_t)bh * N + i) * N;
  const T* pack_bh = reinterpret_cast<const T*>(a.packq) + (int64_t)bh * a.NP * a.NP * 1024;

  // ---- prologue -----------------------------------------------------------------
  // K row -> LDS (rows past the end repeat the last key; their keep bits are clear)
  Tile::template fill<KEYS, NW>(tri_smem, [&](int r) { return krow + (int64_t)min(r, N - 1) * a.sk.j; }, wave, lane);
  // Stages.  The loads are written as asm: the compiler makes every LDS read that follows a global->LDS load it knows of wait for that
  // load.  Here a stage in flight is not read before the wait at the end of a query tile's first step.  The compiler's own waits stay
  // correct: loads return in issue order, and a load it does not know of only makes the counter it waits on larger.
  // A stage is three tiles of LT wave loads of 1 KiB, dealt to the waves in turn: GX loads for each; fill[] are the first rows
  // of the next stage to request, per load or (one wave) per tensor.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(TRI_L3 unsigned char*)tri_smem;
  constexpr int LT = 32 * Tile::CPR / 64, GS = 3 * LT, GX = (GS + NW - 1) / NW, NF = NW == 1 ? 3 : GX;
  const T* fill[NF];
  int64_t fill_step[NF];
  uint32_t fill_row[NF];  // bytes between rows (below 2^24)
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int tensor = NW == 1 ? f : (f * NW + wave) / LT;
    fill[f] = tensor == 0 ? qrow : tensor == 1 ? dorow : orow;
    const int64_t stride = tensor == 0 ? a.sq.j : tensor == 1 ? a.sdo.j : D;
    fill_step[f] = 32 * stride;
    fill_row[f] = (uint32_t)stride * (uint32_t)sizeof(T);
  }
  int fill_rows = N - 1;  // the last row of the pair row, counted from them
  auto issue_stage = [&](int buf) {
    asm volatile("" : "+v"(lane_o));
    const uint32_t ln = (uint32_t)lane_o;
    static_assert(Tile::CPR <= 4, "the swizzle below");
#pragma unroll
    for (int x = 0; x < GX; ++x) {
      const int gi = x * NW + wave, f = NW == 1 ? gi / LT : x;
      const uint32_t r = (uint32_t)(gi % LT * (64 / Tile::CPR)) + ln / Tile::CPR, cc = (ln ^ (r / Tile::RPB)) % Tile::CPR;
      // a 64-bit base per tile (scalar registers) and a 32-bit byte offset per lane; rows past
      // the end of the pair row (last tile only) read the last row again
      const uint32_t voff = __umul24((uint32_t)min((int)r, fill_rows), fill_row[f]) + 16 * cc;
      const T* base = fill[f];
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(OFF_ST + buf * STAGE + gi * 1024));
      if constexpr (GS % NW != 0) {
        // (the last round has no load for the second wave: no lane.  Its counted wait is then for one load fewer, and the other wave's
        // load is waited for by that wave, in front of the barrier)
        const int mine = __builtin_amdgcn_readfirstlane(gi < GS ? -1 : 0);
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" : : "s"(dst), "v"(voff), "s"(base), "s"(mine) : "memory", "m0");
      } else {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(voff), "s"(base) : "memory", "m0");
      }
    }
    // (behind the last query tile the last one is requested again, into a stage nobody reads any more)
    const int more = __builtin_amdgcn_readfirstlane(fill_rows >= 32 ? -1 : 0);
#pragma unroll
    for (int f = 0; f < NF; ++f) fill[f] += fill_step[f] & (int64_t)more;
    fill_rows -= 32 & more;
  };
  issue_stage(0);
  issue_stage(1);

  // (a fully masked row goes its own way; these words come through the scalar cache, all in flight together and apart from the
  // vector loads around them)
  if (uniform_word(a.rowflag, b * N + i) != 0) {
    wait_dma();  // (the loads on their way into the LDS it uses)
    __syncthreads();
    bwd_uniform_row<T, D, NW>(a, bh, i, tri_smem, wave, lane);
    return;
  }
  // keep words of this wave's key tiles (bit k set = key k of the tile is attended)
  uint32_t kw[KT];
#pragma unroll
  for (int t = 0; t < KT; ++t) kw[t] = uniform_word(a.keep, (b * N + i) * a.nwords + min(NW * t + wave, NJ - 1));
#pragma unroll
  for (int t = 0; t < KT; ++t)
    if (NW * t + wave >= NJ) kw[t] = 0u;
  TRI_ROW_MARK(t_p1);

  // V rows of this lane's keys as B operands: in registers for the wave's first VR key
  // tiles, in a private piece of LDS (operand by operand, 16 bytes per lane) for the rest
  frag vf[VR > 0 ? VR : 1][DS];
  frag* const v_lds = reinterpret_cast<frag*>(tri_smem + OFF_V + wave * VL * DS * 1024) + lane;
  frag vx[KT][DS];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int key = min(32 * (NW * t + wave) + kl, N - 1);
#pragma unroll
    for (int s = 0; s < DS; ++s) vx[t][s] = *reinterpret_cast<const frag*>(vrow + (int64_t)key * a.sv.j + 2 * KP * s + KP * g);
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
  // the planes of operand words (-delta, -lse sqrt(d) per query) that the db kernel reads
  uint32_t* const dplane = a.delta + ((int64_t)bh * N + i) * N;
  uint32_t* const lplane = a.lse2 + ((int64_t)bh * N + i) * N;

  // lane-constant LDS offsets.  Q, dO, o tiles: natural A operands (tile row m stands for
  // query perm32(m)) and transposed A operands; K tiles: natural B operand of this lane's
  // key and transposed A operand; the wave's dS tile: write offsets and transposed reads.
  OperandOffsets<T, D> ofq, ofk;
  ofq.init(perm32(kl), lane);
  ofk.init(kl, lane);
  ofk.shift(wave * 32 * ROWB);  // key tile t of this wave starts (NW t + wave) * 32 rows into K
  OperandOffsets<T, 32, 2> ofd;
  ofd.init(0, lane);
  // (one tile: the wave reads dS of a key tile back before it writes the next one)
  unsigned char* const ds_tile = tri_smem + OFF_DS + wave * 2048;
  const int ds_w0 = DsTile::off(kl, 16 * g), ds_w1 = DsTile::off(kl, 32 + 16 * g);

  // packed bias tiles of this lane: tile (jt, kt) is 2 x 16 bytes per lane, an A operand as it is (operand row m stands for query
  // perm32(m)); a tile's address is a wave-uniform base plus this lane's constant 32-bit byte offset
  typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
  uint32_t bias_lane = (uint32_t)((perm32(kl) + 32 * g) * 8 * sizeof(T));
  auto bias_load = [&](int jt, int t, u32x4v* dst) {
    const char* tile = reinterpret_cast<const char*>(pack_bh + ((int64_t)min(jt, a.NP - 1) * a.NP + min(NW * t + wave, a.NP - 1)) * 1024);
    asm volatile("" : "+v"(bias_lane));  // (opaque here: the sum of the lane offset and the head's base is not hoisted as a 64-bit vector)
    dst[0] = *reinterpret_cast<const u32x4v*>(tile + (uint64_t)bias_lane);
    dst[1] = *reinterpret_cast<const u32x4v*>(tile + (uint64_t)bias_lane + 512 * sizeof(T));
  };
  const float c = a.c;

  // sqrt(d) * bias through the matrix pipe, the constant operand (see tri_bwd_row_kernel)
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

  // dq of a query tile.  Quarter q of a tile is the f32x4 of every lane that holds head-dim elements 8 q + 4 g + 0..3 of query
  // 32 jt + kl.  One wave: its tile is the sum.  Two: wave w sums quarters w and w + 2, its own part first; parts wait in LDS as
  // [quarter][lane], a wave's own ones apart from the two buffers (deterministic, no atomics).
  constexpr int NQ = 4 / NW;  // quarters a wave sums
  T* dqrow = reinterpret_cast<T*>(a.dq) + b * a.sdq.b + h * a.sdq.h + i * a.sdq.i;
  typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
  auto store_partials = [&](int buf, const f32x16& acc) {
    asm volatile("" : "+v"(lane_o));
    const int ln = lane_o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = acc[4 * q + e];
      const int at = q % NW == wave ? OFF_OWN + q * 1024 : OFF_RED + (buf ? RED_BYTES : 0) + q * 1024;
      *(reinterpret_cast<f32x4*>(tri_smem + at) + ln) = x;
    }
  };
  // The sum, scaled and rounded, as the stores will write it, in pieces (0 .. kSumPieces - 1, in this order) that stand between the
  // MFMAs of a step: a quarter's parts are read in one and added in the next.
  constexpr int kAddPieces = NW > 1 ? NQ : 0, kSumPieces = kAddPieces + 3;
  struct DqOut {
    f32x4 part[2], sum[NQ];
    u32x4 out[NQ / 2];
    uint32_t off;   // this lane's byte offset from the start of the query tile in dq
    uint64_t live;  // the lanes that store
  };
  auto sum_dq_piece = [&](auto piece_tag, int buf, int jt, const f32x16& acc, DqOut& o) __attribute__((always_inline)) {
    constexpr int piece = decltype(piece_tag)::value;
    if constexpr (piece > 0 && piece <= kAddPieces) o.sum[piece - 1] = o.part[0] + o.part[1];
    if constexpr (piece < kAddPieces) {
      asm volatile("" : "+v"(lane_o));
      const int q = wave + NW * piece;
      o.part[0] = *(reinterpret_cast<const f32x4*>(tri_smem + OFF_OWN + q * 1024) + lane_o);
      o.part[1] = *(reinterpret_cast<const f32x4*>(tri_smem + OFF_RED + (buf ? RED_BYTES : 0) + q * 1024) + lane_o);
    }
    if constexpr (piece == kAddPieces) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (NW == 1) o.sum[q][e] = acc[4 * q + e];
          o.sum[q][e] *= a.scale;
        }
    } else if constexpr (piece == kAddPieces + 1) {
      auto rounded = [&](const f32x4& x) {
        typename E::vec4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (T)x[e];
        return __builtin_bit_cast(u32x2v, v);
      };
      // quarters h and h + 2 trade halves between the two lanes of a query (see store_rows_wide): 16 bytes per lane
#pragma unroll
      for (int hf = 0; hf < NQ / 2; ++hf) {
        const u32x2v x = rounded(o.sum[hf]), y = rounded(o.sum[hf + NQ / 2]);
        const auto r0 = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
        const auto r1 = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
        o.out[hf] = u32x4{(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
      }
    } else if constexpr (piece == kAddPieces + 2) {
      asm volatile("" : "+v"(lane_o));
      const int jl = lane_o & 31, d0 = 16 * (lane_o >> 5) + 8 * wave;  // (head dim 16: columns past the end have no live lane)
      o.live = __builtin_amdgcn_ballot_w64((int)(jl < N - 32 * jt) & (int)(d0 < D)) & (jt < 0 ? 0ull : ~0ull);
      // (row strides of the gradients are below 2^24 bytes, like those of the inputs)
      o.off = (__umul24((uint32_t)jl, (uint32_t)a.sdq.j) + (uint32_t)d0) * (uint32_t)sizeof(T);
    }
  };
  // (a 64-bit base per query tile in scalar registers and the 32-bit byte offset of the lane; every lane of the wave is active here)
  auto store_dq = [&](const T* base, const DqOut& o) {
#pragma unroll
    for (int hf = 0; hf < NQ / 2; ++hf)
      asm volatile("s_mov_b64 exec, %4\n\tglobal_store_dwordx4 %0, %1, %2 offset:%3\n\ts_mov_b64 exec, -1" : : "v"(o.off), "v"(o.out[hf]), "s"(base), "n"(16 * hf), "s"(o.live) : "memory");
  };

  TRI_ROW_MARK(t_p3);
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
  // tiles attended (no mask work) and some keys masked out.
  auto query_tiles = [&](auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    // The masked operands of all key tiles are kept where the registers allow; one wave of eight tiles makes them in the step (n = 256,
    // h = 4: 47.1 -> 45.8 us, nothing of the loop is in scratch any more; two waves lose by it: n = 512 with padding 286 -> 290).
    constexpr bool MASK_BITS = MASKED && KT == 8 && NW == 1;
    int masked_bits = 0;  // bit t set: this lane's key of tile t is masked
    if constexpr (MASK_BITS) {
#pragma unroll
      for (int t = 0; t < KT; ++t) masked_bits |= (kw[t] >> kl & 1u ? 0 : 1) << t;
    }
    // (each version has its own accumulators, from zeroing to the final stores: merging
    // the versions' accumulators where they meet would copy all of them)
    f32x16 dkacc[KT], dvacc[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      E::mfma_acc_zero(dkacc[t]);
      E::mfma_acc_zero(dvacc[t]);
    }
    // One wave per SIMD leaves hiding a latency to the wave's own instruction
    // order: the code below is laid out as the schedule it should run in, and scheduling
    // barriers between the pieces keep the compiler from re-ordering it.
    auto SB = [] { __builtin_amdgcn_sched_barrier(0); };
    constexpr int NACC = 2 * PS;  // dv, dk MFMAs of a tile
    // packed bias of key tile t (t >= KT: tile t - KT of the next query tile) -> the ring slot
    // of that tile's parity, fetched two steps before its use (global memory, through L2).
    // (With an odd KT, tile 0 of the next query tile goes to the slot that tile KT-1 is read
    // from in the same step: its fetch follows the last MFMA that reads bias words.)
    u32x4v bias_ring[2][2] = {};
    auto fetch_bias = [&](int jt, int t) { bias_load(jt + t / KT, t % KT, bias_ring[(t % KT) % 2]); };
    fetch_bias(0, 0);
    const T* dq_base = dqrow;  // dq of the query tile before the current one (from the second on)
    int buf = 0;               // jt % 2: the stage of this query tile
    int jt = 0;
#ifdef TRI_ROW_TIMING
    uint32_t tacc[KT + 5] = {};  // shader clocks per step, summed over the query tiles
    const uint32_t t_clk0 = (uint32_t)__builtin_amdgcn_s_memtime(), t_loop0 = (uint32_t)__builtin_amdgcn_s_memrealtime();
    uint32_t tprev = t_clk0;
#endif

    // ---- the state that moves from step to step --------------------------------------
    DqOut dq_out;
    f32x16 dqacc = zero16();       // (the first dq MFMA of a query tile starts it from zero)
    frag qn[DS], don[DS], on[DS];  // Q, dO rows (A operands) of the pair that is started next; o rows, until delta is known
    frag qtr[PS], dotr[PS];        // Q^T, dO^T (A operands of dk, dv) of the pair that is finished next
    f32x16 s_cur, p_cur;           // scores and dP of the pair whose P, dS the step computes
    f32x16 s_nxt, p_nxt;           // ... of the pair after it, accumulating
    float p[16], ds[16];
    frag kn[DS];           // K rows of the next tile as B operand
    frag pf[PS], dsf[PS];  // P and dS of the last finished tile as B operands
    frag dst_prev[PS], ktr_prev[PS];
    frag vn[DS];           // V operands of the next tile when they live in LDS
    float lse_next = 0.f, dsum = 0.f;
    // (before the first query tile the pipeline runs on zeros; its dq is not stored)
#pragma unroll
    for (int s2 = 0; s2 < PS; ++s2) qtr[s2] = dotr[s2] = pf[s2] = dsf[s2] = E::zero();
    auto load_qd_tr = [&] {
      const unsigned char *qt = tri_smem + OFF_ST + buf * STAGE, *dot = qt + 32 * ROWB;
#pragma unroll
      for (int s2 = 0; s2 < PS; ++s2) {
        qtr[s2] = ofq.transposed_all(qt, s2, 0);
        dotr[s2] = ofq.transposed_all(dot, s2, 0);
      }
    };
    // (transposed_all, here and for K: head dim 16 fills half of the operand's rows, and the results of the others, made of whatever lies
    // behind a row, are never stored)
    // Q, dO, o rows in stage st (behind the last query tile: of anything, the pair is not used)
    auto load_query = [&](int st) {
      const unsigned char *qt = tri_smem + OFF_ST + st * STAGE, *dot = qt + 32 * ROWB;
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        qn[s] = ofq.natural(qt, s);
        don[s] = ofq.natural(dot, s);
        on[s] = ofq.natural(dot + 32 * ROWB, s);
      }
    };
    // The operand words of query tile jq (lanes 32..63 carry zeros); delta comes from the o and dO rows, of which a lane holds
    // half, in two pieces.
    auto fetch_lse = [&](int jq) { lse_next = lserow[min(32 * jq + perm32(kl), N - 1)]; };
    auto set_lse = [&](int jq) {
      const uint32_t word = split_word<T>(perm32(kl) < N - 32 * jq ? -lse_next * a.sqrt_d : E::kMaskElem);  // queries past the end: P = dS = 0
      s_off.set_raw(word & (uint32_t)(g - 1));
    };
    auto set_delta = [&](int jq, int piece) __attribute__((always_inline)) {
      if (piece == 0) {
        dsum = 0.f;
#pragma unroll
        for (int s = 0; s < DS; ++s)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            typedef T pair __attribute__((ext_vector_type(2)));
            dsum = pair_dot(pair{on[s][e], on[s][e + 1]}, pair{don[s][e], don[s][e + 1]}, dsum);
          }
      } else {
        const uint32_t word = split_word<T>(-half_sum(dsum)), live = (uint32_t)-((int)(g == 0) & (int)(perm32(kl) < N - 32 * jq));
        d_off.v[0] = word & live;
      }
    };
    // The first wave leaves the words of this query tile for the db kernel.
    auto store_words = [&] {
      asm volatile("" : "+v"(lane_o));
      const int q = perm32(lane_o & 31);
      const uint64_t live = __builtin_amdgcn_ballot_w64((int)(q < N - 32 * jt) & (int)(lane_o < 32)) & (wave == 0 ? ~0ull : 0ull);
      uint32_t *const dwords = dplane + 32 * jt, *const lwords = lplane + 32 * jt;
      const uint32_t dw = d_off.v[0], lw = s_off.v[0];
      asm volatile("s_mov_b64 exec, %5\n\tglobal_store_dword %0, %1, %2\n\tglobal_store_dword %0, %3, %4\n\ts_mov_b64 exec, -1" : : "v"(4 * q), "v"(dw), "s"(dwords), "v"(lw), "s"(lwords), "s"(live) : "memory");
    };
    auto load_kn = [&](int t) {
#pragma unroll
      for (int s = 0; s < DS; ++s) kn[s] = ofk.natural(tri_smem + NW * t * 32 * ROWB, s);
    };

    // Step t (0 .. KT-1): the vector work of key tile t (P, dS, their conversions) between
    // the MFMAs of its neighbours: dv, dk and dq of the pair before, scores and dP of the pair after,
    // in the order of RowSched.  Step -1 only starts the first pair, step KT only finishes the last.
    auto step = [&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value - 1;
      constexpr bool has_prev = t >= 0, has_next = t < KT, valu = has_prev && has_next;
      constexpr int tn = (t + 1) % KT, tp = (t - 1 + KT) % KT;  // the tiles that are started and finished
      constexpr bool new_query = has_next && tn == 0;           // the tile that is started is the next query tile's
      using Sch = RowSchedOf<has_prev, has_next, NSB, DS, NACC, PS, true>;
      constexpr int NM = Sch::value.n;
      constexpr int NU = valu ? 16 : 0;  // vector units of four instructions
      constexpr bool fetch_late = KT % 2 != 0 && (t + 2) % KT == 0;
      SB();
      frag kb = keys_op.plain();
      if constexpr (has_next && MASK_BITS) {
        kb = keys_op.masked_bit(masked_bits, tn);
        SB();
      }
      if constexpr (valu) TRI_ROW_TICK(t);  // (slot 0: step KT-1; slot k: step k-1, less the end of step 0, see below)
      if constexpr (new_query) {
        set_lse(jt + (t < 0 ? 0 : 1));
        if constexpr (KT == 2 && t < 0) fetch_lse(1);
      }
      if constexpr (has_next && !fetch_late) fetch_bias(jt, t + 2);
      // (Without masked keys the product of a query's words is the same for every key tile, and the compiler keeps both of them; one
      // wave of eight key tiles has no registers for that and would reload its V operands from scratch, which waits for every load in flight:
      // h = 8, n = 256 98.9 -> 97.1 us with the scores' product made anew.  Two waves have: n = 512 302.4, made anew 303.7.)
      if constexpr (KT == 8 && NW == 1 && has_next && !MASKED) asm volatile("" : "+v"(s_off.v[0]));
      if constexpr (has_next && MASKED && !MASK_BITS) kb = keys_op.masked(kw[tn]);
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
          if constexpr (idx % 2 == 0) E::mfma_acc(dotr[idx / 2], pf[idx / 2], dvacc[tp]);
          else E::mfma_acc(qtr[idx / 2], dsf[idx / 2], dkacc[tp]);
        } else {
          if constexpr (tp == 0 && idx == 0) dqacc = E::mfma(ktr_prev[idx], dst_prev[idx], zero16());
          else dqacc = E::mfma(ktr_prev[idx], dst_prev[idx], dqacc);
        }
        SB();
        // dq of the query tile before this one is summed and stored in the step after the barrier that follows its last partial tile
        if constexpr (t == 1 && has_next) {
          static_for<kSumPieces>([&](auto pc) __attribute__((always_inline)) {
            constexpr int piece = decltype(pc)::value, at = NW > 1 ? piece * 3 : piece;
            if constexpr ((at < NM ? at : NM - 1) == x) sum_dq_piece(pc, (jt + 1) & 1, jt - 1, dqacc, dq_out);
          });
          if constexpr (x == NM - 1) {
            store_dq(dq_base, dq_out);
            dq_base += jt > 0 ? 32 * a.sdq.j : 0;
          }
        }
        // The stage after next is requested in the same step, behind its last read of bias words: loads return in issue order, so the
        // next wait for bias words is a wait for these loads too, and from there it is the furthest away.  With them lse of the next
        // query tile (of the one after, where this step is the last one) and the words' stores.
        if constexpr (t == 1 && has_next && x == Sch::value.last_sb) {
          issue_stage(buf);
          fetch_lse(jt + (KT == 2 ? 2 : 1));
          if constexpr (KT > 2) store_words();
        }
        if constexpr (KT == 2 && t == 0 && x == Sch::value.last_sb) store_words();
        if constexpr (has_next && x == Sch::value.last_sqk) load_kn((tn + 1) % KT);
        // (in front of the MFMA that dP starts with)
        if constexpr (new_query && x == 0) set_delta(jt + (t < 0 ? 0 : 1), 0);
        if constexpr (new_query && x == 2) set_delta(jt + (t < 0 ? 0 : 1), 1);
        if constexpr (has_next && tn >= VR && x == Sch::value.v_reads_at) {
#pragma unroll
          for (int s = 0; s < DS; ++s) vn[s] = v_lds[((tn - VR) * DS + s) * 64];
        }
        // Q^T, dO^T of this query tile: first used by the next step (transposing reads are the slowest LDS reads: once per query tile)
        if constexpr (t == 0 && x == Sch::value.last_acc) load_qd_tr();
        if constexpr (has_prev && x == Sch::value.dq_reads_at) {
          // dS of the pair before comes back from LDS with the key index in-lane, with the K
          // rows of its tile transposed beside it
#pragma unroll
          for (int s2 = 0; s2 < PS; ++s2) {
            dst_prev[s2] = ofd.transposed(ds_tile, s2, 0);
            ktr_prev[s2] = ofk.transposed_all(tri_smem + NW * tp * 32 * ROWB, s2, 0);
          }
        }
        if constexpr (has_next && fetch_late && x == Sch::value.last_sb) fetch_bias(jt, t + 2);
#pragma unroll
        for (int u = x * NU / NM; u < (x + 1) * NU / NM; ++u) unit(u);
        SB();
      });
      if constexpr (valu) {
        // dS -> the wave's LDS tile [key][query]
        *reinterpret_cast<frag*>(ds_tile + ds_w0) = dsf[0];
        *reinterpret_cast<frag*>(ds_tile + ds_w1) = dsf[1];
        SB();
      }
      if constexpr (t == 0) {
        // dq of the query tile before this one is complete in this wave.  The barrier behind its partial tiles is the only one
        // of a query tile; it also says that every wave has read Q^T and dO^T of this query tile, whose stage is then refilled, and
        // that the stage requested a query tile ago has landed: of all that was issued since, only this step's two loads of bias words
        // may be in flight (two key tiles: this step's stores; a wave waits for its bias words, and with them for everything older).  A barrier
        // without a fence: a fence would wait for the loads in flight.  The buffer that the partials are in is written again
        // two query tiles on, behind the next barrier.
        TRI_ROW_TICK(KT);
        if constexpr (NW > 1) store_partials((jt + 1) & 1, dqacc);
        TRI_ROW_TICK(KT + 1);
        if constexpr (NW > 1) ring_sync<2>();
        else asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" : : : "memory");
        TRI_ROW_TICK(KT + 2);
      }
      if constexpr (has_next && (t + 2) % KT == 0) load_query(buf ^ 1);
      if constexpr (has_next) { s_cur = s_nxt; p_cur = p_nxt; }
    };
    fetch_lse(0);
    load_query(0);
    load_kn(0);
    step(std::integral_constant<int, 0>{});
    for (; jt < NJ; ++jt) {
      static_for<KT>([&](auto tc) __attribute__((always_inline)) { step(std::integral_constant<int, decltype(tc)::value + 1>{}); });
      buf ^= 1;
    }
    step(std::integral_constant<int, KT + 1>{});
    // dq of the last query tile (the requests behind it have landed in LDS when the wave ends)
    if constexpr (NW > 1) {
      store_partials((NJ - 1) & 1, dqacc);
      ring_sync<0>();
    } else {
      wait_dma();
    }
    static_for<kSumPieces>([&](auto pc) __attribute__((always_inline)) { sum_dq_piece(pc, (NJ - 1) & 1, NJ - 1, dqacc, dq_out); });
    store_dq(dq_base, dq_out);
#ifdef TRI_ROW_TIMING
    const uint32_t t_clk1 = (uint32_t)__builtin_amdgcn_s_memtime(), t_loop1 = (uint32_t)__builtin_amdgcn_s_memrealtime();
#endif

    // ---- dk, dv of this wave's keys -------------------------------------------------------
    // (the accumulators were last written by MFMAs inside asm statements, which the compiler
    // does not know to be MFMAs: each is read only after that MFMA has had time to retire)
    T* dkrow = reinterpret_cast<T*>(a.dk) + b * a.sdk.b + h * a.sdk.h + i * a.sdk.i;
    T* dvrow = reinterpret_cast<T*>(a.dv) + b * a.sdv.b + h * a.sdv.h + i * a.sdv.i;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int key = 32 * (NW * t + wave) + kl;
#ifndef TRI_MFMA_ACC_BUILTIN
      asm volatile("s_nop 15" : "+a"(dkacc[t]));
      asm volatile("s_nop 15" : "+a"(dvacc[t]));
#endif
      store_rows_wide<T, D, 1>(dkrow + (int64_t)key * a.sdk.j, &dkacc[t], a.scale, g, key < N);
      store_rows_wide<T, D, 1>(dvrow + (int64_t)key * a.sdv.j, &dvacc[t], 1.0f, g, key < N);
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
      for (int x = 0; x < KT + 3; ++x) rec[11 + x] = tacc[x];
      rec[28] = KT;
      rec[29] = NW;
      rec[30] = 1;
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
