// Forward kernel: flash-style triangle attention.
//
// Work unit: (batch*head, R consecutive pair rows i, block of NW*32 queries j).
// Wave w owns one tile of 32 queries for all R rows.  The three operands of the
// iteration space (i, j, k) live in three places:
//   * bias[j, k] does not depend on the row: one packed bias tile (registers) is
//     reused by the R rows, which divides its L2 traffic by R;
//   * K[i], V[i] do not depend on the query: they are streamed through LDS in
//     tiles of BK keys (direct global->LDS loads, swizzled, double-buffered) and
//     shared by the NW waves;
//   * Q[i, j] and the output accumulator stay in registers for the whole sweep.
// Scores are computed TRANSPOSED, S^T = K Q^T, so that a lane owns one query
// (column) and 16 keys of every 32-key tile: the softmax running reference / sum
// are per-lane scalars, and the probabilities are already in B-operand layout
// for O^T += V^T P^T, whose A operand V^T comes from the natural V tile through
// transposing LDS reads.
//
// Raw-score domain: acc = sqrt(d) * bias + q.k (the converted bias tile is the
// accumulator init of the score MFMA and is shared by the R rows);
// p = exp2(acc * c - ref * c) with c = log2(e) / sqrt(d).  `ref` is the running
// reference of the online softmax: it is raised to the running maximum only when
// the probabilities of some query of the wave sum to more than 2^kLazy within a
// tile, so the accumulator rescale is rare and no maximum is searched otherwise;
// p stays below 2^kLazy, which fp32/bf16/fp16 hold.
//
// Masks: a bitmap over the key tiles says which stages are live (others are
// skipped) and whether all of them are plain (every row attends to every key:
// the workgroup then runs a loop with no mask work and no per-tile branch).
// Otherwise a masked key gets a large negative score through one extra MFMA
// (see OffsetMask).  The scheduled loop further down exists in both forms and takes any n.
// Workgroups of fully masked rows write the mean of V; those that mix such rows with others, and
// fp32, take the general stage loop.
//
// Replaces _fwd of reference src/trifast/triton.py:19-132.
#pragma once
#include <type_traits>

#include "tri_args.hpp"
#include "tri_common.hpp"
#include "tri_f32_plain.hpp"
#include "tri_tile.hpp"

namespace tri {

constexpr float kLazy = 8.0f;
constexpr float kLazyLimit = 256.0f;  // 2^kLazy

// BKF: keys per stage of the general stage loop, plus kFwdFast when a workgroup without a fully
// masked row takes the scheduled loop below.
constexpr int kFwdFast = 256;
// LDS bytes of the two loops (without the key-tile bitmaps that follow them)
constexpr int fwd_stage_bytes(int D, int es, int NW, int R, int BK) { return 2 * R * BK * lds_row_bytes(D, es) + (es == 4 ? 0 : NW * (BK / 32) * 1024 * es) + 256; }
// stages of the scheduled loop's ring: what is in use, what the next barrier publishes, and
// the rest in flight: four where two workgroups per compute unit then still fit in its LDS,
// else three (four pair rows, or 128-byte rows: their loads are then issued a stage's last tile
// before the barrier that needs them; one workgroup with four stages is slower, 2.1 against
// 1.6 ms at n = 768, h = 8, d = 64)
constexpr int fwd_fast_stages(int D, int es, int NW, int R) { return 2 * 4 * ring_stage_bytes(D, es, NW, R) <= 150 * 1024 ? 4 : 3; }
constexpr int fwd_main_lds_bytes(int D, int es, int NW, int R, int BKF) {
  const int gen = 2 * fwd_stage_bytes(D, es, NW, R, BKF % kFwdFast);
  const int fast = BKF >= kFwdFast ? fwd_fast_stages(D, es, NW, R) * ring_stage_bytes(D, es, NW, R) : 0;
  return gen > fast ? gen : fast;
}

// R fully masked rows (the padding of a padded batch): all logits of such a row are equal, so
// every query's output is the mean of the row's V and its log-sum-exp is ln n.  One pass over V
// instead of a sweep of score tiles: the workgroup's threads take the 16-byte chunks of V's rows
// in turn, add them in fp32 in a fixed order and meet in LDS, all rows at the same barriers.  (n = 512 of which 115 rows are
// padding: 160 -> 136 us.  Row after row, with a barrier of its own for the dropped first stage, what that stage costs these rows
// was not made up for: half of the rows padding, bf16, us, before the stage was requested early / with it / now: h = 4, d = 16, n = 256
// 16.9 / 17.7 / 16.4, n = 512 63.7 / 63.4 / 57.2; h = 8, d = 64, n = 256 46.9 / 48.0 / 45.9; h = 4, d = 128, n = 300 69.5 / 71.0 / 68.2, 512
// 232 / 236 / 219.  One row per workgroup gains nothing by meeting: d = 128, n = 128 16.0 / 16.2 / 16.2.  Keys that do
// not fill the last round of loads: taken one after the other they cost a trip to memory each, d = 128, h = 8, n = 77 17.9 us, now 16.8, n = 230 83.7 / 77.9, n = 450
// 377 / 367; d = 32, h = 8, n = 230 33.2 / 32.2.)
template <typename T, int D, int NW, int R, int LDS>
TRI_DEV void fwd_uniform_rows(const FwdArgs& a, const T* vbh, int bh, int i0, int j_blk, unsigned char* smem) {
  using vec = typename Elem<T>::vec;
  constexpr int VEC = Elem<T>::VEC, CH = D / VEC, SLOTS = NW * 64 / CH;  // chunks per row, threads per chunk
  const int N = a.N, tid = threadIdx.x, ch = tid % CH, slot = tid / CH;
  // rows at a time: their parts meet in the LDS of the workgroup's stages
  constexpr int G = R * SLOTS * D * 4 <= LDS ? R : R / 2;
  static_assert(G * SLOTS * D * 4 <= LDS);
  float (*part)[SLOTS][D] = reinterpret_cast<float (*)[SLOTS][D]>(smem);  // [G]
  const float lse = kLn2 * fast_log2((float)N) + a.neg_inf;
#pragma unroll 1
  for (int r0 = 0; r0 < R; r0 += G) {
    const T* v[G];
    float acc[G][VEC] = {};
#pragma unroll
    for (int r = 0; r < G; ++r) v[r] = vbh + min(i0 + r0 + r, N - 1) * a.sv.i + ch * VEC;  // (rows past the end are not stored)
    constexpr int U = 8 / G;  // (eight loads in flight, the last ones too: past the last key the last one is read again and counts as zero)
#pragma unroll 1
    for (int k0 = 0; k0 < N; k0 += U * SLOTS) {
      typedef uint32_t words __attribute__((ext_vector_type(4)));
      words x[U][G];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < G; ++r) x[u][r] = *reinterpret_cast<const words*>(v[r] + (int64_t)min(k0 + u * SLOTS + slot, N - 1) * a.sv.j);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t live = (uint32_t)-(int)(k0 + u * SLOTS + slot < N);
#pragma unroll
        for (int r = 0; r < G; ++r) {
          const vec y = __builtin_bit_cast(vec, x[u][r] & live);
#pragma unroll
          for (int e = 0; e < VEC; ++e) acc[r][e] += (float)y[e];
        }
      }
    }
    if (r0 == 0) wait_dma();  // (the first stage, requested before the row flags were read, has landed in this LDS)
    __syncthreads();          // (the rows before have been read)
#pragma unroll
    for (int r = 0; r < G; ++r)
#pragma unroll
      for (int e = 0; e < VEC; ++e) part[r][slot][ch * VEC + e] = acc[r][e];
#pragma unroll
    for (int half = SLOTS / 2; half > 0; half /= 2) {
      __syncthreads();
      if (slot < half) {
#pragma unroll
        for (int r = 0; r < G; ++r)
#pragma unroll
          for (int e = 0; e < VEC; ++e) part[r][slot][ch * VEC + e] += part[r][slot + half][ch * VEC + e];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < G; ++r) {
      const int i = i0 + r0 + r;
      if (i >= N) break;
      vec out;
#pragma unroll
      for (int e = 0; e < VEC; ++e) out[e] = (T)(part[r][0][ch * VEC + e] / (float)N);
      const int64_t row = ((int64_t)bh * N + i) * N;
      T* o = reinterpret_cast<T*>(a.o) + row * D + ch * VEC;
      for (int j = j_blk + slot; j < min(j_blk + NW * 32, N); j += SLOTS) *reinterpret_cast<vec*>(o + (int64_t)j * D) = out;
      if (tid < NW * 32 && j_blk + tid < N) a.lse[row + j_blk + tid] = lse;
    }
  }
}

// the probabilities of an operand on top of a row sum: as the MFMA sees them (16-bit types round)
template <typename T, typename F>
TRI_DEV float row_sum(const F& pf, const float* p, float acc) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc += p[e];
    return acc;
  } else {
    return frag_sum(pf, acc);
  }
}

template <typename T, int D, int NW, int R, int BKF>
__global__ __launch_bounds__(NW * 64, (R * ((BKF % kFwdFast) / 32) >= 8 || D * sizeof(T) > 256) ? 1 : 2) void tri_fwd_kernel(const FwdArgs a) {
  constexpr int BK = BKF % kFwdFast;
  constexpr bool FAST = BKF >= kFwdFast;
  using E = Elem<T>;
  using frag = typename E::frag;
  constexpr int KP = E::KP;
  constexpr int DS = D / (2 * KP);   // MFMA steps over the head dim
  constexpr int DM = (D + 31) / 32;  // 32-row tiles of O^T
  constexpr int PS = 32 / (2 * KP);  // MFMA steps over a 32-key tile
  constexpr int KU = BK / 32;

  // One stage: K rows of the R pair rows | V rows | packed bias tiles of the NW waves.
  // Two stages (double buffer), then the key-tile bitmaps.
  using Tile = typename OperandOffsets<T, D>::Tile;
  constexpr int ROWB = lds_row_bytes(D, (int)sizeof(T));
  constexpr int OFF_K = 0, OFF_V = R * BK * ROWB, OFF_B = 2 * R * BK * ROWB;
  constexpr int BIAS_B = sizeof(T) == 4 ? 0 : 2 * 64 * 8 * (int)sizeof(T);  // one packed 32 x 32 bias tile
  constexpr int OFF_KW = OFF_B + NW * KU * BIAS_B;  // keep words of the stage's tiles, [R][KU] (64 slots)
  constexpr int STAGE = OFF_KW + 256;
  static_assert(STAGE == fwd_stage_bytes(D, (int)sizeof(T), NW, R, BK), "the launcher sizes LDS with fwd_stage_bytes");
  constexpr int LDS_MAIN = fwd_main_lds_bytes(D, (int)sizeof(T), NW, R, BKF);  // the key-tile bitmaps follow
  static_assert(R * KU <= 64, "the keep words of a stage are one 64-lane load");
  extern __shared__ __attribute__((aligned(16))) unsigned char tri_smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int jl = lane & 31, g = lane >> 5;
  const int N = a.N;
  int bx, by;
  xcd_remap(gridDim.x, bx, by);
  const int i0 = by * R;
  if (i0 >= N) return;
  const int bh = blockIdx.z;
  const int b = bh / a.H, h = bh % a.H;
  const int j_wave = bx * (NW * 32) + wave * 32;
  const int j = j_wave + jl;
  const bool wave_active = j_wave < N;
  const int jt = j_wave >> 5;

  const T* qbh = reinterpret_cast<const T*>(a.q) + b * a.sq.b + h * a.sq.h;
  const T* kbh = reinterpret_cast<const T*>(a.k) + b * a.sk.b + h * a.sk.h;
  const T* vbh = reinterpret_cast<const T*>(a.v) + b * a.sv.b + h * a.sv.h;
  const T* pack_bh = reinterpret_cast<const T*>(a.packq) + (int64_t)bh * a.NP * a.NP * 1024;

  const int jt_ld = min(jt, a.NP - 1);
  // The first stages of the scheduled loop's ring are requested before anything else: the row
  // flags, keep words and Q rows that decide how the workgroup goes on arrive in the same trip to
  // memory.
  constexpr int RR = FAST ? R : 4;
  using Ring = StageRing<std::conditional_t<FAST, T, __bf16>, D, NW, RR, fwd_fast_stages(D, 2, NW, RR)>;
  Ring ring;
  bool ring_on = false;
  if constexpr (FAST) {
    ring_on = Ring::fits(a.sk) && Ring::fits(a.sv);
    if (ring_on) {
      ring.init(a.sk, a.sv, kbh, vbh, pack_bh + (int64_t)jt_ld * a.NP * 1024, 1024, N, i0, wave, lane, tri_smem);
#pragma unroll
      for (int st = 0; st < Ring::NS - 1; ++st) ring.issue(st * Ring::FSTAGE, a.nwords, wave, lane);
    }
  }
  // (what goes another way starts from empty buffers)
  auto drop_loads = [&] {
    wait_dma();
    __syncthreads();
  };

  // the key mask enters the scores through one extra MFMA: keys operand with the mask
  // element of this lane's key (patched in place per tile) against a constant queries
  // operand (see OffsetMask; its per-query offset is not used here: the word is zero)
  typename OffsetMask<T>::Keys kop;
  typename E::ofrag qzero;

  // per-lane source pointers of the K and V stage tiles for keys 0..BK-1
  // (set up by the general stage loop only: the scheduled loop below has no use for them, and
  // what is live across the choice between the two loops takes registers from both)
  using Stream = std::conditional_t<sizeof(T) == 4, SplitStream<D, R * BK, NW>, TileStream<T, D, R * BK, NW>>;
  Stream kstream, vstream;
  auto setup_general = [&] {
    kop.init(perm32(jl), g);
    typename OffsetMask<T>::Queries qz;
    qz.init(split_word<T>(0.f), g);
    qzero = qz.get();
    kstream.init([&](int x) { return kbh + min(i0 + x / BK, N - 1) * a.sk.i + (int64_t)(x % BK) * a.sk.j; }, wave, lane);
    vstream.init([&](int x) { return vbh + min(i0 + x / BK, N - 1) * a.sv.i + (int64_t)(x % BK) * a.sv.j; }, wave, lane);
  };

  // Stage loads: direct global->LDS.  A stage that lies inside the key range adds
  // one uniform offset to the precomputed pointers; the last, ragged one clamps
  // key indices instead of branching (a clamped key row duplicates the last valid
  // one; its keep bit is clear, so it contributes exactly zero).
  const T* bias_lane;
  // keep words travel with the stage (lane x of wave 0: row x / KU, key tile x % KU);
  // workgroups that attend to every key do not need them
  const uint32_t* kw_lane;
  int kw_u;
  // (set where their loop is prepared: live from here on they cost the scheduled loop 0.7 %, n = 1024 1000 us, now 993)
  auto setup_words = [&] {
    bias_lane = pack_bh + ((int64_t)jt_ld * a.NP * 2 * 64 + lane) * 8;
    kw_lane = a.keep + ((int64_t)b * N + min(i0 + (lane % (R * KU)) / KU, N - 1)) * a.nwords;
    kw_u = lane % KU;
  };
  bool want_keep_words = true;
  f32x4 bias_x[KU][4];   // fp32: packed bias words on their way
  f32x16 bias_cur[KU];   // fp32: the bias tiles of the stage in use
  auto issue_loads = [&](int kt0, int buf) {
    unsigned char* st = tri_smem + buf * STAGE;
    if (want_keep_words && wave == 0)
      __builtin_amdgcn_global_load_lds((const TRI_G1 void*)(kw_lane + min((kt0 >> 5) + kw_u, a.nwords - 1)), (TRI_L3 void*)(st + OFF_KW), 4, 0, 0);
    auto k_row = [&](int x) { return kbh + min(i0 + x / BK, N - 1) * a.sk.i + (int64_t)min(kt0 + x % BK, N - 1) * a.sk.j; };
    auto v_row = [&](int x) { return vbh + min(i0 + x / BK, N - 1) * a.sv.i + (int64_t)min(kt0 + x % BK, N - 1) * a.sv.j; };
    if constexpr (sizeof(T) == 4) {
      // (into registers; store_loads() writes them once the stage in use has been computed)
      if (kt0 + BK <= N) {
        kstream.load((int64_t)kt0 * a.sk.j);
        vstream.load((int64_t)kt0 * a.sv.j);
      } else {
        asm volatile("" ::);
        kstream.load_rows(k_row);
        vstream.load_rows(v_row);
      }
    } else if (kt0 + BK <= N) {
      kstream.issue(st + OFF_K, (int64_t)kt0 * a.sk.j, wave);
      vstream.issue(st + OFF_V, (int64_t)kt0 * a.sv.j, wave);
    } else {
      asm volatile("" ::);  // keeps this rare path a real branch (no speculation into the common one)
      Tile::template fill<R * BK, NW>(st + OFF_K, k_row, wave, lane);
      Tile::template fill<R * BK, NW>(st + OFF_V, v_row, wave, lane);
    }
    // each wave fetches the packed bias tiles of its own query tile: 2 x 1 KiB per key tile
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const T* p = bias_lane + (int64_t)min((kt0 >> 5) + u, a.NP - 1) * 1024;
#pragma unroll
      for (int r2 = 0; r2 < 2; ++r2) {
        if constexpr (sizeof(T) == 4) {
          // (fp32: into registers, which leaves LDS room for another workgroup)
          bias_x[u][2 * r2] = *reinterpret_cast<const f32x4*>(p + r2 * 512);
          bias_x[u][2 * r2 + 1] = *reinterpret_cast<const f32x4*>(p + r2 * 512 + 4);
        } else {
          unsigned char* dst = st + OFF_B + (wave * KU + u) * BIAS_B + r2 * (BIAS_B / 2);
          __builtin_amdgcn_global_load_lds((const TRI_G1 void*)(p + r2 * 512), (TRI_L3 void*)dst, 16, 0, 0);
        }
      }
    }
  };
  auto store_loads = [&](int buf) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int u = 0; u < KU; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) bias_cur[u][e] = bias_x[u][e / 4][e % 4] * a.sqrt_d;
      kstream.store(tri_smem + buf * STAGE + OFF_K);
      vstream.store(tri_smem + buf * STAGE + OFF_V);
    }
  };
  // The first stage of the other tiles' loop is requested here too, whether or not some row attends to it: its loads would otherwise wait
  // for the row flags, the keep words behind those and the key-tile bitmaps made of them, three trips to memory (inference, bf16, us: h = 4, d = 32,
  // n = 130 19.4 -> 18.4; d = 64, b = 2, n = 100 20.0 -> 18.7; h = 2, d = 128, n = 250 42.1 -> 40.8; d = 32, n = 400 padded 58.8 -> 58.3).
  // In fp32 the loads would hold registers meanwhile: 16 spilled at d = 64, two waves per SIMD in place of three at d = 32.
  constexpr bool EARLY = !FAST && sizeof(T) == 2;
  if constexpr (EARLY) {
    setup_general();
    setup_words();
    issue_loads(0, 0);
  }

  // per-row state.  A fully masked row drops the q.k and bias terms (all logits
  // equal): its Q operand is zero and it skips the bias.
  bool flagged[R];
  bool any_flagged = false;
  const uint32_t* keep_row[R];
  frag qf[R][DS];
  f32x16 oacc[R][DM];
  float mref[R], mc[R], lrun[R];
  bool all_flagged = true;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    flagged[r] = uniform_word(a.rowflag, b * N + min(i0 + r, N - 1)) != 0;
    all_flagged &= flagged[r];
  }
  if (all_flagged) {
    fwd_uniform_rows<T, D, NW, R, LDS_MAIN>(a, vbh, bh, i0, bx * (NW * 32), tri_smem);
    return;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = min(i0 + r, N - 1);  // rows past the end repeat the last one and are not stored
    any_flagged |= flagged[r];
    keep_row[r] = a.keep + ((int64_t)b * N + i) * a.nwords;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      if (j < N && !flagged[r])
        qf[r][s] = E::load(qbh + i * a.sq.i + (int64_t)j * a.sq.j + 2 * KP * s + KP * g);
      else
        qf[r][s] = E::zero();
    }
    mref[r] = kNeg;
    mc[r] = kNeg;
    lrun[r] = 0.f;
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) oacc[r][mt] = zero16();
  }
  const float c = a.c;

  KeyTileMasks masks;
  masks.build<R, NW>(reinterpret_cast<uint64_t*>(tri_smem + LDS_MAIN), [&](int r) { return keep_row[r]; }, a.nwords, any_flagged, wave, lane,
                      FAST && (N & 31) != 0 ? 0xffffffffu << (N & 31) : 0u);

  // lane-constant LDS offsets of the operand reads: K rows as natural operands
  // (tile row m stands for key perm32(m)), V rows through transposing reads
  OperandOffsets<T, D> ofs;
  ofs.init(perm32(jl), lane);
  if constexpr (!EARLY) setup_words();

  // the 16 bias values of this lane for key tile u of the stage, raw-score domain
  auto bias_from_lds = [&](int buf, int u) -> f32x16 {
    const unsigned char* src = tri_smem + buf * STAGE + OFF_B + (wave * KU + u) * BIAS_B;
    f32x16 bv;
#pragma unroll
    for (int r2 = 0; r2 < 2; ++r2) {
      const typename E::vec x = *reinterpret_cast<const typename E::vec*>(src + r2 * (BIAS_B / 2) + lane * 16);
#pragma unroll
      for (int e = 0; e < 8; ++e) bv[8 * r2 + e] = (float)x[e] * a.sqrt_d;
    }
    return bv;
  };

  // One stage of compute from LDS buffer `buf`, keys kt0 .. kt0+BK-1.
  //
  // The KU*R tiles of the stage run as a software pipeline inside the wave: the
  // MFMA chain that produces the scores of tile t+1 is issued before the softmax
  // arithmetic of tile t, so the matrix pipe works on t+1 while the vector ALU
  // works on t.  K operands are read from LDS two tiles ahead.
  //
  // Softmax of a tile: p = exp2(acc * c - ref * c) is computed against the current
  // reference without looking for the maximum first; only when the rounded
  // probabilities of some query sum to more than 2^kLazy (which includes the
  // overflow to +inf of a query that outgrew the reference by a lot, and the very
  // first tile, whose reference is -1e30) is the reference raised to the running
  // maximum and the tile recomputed.
  auto compute_stage = [&](auto mode_tag, int kt0, int buf) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_tag)::value;
    constexpr bool PLAIN = MODE == kPlain;
    const unsigned char* st = tri_smem + buf * STAGE;
    if (!wave_active) return;
    constexpr int TS = KU * R;
    // keep words of the stage's tiles (wave-uniform loads)
    uint32_t kw[R][KU];
    if constexpr (!PLAIN) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int w = (kt0 >> 5) + u;
          kw[r][u] = __builtin_amdgcn_readfirstlane((w < a.nwords) ? reinterpret_cast<const uint32_t*>(st + OFF_KW)[r * KU + u] : 0u);
        }
    }
    auto k_operand = [&](int t, frag* kf) {
      const int u = t / R, r = t % R;
#pragma unroll
      for (int sd = 0; sd < DS; ++sd) kf[sd] = ofs.natural(st + OFF_K + (r * BK + 32 * u) * ROWB, sd);
    };
    // The bias tile does not depend on the pair row: it is converted to fp32 in
    // the raw-score domain once per stage and key tile, and then serves as the
    // accumulator init (C operand) of the first score MFMA of each of the R rows.
    f32x16 biasv[KU];
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      if constexpr (sizeof(T) == 4) biasv[u] = bias_cur[u];
      else biasv[u] = bias_from_lds(buf, u);
    }
    auto scores = [&](int t, const frag* kf) -> f32x16 {
      const int u = t / R, r = t % R;
      f32x16 sc;
      if constexpr (PLAIN) {
        sc = E::mfma(kf[0], qf[r][0], biasv[u]);
      } else {
        // Each case ends in the MFMA that defines sc, so that the bias tile is used
        // in place as an accumulator init (a select between inits copies 16 registers).
        if (MODE == kMasked) {
          // no fully masked row in the workgroup: the mask MFMA runs for every tile
          // (its operand is zero where nothing is masked) and nothing branches
          sc = E::mfma(kf[0], qf[r][0], E::mfma(kop.masked(kw[r][u]), qzero, biasv[u]));
        } else if (!flagged[r]) {
          if (kw[r][u] != 0xffffffffu)
            sc = E::mfma(kf[0], qf[r][0], E::mfma(kop.masked(kw[r][u]), qzero, biasv[u]));
          else
            sc = E::mfma(kf[0], qf[r][0], biasv[u]);
        } else {
          // a fully masked row has no bias (and a zero Q: all its scores are equal),
          // but keys past the end of a ragged last tile stay masked for it too
          asm volatile("" ::);
          sc = E::mfma(kop.masked(kw[r][u]), qzero, zero16());
          sc = E::mfma(kf[0], qf[r][0], sc);
        }
      }
#pragma unroll
      for (int sd = 1; sd < DS; ++sd) sc = E::mfma(kf[sd], qf[r][sd], sc);
      return sc;
    };

    frag kf1[DS], kf2[DS];
    k_operand(0, kf1);
    if constexpr (TS > 1) k_operand(1, kf2);
    f32x16 sc = scores(0, kf1);
#pragma unroll
    for (int t = 0; t < TS; ++t) {
      const int u = t / R, r = t % R;
      f32x16 sn;
      if (t + 1 < TS) {
#pragma unroll
        for (int sd = 0; sd < DS; ++sd) kf1[sd] = kf2[sd];
        if (t + 2 < TS) k_operand(t + 2, kf2);
        sn = scores(t + 1, kf1);
      }
      bool tile_on = true;  // a row that attends to no key of this tile adds nothing
      if constexpr (!PLAIN) tile_on = kw[r][u] != 0;
      if (tile_on) {
        // V^T rows as A operand of the second product
        frag vf[DM][PS];
#pragma unroll
        for (int mt = 0; mt < DM; ++mt)
#pragma unroll
          for (int s2 = 0; s2 < PS; ++s2) vf[mt][s2] = ofs.transposed(st + OFF_V + (r * BK + 32 * u) * ROWB, s2, mt);
        frag pf[PS];
        float ts = 0.f;
#pragma unroll
        for (int s2 = 0; s2 < PS; ++s2) {
          float p[KP];
#pragma unroll
          for (int e = 0; e < KP; ++e) p[e] = fast_exp2(__builtin_fmaf(sc[KP * s2 + e], c, -mc[r]));
          pf[s2] = E::pack(p);
          ts = row_sum<T>(pf[s2], p, ts);
        }
        if (__any(!(ts <= kLazyLimit))) {
          // some query outgrew the reference: raise it to the running maximum.
          // (The empty volatile asm keeps the compiler from executing this rare
          // path speculatively in line with the common one.)
          asm volatile("" ::);
          float mx = fmaxf(sc[0], sc[1]);
#pragma unroll
          for (int v = 2; v < 16; ++v) mx = fmaxf(mx, sc[v]);
          mx = half_max(mx);
          const float mnew = fmaxf(mref[r], mx);
          const float alpha = fast_exp2((mref[r] - mnew) * c);
          lrun[r] *= alpha;
#pragma unroll
          for (int mt = 0; mt < DM; ++mt)
#pragma unroll
            for (int v = 0; v < 16; ++v) oacc[r][mt][v] *= alpha;
          mref[r] = mnew;
          mc[r] = mnew * c;
          ts = 0.f;
#pragma unroll
          for (int s2 = 0; s2 < PS; ++s2) {
            float p[KP];
#pragma unroll
            for (int e = 0; e < KP; ++e) p[e] = fast_exp2(__builtin_fmaf(sc[KP * s2 + e], c, -mc[r]));
            pf[s2] = E::pack(p);
            ts = row_sum<T>(pf[s2], p, ts);
          }
        }
        lrun[r] += ts;
#pragma unroll
        for (int s2 = 0; s2 < PS; ++s2)
#pragma unroll
          for (int mt = 0; mt < DM; ++mt) oacc[r][mt] = E::mfma(vf[mt][s2], pf[s2], oacc[r][mt]);
      }
      if (t + 1 < TS) sc = sn;
    }
  };
  // ---- the scheduled loop: workgroups without a fully masked row ------------------------------
  // Same work as the plain stage loop above, laid out as the schedule it should run in.  A
  // wave issues in order, so everything a tile needs is asked for a whole tile ahead:
  //   * a ring of three or four 32-key stages (K rows, V rows and the waves' packed bias
  //     tiles), filled by global->LDS loads that are issued two or three stages ahead; one barrier per stage, before
  //     its last tile, publishes the next stage.  Every load in the loop is an asm statement
  //     and every wait for them is a counted one written here: a load the compiler knows of
  //     (or a register it reloads from scratch) would make it wait for everything in flight;
  //   * in the slot of tile t the wave reads the K operand of tile t+1 and the V operand of
  //     tile t from LDS, issues the P.V MFMAs of tile t-1 and the score MFMAs of tile t+1,
  //     and spreads the softmax arithmetic of tile t (in units of two scores: two fma, two
  //     exp2, a packed conversion and a row-sum step) between them;
  //   * the bias tile of the next stage enters through the matrix pipe in the last slot of a
  //     stage: its packed words are the B operand against a constant A operand that holds
  //     sqrt(d) where the contraction slot is the row's key (sqrt(32) as hi + lo parts), and
  //     the product is the accumulator init of the score MFMAs of the R rows.
  // masked_tag: the rows have masked keys (none of them is fully masked): every tile takes one
  // more MFMA, which gives the masked keys a large negative score, and the stages after the
  // last one with an attended key are left out
  auto fast_loop = [&](auto masked_tag) __attribute__((always_inline)) {
    static_assert(!FAST || (sizeof(T) == 2 && BK == 32 && R >= 2), "16-bit types, 32-key stages, two or more pair rows");
    if constexpr (FAST) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
    typedef T pair_t __attribute__((ext_vector_type(2)));
    constexpr int NS = Ring::NS, FSTAGE = Ring::FSTAGE, FOFF_V = Ring::FOFF_V, FOFF_B = Ring::FOFF_B, NLD = Ring::NLD;
    auto SB = [] { __builtin_amdgcn_sched_barrier(0); };
    const int ns = MASKED ? masks.last_live() : a.nwords;
    // A ragged last key tile: its missing keys are masked like any others in the masked loop
    // (their keep bits are clear); the plain loop adds the mask product to that stage's bias tile.
    const int tail = ring.tail;
    const uint32_t tail_word = (1u << tail) - 1u;
    const uint32_t lds0 = ring.lds0, lane16 = ring.lane16;
    auto issue_fast = [&](int boff) { ring.issue(boff, ns, wave, lane); };
    // the keep words of the stage in use and of the next one, one per pair row (wave-uniform:
    // scalar loads, issued a stage ahead of their use)
    uint32_t kwc[R], kwn[R];
    auto fetch_keep_words = [&](int stage, uint32_t* kw) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < R; ++r) kw[r] = MASKED ? uniform_word(keep_row[r], min(stage, a.nwords - 1)) : 0xffffffffu;
    };
    kop.init(perm32(jl), g);
    typename OffsetMask<T>::Queries qz;
    qz.init(split_word<T>(0.f), g);
    qzero = qz.get();
    if constexpr (MASKED) {
      fetch_keep_words(0, kwc);
      fetch_keep_words(1, kwn);
    }

    // A operand of the bias products: row m of the score tile stands for key perm32(m); half r2
    // of the packed words gives the contraction slots 8 g + e the keys 16 r2 + 8 g + e
    constexpr int NPART = D == 32 ? 2 : 1;
    constexpr int NB = 2 * NPART;
    frag bsel[2][NPART];
    {
      const T hi = (T)a.sqrt_d;
      const T part[2] = {hi, (T)(a.sqrt_d - (float)hi)};
#pragma unroll
      for (int r2 = 0; r2 < 2; ++r2)
#pragma unroll
        for (int pp = 0; pp < NPART; ++pp) {
          const int e = perm32(jl) - 16 * r2 - 8 * g;
          const uint32_t bits = (uint32_t)__builtin_bit_cast(uint16_t, part[pp]) << (16 * (e & 1));
          u32x4v w;
#pragma unroll
          for (int x = 0; x < 4; ++x) w[x] = (e >= 0 && e < 8 && (e >> 1) == x) ? bits : 0u;
          asm volatile("" : "+v"(w));  // resident: not rebuilt from the lane id at every use
          bsel[r2][pp] = __builtin_bit_cast(frag, w);
        }
    }
    const pair_t ones = {(T)1.0f, (T)1.0f};

    // absolute LDS addresses of this lane's operand reads in the stage in use (K rows as natural
    // operands, V rows through transposing reads, the wave's bias words); they move with the ring
    uint32_t ak[DS], avl[DM], avh[DM], ab;
#pragma unroll
    for (int sd = 0; sd < DS; ++sd) ak[sd] = lds0 + (uint32_t)ofs.nat[sd];
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      avl[mt] = lds0 + (uint32_t)(FOFF_V + ofs.tlo[mt]);
      avh[mt] = lds0 + (uint32_t)(FOFF_V + ofs.thi[mt]);
    }
    ab = lds0 + (uint32_t)(FOFF_B + wave * 2048) + lane16;
    auto lds_frag = [](uint32_t addr) { return *reinterpret_cast<TRI_L3 const frag*>((uintptr_t)addr); };
    auto lds_tr = [](uint32_t lo, uint32_t hi) {
      const auto x = lds_tr4(reinterpret_cast<TRI_L3 const T*>((uintptr_t)lo));
      const auto y = lds_tr4(reinterpret_cast<TRI_L3 const T*>((uintptr_t)hi));
      frag f;
#pragma unroll
      for (int e = 0; e < 4; ++e) { f[e] = x[e]; f[4 + e] = y[e]; }
      return f;
    };

    // ---- the state that moves from slot to slot ----
    f32x16 sc_cur = zero16(), bias_s = zero16();
    frag vf_prev[DM][PS], pf_prev[PS];
#pragma unroll
    for (int s2 = 0; s2 < PS; ++s2) {
      pf_prev[s2] = E::zero();
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) vf_prev[mt][s2] = E::zero();
    }

    // ---- prologue: bias tile and scores of the first tile ----
    // (a wait the compiler knows: the loads made before the loop, the Q operands among them, no
    // longer count as in flight, or it would wait for everything again where the loop first
    // uses them, in every trip)
    wait_dma_known();
    ring_sync<0>();
    if (wave_active) {
#pragma unroll
      for (int x = 0; x < NB; ++x)
        bias_s = E::mfma(bsel[x / NPART][x % NPART], lds_frag(ab + (x / NPART) * 1024), bias_s);
      if (!MASKED && tail != 0 && ns == 1) bias_s = E::mfma(kop.masked(tail_word), qzero, bias_s);
      sc_cur = bias_s;
      if constexpr (MASKED) sc_cur = E::mfma(kop.masked(kwc[0]), qzero, sc_cur);
#pragma unroll
      for (int sd = 0; sd < DS; ++sd) sc_cur = E::mfma(lds_frag(ak[sd]), qf[0][sd], sc_cur);
    }

    enum { F_B, F_PV, F_S, F_M };
    // (the loop exists twice: for waves with queries, and for the waves past the end of the pair
    // row, which only take part in the loads and barriers; one loop with the test inside would
    // make the compiler copy the state where the two cases meet)
    auto stage_loop_fast = [&](auto active_c) __attribute__((always_inline)) {
    constexpr bool ACTIVE = decltype(active_c)::value;
    // offsets of the ring: the stage in use, the one after it, the one the next loads go to
    int boff = 0;
    for (int stage = 0; stage < ns; ++stage) {
      const int boff_next = boff == (NS - 1) * FSTAGE ? 0 : boff + FSTAGE;
      const int boff_fill = boff == 0 ? (NS - 1) * FSTAGE : boff - FSTAGE;  // stage + NS - 1
      const int step_next = boff_next - boff;
      static_for<R>([&](auto r_c) __attribute__((always_inline)) {
        constexpr int r = decltype(r_c)::value;
        constexpr bool last_r = r == R - 1;
        constexpr int rn = (r + 1) % R, rp = (r + R - 1) % R;
        constexpr int NPV = PS * DM;
        constexpr int NM = DS + NPV + (last_r ? NB : 0) + (MASKED ? 1 : 0);
        constexpr int NU = 8;
        // MFMA order: the P.V products of the last tile, (the bias products,) (the key mask,) the score products
        struct Order { int kind[NM], idx[NM]; };
        constexpr Order ord = [] {
          Order o{};
          int n = 0;
          for (int i = 0; i < NPV; ++i) { o.kind[n] = F_PV; o.idx[n++] = i; }
          if (last_r) for (int i = 0; i < NB; ++i) { o.kind[n] = F_B; o.idx[n++] = i; }
          if (MASKED) { o.kind[n] = F_M; o.idx[n++] = 0; }
          for (int i = 0; i < DS; ++i) { o.kind[n] = F_S; o.idx[n++] = i; }
          return o;
        }();
        if constexpr (ACTIVE) {
          SB();
          // operand reads: K rows of the next tile, V rows of this one, (the next stage's bias words)
          const uint32_t knext = last_r ? (uint32_t)step_next : (uint32_t)(rn * 32 * ROWB);
          frag kf[DS], vf[DM][PS], bwf[2];
#pragma unroll
          for (int sd = 0; sd < DS; ++sd) kf[sd] = lds_frag(ak[sd] + knext);
#pragma unroll
          for (int mt = 0; mt < DM; ++mt)
#pragma unroll
            for (int s2 = 0; s2 < PS; ++s2)
              vf[mt][s2] = lds_tr(avl[mt] + (uint32_t)(r * 32 * ROWB + 16 * s2 * ROWB), avh[mt] + (uint32_t)(r * 32 * ROWB + 16 * s2 * ROWB));
          if constexpr (last_r) {
            bwf[0] = lds_frag(ab + (uint32_t)step_next);
            bwf[1] = lds_frag(ab + (uint32_t)step_next + 1024u);
          }
          SB();
          f32x16 sc_next, bias_next = zero16();
          frag mk;
          if constexpr (MASKED) {
            // keys operand of the next tile's mask product (the next row of this stage, or the first row of the next)
            mk = kop.masked(last_r ? kwn[0] : kwc[rn]);
          }
          uint32_t pw[NU];
          const float mcr = mc[r], l_old = lrun[r];
          float l_new = l_old;  // the running row sum with this tile's probabilities on top
          // The arithmetic of a unit is a chain (fma -> exp2 -> conversion -> row sum), and a wave
          // that issues a dependent instruction right behind its producer waits for it: the
          // chain is cut into three steps that run one piece apart, so that between two MFMAs
          // the wave converts the units of the piece before, exponentiates its own and scales
          // those of the next.
          float xs[2 * NU], ps[2 * NU];
          auto scale_unit = [&](int u) __attribute__((always_inline)) {
            xs[2 * u] = __builtin_fmaf(sc_cur[2 * u], c, -mcr);
            xs[2 * u + 1] = __builtin_fmaf(sc_cur[2 * u + 1], c, -mcr);
          };
          auto exp_unit = [&](int u) __attribute__((always_inline)) {
            ps[2 * u] = fast_exp2(xs[2 * u]);
            ps[2 * u + 1] = fast_exp2(xs[2 * u + 1]);
          };
          auto pack_unit = [&](int u) __attribute__((always_inline)) {
            const pair_t w = {(T)ps[2 * u], (T)ps[2 * u + 1]};
            pw[u] = __builtin_bit_cast(uint32_t, w);
            l_new = pair_sum(w, ones, l_new);
          };
#pragma unroll
          for (int u = 0; u < NU / NM; ++u) scale_unit(u);
          SB();
          static_for<NM>([&](auto xc) __attribute__((always_inline)) {
            constexpr int x = decltype(xc)::value;
            constexpr int kind = ord.kind[x], idx = ord.idx[x];
            if constexpr (kind == F_B) {
              bias_next = E::mfma(bsel[idx / NPART][idx % NPART], bwf[idx / NPART], bias_next);
              if constexpr (!MASKED && idx == NB - 1) {
                if (tail != 0 && stage + 2 == ns) {  // the next stage is the ragged one
                  asm volatile("" ::);
                  bias_next = E::mfma(kop.masked(tail_word), qzero, bias_next);
                }
              }
            } else if constexpr (kind == F_PV) {
              constexpr int s2 = idx / DM, mt = idx % DM;
              oacc[rp][mt] = E::mfma(vf_prev[mt][s2], pf_prev[s2], oacc[rp][mt]);
            } else if constexpr (kind == F_M) {
              sc_next = E::mfma(mk, qzero, last_r ? bias_next : bias_s);
            } else {
              if constexpr (idx == 0 && !MASKED) sc_next = E::mfma(kf[0], qf[rn][0], last_r ? bias_next : bias_s);
              else sc_next = E::mfma(kf[idx], qf[rn][idx], sc_next);
            }
            SB();
            // (the stage's bias tile stays in use past the first product on top of it: where that is its last
            // one the compiler would accumulate in place and copy all 16 registers further on, behind a wait for
            // the matrix pipe: n = 768, h = 8, d = 64 1.55 -> 1.51 ms)
            if constexpr (r == R - 2 && (kind == F_M || (kind == F_S && idx == 0))) asm volatile("" : : "v"(bias_s));
            if constexpr (x > 0) {
#pragma unroll
              for (int u = (x - 1) * NU / NM; u < x * NU / NM; ++u) pack_unit(u);
            }
#pragma unroll
            for (int u = x * NU / NM; u < (x + 1) * NU / NM; ++u) exp_unit(u);
            if constexpr (x + 1 < NM) {
#pragma unroll
              for (int u = (x + 1) * NU / NM; u < (x + 2) * NU / NM; ++u) scale_unit(u);
            } else {
#pragma unroll
              for (int u = x * NU / NM; u < (x + 1) * NU / NM; ++u) pack_unit(u);
            }
            SB();
          });
          if (__any(!(l_new - l_old <= kLazyLimit))) {
            // some query outgrew the reference: raise it to the running maximum and redo the tile
            // (the reference lives in the log2 domain only: mc = c * max)
            asm volatile("" ::);
            float mx = fmaxf(sc_cur[0], sc_cur[1]);
#pragma unroll
            for (int v = 2; v < 16; ++v) mx = fmaxf(mx, sc_cur[v]);
            mx = half_max(mx);
            // A row that attends to no key of this tile (its keep word says so; the same for all its
            // queries): every score is the mask value.  The tile then adds nothing and must not become
            // the reference: exp2(c * score - reference) would be exp2 of the rounding error of
            // two numbers of the mask value's size.  (With a reference from real scores such a
            // tile's probabilities are exactly zero and it never gets here.)
            const bool no_key = MASKED && kwc[r] == 0u;
            const float mcn = no_key ? mc[r] : fmaxf(mc[r], mx * c);
            const float alpha = fast_exp2(mc[r] - mcn);
#pragma unroll
            for (int mt = 0; mt < DM; ++mt)
#pragma unroll
              for (int v = 0; v < 16; ++v) oacc[r][mt][v] *= alpha;
            mc[r] = mcn;
            l_new = l_old * alpha;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
              const float e0 = fast_exp2(__builtin_fmaf(sc_cur[2 * u], c, -mcn));
              const float e1 = fast_exp2(__builtin_fmaf(sc_cur[2 * u + 1], c, -mcn));
              const float p0 = no_key ? 0.f : e0, p1 = no_key ? 0.f : e1;
              const pair_t w = {(T)p0, (T)p1};
              pw[u] = __builtin_bit_cast(uint32_t, w);
              l_new = pair_sum(w, ones, l_new);
            }
          }
          lrun[r] = l_new;
#pragma unroll
          for (int s2 = 0; s2 < PS; ++s2) {
            pf_prev[s2] = __builtin_bit_cast(frag, (u32x4v){pw[4 * s2], pw[4 * s2 + 1], pw[4 * s2 + 2], pw[4 * s2 + 3]});
#pragma unroll
            for (int mt = 0; mt < DM; ++mt) vf_prev[mt][s2] = vf[mt][s2];
          }
          sc_cur = sc_next;
          if constexpr (last_r) bias_s = bias_next;
        }
        if constexpr (MASKED && last_r) {
#pragma unroll
          for (int r2 = 0; r2 < R; ++r2) kwc[r2] = kwn[r2];
          fetch_keep_words(stage + 2, kwn);
        }
        // The next slot reads stage s+1: every wave's loads of it have landed (a ring of four
        // leaves one younger stage in flight), and nobody reads stage s-1 any more: its buffer
        // takes the loads issued here, a slot earlier than at the end of the stage (with two pair rows
        // and a ring of three that is two slots instead of one until they are needed: n = 768, h = 8,
        // d = 64 1.57 -> 1.55 ms; four rows, n = 1531, 3.54 -> 3.53).
        if constexpr (r == R - 2) {
          ring_sync<(NS - 3) * NLD>();
          issue_fast(boff_fill);
        }
      });
      // the ring moves on
#pragma unroll
      for (int sd = 0; sd < DS; ++sd) ak[sd] += (uint32_t)step_next;
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) {
        avl[mt] += (uint32_t)step_next;
        avh[mt] += (uint32_t)step_next;
      }
      ab += (uint32_t)step_next;
      boff = boff_next;
    }
    };
    if (wave_active) stage_loop_fast(std::true_type{});
    else stage_loop_fast(std::false_type{});
    // P.V of the last tile
    if (wave_active) {
#pragma unroll
      for (int s2 = 0; s2 < PS; ++s2)
#pragma unroll
        for (int mt = 0; mt < DM; ++mt) oacc[R - 1][mt] = E::mfma(vf_prev[mt][s2], pf_prev[s2], oacc[R - 1][mt]);
    }
    wait_dma();  // (the last prefetches are still on their way into LDS)
    }
  };

  // Stage loop over the live stages, unrolled by two for the two LDS buffers.  A
  // workgroup whose rows attend to every key runs the loop specialised for plain
  // stages; any other one runs the general loop for all of its stages (mixing the
  // two inside one loop would copy the accumulators where the versions meet).
  __syncthreads();  // key-tile bitmaps visible
  const int ntiles = a.nwords;
  auto stage_loop = [&](auto mode_tag) __attribute__((always_inline)) {
    constexpr bool PLAIN = decltype(mode_tag)::value == kPlain;
    want_keep_words = !PLAIN;
    auto next = [&](int t) { return PLAIN ? min(t, ntiles) : masks.next_live<KU>(t); };
    int t0 = next(0);
    if (!EARLY || t0 != 0) {  // (or on its way)
      if constexpr (EARLY) drop_loads();
      issue_loads(min(32 * t0, N - 1), 0);
    }
    store_loads(0);
    wait_dma();
    __syncthreads();
    while (t0 < ntiles) {
      // past the last live stage the prefetch re-reads a valid stage that nobody uses
      const int t1 = next(t0 + KU);
      issue_loads(min(32 * t1, N - 1), 1);
      compute_stage(mode_tag, 32 * t0, 0);
      store_loads(1);
      wait_dma();
      __syncthreads();
      if (t1 >= ntiles) break;
      t0 = next(t1 + KU);
      issue_loads(min(32 * t0, N - 1), 0);
      compute_stage(mode_tag, 32 * t1, 1);
      store_loads(0);
      wait_dma();
      __syncthreads();
    }
  };
  // (a last stage with fewer than KU key tiles is not plain: its missing tiles are masked)
  bool fast = false, fast_masked = false;
  if constexpr (FAST) {
    fast = ring_on && masks.all_plain();
    // (a fully masked row drops its bias and q.k: such workgroups take the general loop)
    fast_masked = ring_on && !fast && !any_flagged && masks.last_live() > 0;
  }
  if (fast) {
    if constexpr (FAST) fast_loop(std::false_type{});
  } else if (fast_masked) {
    if constexpr (FAST) fast_loop(std::true_type{});
  } else {
    if constexpr (FAST) drop_loads();
    if constexpr (!EARLY) setup_general();
    if (masks.all_plain() && ntiles % KU == 0 && (N & 31) == 0) stage_loop(std::integral_constant<int, kPlain>{});
    else if (!any_flagged) stage_loop(std::integral_constant<int, kMasked>{});
    else stage_loop(std::integral_constant<int, kGeneral>{});
  }

  if (!wave_active) return;
  float check = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = i0 + r;
    const float ltot = half_sum(lrun[r]);
    if (i >= N) continue;  // (wave-uniform; the lanes of queries past the end stay for the exchange inside the store)
    T* orow = reinterpret_cast<T*>(a.o) + (((int64_t)bh * N + i) * N) * D;
    store_rows_any<T, D, DM>(orow + (int64_t)j * D, oacc[r], 1.0f / ltot, g, j < N);
    if (g == 0 && j < N) {
      float lse = kLn2 * (mc[r] + fast_log2(ltot));
      if (flagged[r]) lse = a.neg_inf + lse;
      a.lse[((int64_t)bh * N + i) * N + j] = lse;
    }
    if constexpr (sizeof(T) == 4) {
      check = __builtin_fmaf(ltot, 0.f, check);
#pragma unroll
      for (int mt = 0; mt < DM; ++mt) check = finite_check<(D < 32 ? 8 : 16)>(oacc[r][mt], check);
    }
  }
  if constexpr (sizeof(T) == 4) {
    if (__any(!(check == 0.f))) plain_fwd<D, R>(arg_words(), bh, i0, j_wave, fresh_lane());
  }
}

}  // namespace tri
