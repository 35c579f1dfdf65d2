// The linear layers of a triangle-attention block over its pair representation (rows = b n^2, in
// the hundreds of thousands; K input channels and a few hundred outputs), forward and backward,
// with the output gate folded into the layer that reads it:
//   linear_fwd        y_p = x W_p^T + bias_p for several layers in one pass
//   gated out layer   out = (o * sigmoid(g)) W^T + bias             (linear_fwd with a gated source)
//   gate backward     do, dg from dout W                            (linear_gate_bwd, or with dW: linear_dw)
//   linear_dx         dx = sum_p dy_p W_p
//   linear_dw         dW_p = dy_p^T x, db_p = column sums of dy_p, several layers in one pass
// All of them are bound by HBM: a row is a few hundred bytes per tensor and 10^5 multiply-adds.
// The rules they share:
//   * A row's operand fragments (16 bytes: 8 consecutive channels of one row) are loaded from
//     global memory straight into registers: the MFMA's "columns" are rows of the tensor, so a
//     lane owns a row, and the eight loads of a 256-byte row hit the same cache lines.
//   * Weights pass through LDS (direct global->LDS loads, swizzled tiles, see LdsTile), shared by
//     the four waves of a workgroup, or stay there for all layers (eight waves, see ResidentPlan).
//   * Products are computed transposed (W x^T) with the weight rows in the order perm32, so that
//     a lane ends up with two runs of 8 consecutive channels of its own row: 16-byte stores.
//   * Workgroups that share rows (different output columns of the same rows) run on one XCD, next
//     to each other in time: the rows are fetched from HBM once.
// No counterpart in the reference: the linear layers around its operator are only hinted
// at by the module of reference tests/unit/test_trifast.py:152-169.
#pragma once
#include <type_traits>

#include "tri_common.hpp"
#include "tri_dispatch.hpp"
#include "tri_gate.hpp"
#include "tri_linear_args.hpp"
#include "tri_tile.hpp"

namespace tri {

// A layer's output (or output gradient) is [rows, N] or, "heads outermost", [N / hd][rows][hd]:
// the layout the attention operator reads q, k, v in (and writes dq, dk, dv in) without the
// two heads of a 128-byte line belonging to different workgroups.  hd = 0: plain.
// (hd is a multiple of 8 and divides N, so a 16-byte piece never straddles two heads.)
TRI_DEV int64_t linear_offset(int64_t row, int col, int N, int hd, int64_t rows) {
  return hd ? ((int64_t)(col / hd) * rows + row) * hd + col % hd : row * N + col;
}
// The same for a piece of a 32-column chunk that starts at col0 (wave-uniform): where heads are
// whole chunks wide (or the layer is plain) the division is a scalar one.
struct ChunkColumns {
  int64_t base;
  int pitch, col0, N, hd;
  bool uniform;
  int64_t rows;
  TRI_DEV ChunkColumns(int col0_, int N_, int hd_, int64_t rows_) : col0(col0_), N(N_), hd(hd_), uniform(hd_ % 32 == 0), rows(rows_) {
    pitch = hd ? hd : N;
    base = hd && uniform ? (int64_t)(col0 / hd) * rows * hd + col0 % hd : col0;
  }
  TRI_DEV int64_t at(int64_t row, int in_chunk) const {
    return uniform ? base + row * pitch + in_chunk : linear_offset(row, col0 + in_chunk, N, hd, rows);
  }
};

// x / v.d for x < 2^31
TRI_DEV uint32_t quotient(uint32_t x, const Divisor& v) { return v.mul == 0 ? x : __umulhi(x, v.mul) >> v.shift; }

// row of a tensor in pair order (b, i, j) for row `r` of the order the operator works in
TRI_DEV int64_t mapped_row(const RowMap& m, int64_t r) {
  if (m.by.d == 0) return r;
  const uint32_t n = m.by.d, q = quotient((uint32_t)r, m.by), j = (uint32_t)r - q * n;  // q = b n + i
  const uint32_t b = quotient(q, m.by), i = q - b * n;
  return (b * n + j) * n + i;
}

// Element offset of head row 0 of row r in the operator's layout [b, H, n, n, D] (head h: + h * plane * D)
TRI_DEV int64_t outer_row(int64_t r, const Divisor& plane, int H, int D) {
  const uint32_t b = quotient((uint32_t)r, plane);
  return ((int64_t)b * H * plane.d + ((uint32_t)r - b * plane.d)) * D;
}
// ... and of channel k (of H * D) from there; D is a power of two
TRI_DEV int64_t outer_channel(int k, uint32_t plane, int lgD) { return ((int64_t)(k >> lgD) * plane << lgD) + (k & ((1 << lgD) - 1)); }

// Which layer and which of its 32-column chunks chunk number `q` is (layers in order, each of
// ceil(n / 32) chunks; wave-uniform).
struct ChunkAt {
  int p, col0;
};
template <typename Args>
TRI_DEV ChunkAt chunk_at(const Args& a, int q) {
  int p = 0;
  while (p + 1 < a.nlayers && q >= (a.n[p] + 31) / 32) q -= (a.n[p++] + 31) / 32;
  return ChunkAt{p, 32 * q};
}

// (row block, column group) of this workgroup: the groups of one row block are consecutive slots
// of one XCD.  The launcher pads the row blocks to a multiple of 8; row_block >= blocks: no work.
TRI_DEV void rows_remap(int groups, int& row_block, int& group) {
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  group = slot % groups;
  row_block = 8 * (slot / groups) + xcd;
}

// Every LDS operation of the wave has returned, then meet the other waves.  (The fence of
// __syncthreads() would wait for the loads in flight as well.)
TRI_DEV void lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// eight consecutive channels of a gated row: o * sigmoid(g), rounded to T
template <typename T>
TRI_DEV typename Elem<T>::vec gated_piece(typename Elem<T>::vec o, typename Elem<T>::vec g) {
  typename Elem<T>::vec y;
#pragma unroll
  for (int e = 0; e < Elem<T>::VEC; ++e) {
    float s, ds;
    gate_sigmoid<T>((float)g[e], s, ds);
    y[e] = (T)((float)o[e] * s);
  }
  return y;
}

// ---------------------------------------------------------------------------------------
// y_p[r, :] = x[r, :] W_p^T + bias_p.  A workgroup takes 128 * RT rows and a run of 32-column
// chunks of the layers' outputs (up to a.chunks of them, their weights in LDS at once).  Its x
// fragments stay in registers for all of its chunks.
//
// GATED: x is o * sigmoid(g), o in the operator's layout and g [rows, K], gated on the way
// into the fragments (what the output layer of the block reads; y itself never exists).
//
// Split over the column chunks as well as the rows (one workgroup per row block did all layers
// before): 577 workgroups of 256 rows on 512 resident slots ran two rounds at n = 384, and 24
// workgroups did all the work at n = 77.
// ---------------------------------------------------------------------------------------
template <typename T, int KD, int RT, bool GATED>
__global__ __launch_bounds__(256) void linear_fwd_kernel(const LinearFwdArgs a) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using Tile = LdsTile<T, KD>;
  constexpr int KS = KD / 16;              // MFMA steps over K
  constexpr int CHUNK_B = 32 * Tile::ROWB;  // bytes of a chunk's weights
  extern __shared__ __attribute__((aligned(16))) unsigned char lin_smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cl = lane & 31, g = lane >> 5;
  int rb, grp;
  rows_remap(a.groups, rb, grp);
  const int64_t row0 = (int64_t)rb * (128 * RT) + wave * (32 * RT);
  if ((int64_t)rb * (128 * RT) >= a.rows) return;
  const int q0 = grp * a.chunks, nq = min(a.chunks, a.total_chunks - q0);

  // this workgroup's weights -> LDS (rows past the layer's last repeat it: their outputs are not stored)
  for (int q = 0; q < nq; ++q) {
    const ChunkAt at = chunk_at(a, q0 + q);
    const T* w = reinterpret_cast<const T*>(a.w[at.p]);
    const int last = a.n[at.p] - 1;
    Tile::template fill<32, 4>(lin_smem + q * CHUNK_B, [&](int r) { return w + (int64_t)min(at.col0 + r, last) * KD; }, wave, lane);
  }
  // ... and their biases (a bias loaded in front of a chunk's products waits for the stores of the chunk before:
  // gated, K = 128, 128 outputs with bias, 40000 rows 12.0 -> 11.7 us, 147456 25.4 -> 24.0; K = 64 20.1 -> 19.7)
  T* const biases = reinterpret_cast<T*>(lin_smem + nq * CHUNK_B);
  for (int q = wave; q < nq; q += 4) {
    const ChunkAt at = chunk_at(a, q0 + q);
    const T* bias = reinterpret_cast<const T*>(a.bias[at.p]);
    T value = (T)0.0f;
    if (bias && at.col0 + cl < a.n[at.p]) value = bias[at.col0 + cl];
    biases[32 * q + cl] = value;
  }
  // the rows' fragments (rows past the end repeat the last one and are not stored)
  int64_t row[RT];
  frag xf[RT][KS];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    row[t] = row0 + 32 * t + cl;
    const int64_t rr = min(row[t], a.rows - 1);
    if constexpr (GATED) {
      const T* o = reinterpret_cast<const T*>(a.o) + outer_row(rr, a.plane, a.H, a.D);
      const T* gt = reinterpret_cast<const T*>(a.g) + rr * KD;
      // Heads are 16 channels wide at least: the offset of a step's channels is wave-uniform.  The pieces
      // are gated one after the other, eight loads ahead: left to itself the compiler keeps what all of them
      // are made of (88 registers in place of 76 at K = 128, 256 in place of 120 at K = 256, and with
      // the shorter sigmoid it took a workgroup per CU from it: n = 384, 128 outputs 70 -> 90 us).
      constexpr int AHEAD = KS < 8 ? KS : 8;
      vec ov[AHEAD], gv[AHEAD];
      auto piece = [&](int s) __attribute__((always_inline)) {
        ov[s % AHEAD] = *reinterpret_cast<const vec*>(o + 8 * g + outer_channel(16 * s, a.plane.d, a.lgD));
        gv[s % AHEAD] = *reinterpret_cast<const vec*>(gt + 16 * s + 8 * g);
      };
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) piece(s);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        xf[t][s] = gated_piece<T>(ov[s % AHEAD], gv[s % AHEAD]);
        asm volatile("" : "+v"(xf[t][s]));
        if (s + AHEAD < KS) piece(s + AHEAD);
      }
    } else {
      const T* x = reinterpret_cast<const T*>(a.x) + mapped_row(a.xmap, rr) * KD;
#pragma unroll
      for (int s = 0; s < KS; ++s) xf[t][s] = *reinterpret_cast<const frag*>(x + 16 * s + 8 * g);
    }
  }
  // (a wait the compiler knows: it would otherwise put one in front of every LDS read below, and wait
  // for the stores of the chunk before with it)
  wait_dma_known();
  __syncthreads();

  OperandOffsets<T, KD> ofs;
  ofs.init(perm32(cl), lane);
  for (int q = 0; q < nq; ++q) {
    const ChunkAt at = chunk_at(a, q0 + q);
    const int N = a.n[at.p], hd = a.hd[at.p];
    T* y = reinterpret_cast<T*>(a.y[at.p]);
    const bool wide = (N % 8) == 0;
    const ChunkColumns cols(at.col0, N, hd, a.rows);
    // this lane's 16 columns: col0 + 16 half + 8 g + 0..7
    f32x16 acc[RT];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const vec bv = *reinterpret_cast<const vec*>(biases + 32 * q + 16 * half + 8 * g);
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t][8 * half + e] = (float)bv[e];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const frag wf = ofs.natural(lin_smem + q * CHUNK_B, s);
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t] = E::mfma(wf, xf[t][s], acc[t]);
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      if (row[t] >= a.rows) continue;
      const int64_t orow = mapped_row(a.ymap, row[t]);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int col = at.col0 + 16 * half + 8 * g;
        if (col >= N) continue;
        vec v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (T)acc[t][8 * half + e];
        T* dst = y + cols.at(orow, 16 * half + 8 * g);
        if (wide) {
          *reinterpret_cast<vec*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (col + e < N) dst[e] = v[e];
        }
      }
    }
  }
}

// The resident kernels (below, and for dx): one workgroup of eight waves per CU fills LDS with every
// layer's weights once, then each wave walks row tiles of its own without another barrier.  The layers are
// whole 32-column chunks in rows of one pitch (chunk q's address in row 0 and pitch stand in an
// LDS table), in multiples of four chunks, but for one layer of an even number of outputs up to 16, whose
// columns move 4 bytes at a time.
struct ResidentPlan {
  int chunks, narrow;  // whole chunks; the narrow layer, or -1; chunks = 0: not for these kernels
};
template <typename Args>
inline ResidentPlan resident_plan(const Args& a) {
  ResidentPlan plan{0, -1};
  for (int p = 0; p < a.nlayers; ++p) {
    if (a.n[p] % 32 == 0 && a.hd[p] % 32 == 0) plan.chunks += a.n[p] / 32;
    else if (a.n[p] <= 16 && a.n[p] % 2 == 0 && a.hd[p] == 0 && plan.narrow < 0) plan.narrow = p;
    else return ResidentPlan{0, -1};
  }
  return plan.chunks % 4 ? ResidentPlan{0, -1} : plan;
}
constexpr int kResidentWgs = 256, kResidentWaves = 8, kResidentLds = 160 * 1024;
struct ChunkRow {
  uint64_t base;   // byte address of the chunk in row 0
  uint32_t pitch;  // bytes from row to row
  uint32_t pad;
};
// Tiles of 32 rows: number k of a wave.  The rounds of all workgroups interleave, so that a last
// round that is not full occupies a part of every CU.
TRI_DEV int resident_tile(int k, int wave) { return (kResidentWaves * k + wave) * kResidentWgs + (int)blockIdx.x; }

// The same for many rows: bound by HBM, and by how long a workgroup that loads, multiplies and stores once
// has nothing in flight.  A wave stores a tile while the next one's rows arrive.  No store of whole
// chunks stands behind a branch, and at least four chunks follow the loads: where the paths of a loop
// differ, the compiler's waits go by the path with the fewest operations, and would wait for the
// stores.  (Lanes past the last row repeat it, values and all.)  rows = 147456, K = 128, four layers of
// 128 outputs and one of 4, launched back to back: 56 -> 45 us, 4.2 TB/s.  (The gated layer stays with the
// kernel above: 32 us with it, 33 with gated fragments here.)
constexpr int linear_fwd_resident_lds(int kd, int chunks) { return (chunks + 1) * (32 * kd * 2 + 32 * 2 + (int)sizeof(ChunkRow)); }
template <typename T, int KD>
__global__ __launch_bounds__(512, 2) void linear_fwd_resident_kernel(const LinearFwdArgs a, const ResidentPlan plan) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using Tile = LdsTile<T, KD>;
  constexpr int KS = KD / 16, CHUNK_B = 32 * Tile::ROWB;
  extern __shared__ __attribute__((aligned(16))) unsigned char lin_smem[];
  T* const biases = reinterpret_cast<T*>(lin_smem + (plan.chunks + 1) * CHUNK_B);
  ChunkRow* const table = reinterpret_cast<ChunkRow*>(biases + (plan.chunks + 1) * 32);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cl = lane & 31, g = lane >> 5;
  const int tiles = (int)((a.rows + 31) / 32);
  auto row_at = [&](int k) { return min((int64_t)min(resident_tile(k, wave), tiles - 1) * 32 + cl, a.rows - 1); };
  frag xn[KS];  // the next tile's rows
  auto load = [&](int k) __attribute__((always_inline)) {
    const T* x = reinterpret_cast<const T*>(a.x) + mapped_row(a.xmap, row_at(k)) * KD;
#pragma unroll
    for (int s = 0; s < KS; ++s) xn[s] = *reinterpret_cast<const frag*>(x + 16 * s + 8 * g);
  };
  load(0);

  int q0 = 0;
  for (int p = 0; p < a.nlayers; ++p) {
    const int N = a.n[p];
    for (int c0 = 0; c0 < N; c0 += 32) {
      const int q = p == plan.narrow ? plan.chunks : q0++;
      // (weight rows past a narrow layer's last repeat it: their outputs are not stored)
      const T* w = reinterpret_cast<const T*>(a.w[p]);
      Tile::template fill<32, kResidentWaves>(lin_smem + q * CHUNK_B, [&](int r) { return w + (int64_t)min(c0 + r, N - 1) * KD; }, wave, lane);
    }
  }
  // The biases and the table, behind every request for weights, a wave per chunk: a bias on its way into LDS has been waited for, and all
  // that was requested before it.  (The first wave did both, chunk by chunk between the requests: rows = 147456, K = 128, 17
  // chunks, four of them with a bias, 50.3 -> 44.2 us; the block in inference at n = 300 103.1 -> 99.5.)
  q0 = 0;
  for (int p = 0; p < a.nlayers; ++p) {
    const int N = a.n[p], hd = a.hd[p];
    const T* bias = reinterpret_cast<const T*>(a.bias[p]);
    for (int c0 = 0; c0 < N; c0 += 32) {
      const int q = p == plan.narrow ? plan.chunks : q0++;
      if (q % kResidentWaves != wave) continue;
      if (lane < 32) biases[32 * q + lane] = bias && c0 + lane < N ? bias[c0 + lane] : (T)0.0f;
      if (lane == 0)
        table[q] = ChunkRow{(uint64_t)(reinterpret_cast<const T*>(a.y[p]) + linear_offset(0, c0, N, hd, a.rows)), (uint32_t)((hd ? hd : N) * sizeof(T)), 0u};
    }
  }
  wait_dma_known();
  __syncthreads();

  OperandOffsets<T, KD> ofs;
  ofs.init(perm32(cl), lane);
  const int nn = plan.narrow >= 0 ? a.n[plan.narrow] : 0;
  for (int k = 0; resident_tile(k, wave) < tiles; ++k) {
    frag xf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) xf[s] = xn[s];
    load(k + 1);  // (past the last tile: its rows again, which nobody uses)
    const uint64_t orow = (uint64_t)mapped_row(a.ymap, row_at(k));
    // this lane's 16 columns of chunk q: 16 half + 8 g + 0..7
    auto product = [&](int q, vec (&v)[2]) __attribute__((always_inline)) {
      f32x16 acc;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const vec bv = *reinterpret_cast<const vec*>(biases + 32 * q + 16 * half + 8 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[8 * half + e] = (float)bv[e];
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = E::mfma(ofs.natural(lin_smem + q * CHUNK_B, s), xf[s], acc);
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[half][e] = (T)acc[8 * half + e];
    };
    int q = 0;
    do {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        vec v[2];
        product(q + u, v);
        const ChunkRow at = table[q + u];
        auto* dst = reinterpret_cast<TRI_G1 vec*>(at.base + orow * at.pitch + 16 * g);
        dst[0] = v[0];
        dst[2] = v[1];
      }
      q += 4;
    } while (q < plan.chunks);
    if (nn) {
      typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));
      vec v[2];
      product(plan.chunks, v);
      const ChunkRow at = table[plan.chunks];
      auto* dst = reinterpret_cast<TRI_G1 uint32_t*>(at.base + orow * at.pitch + 16 * g);
      const u32x4s w = __builtin_bit_cast(u32x4s, v[0]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (8 * g + 2 * e < nn) dst[e] = w[e];
    }
  }
}

// ---------------------------------------------------------------------------------------
// Backward of the gated output layer up to the gate's inputs:
//   dy = dout W (dout [rows, K], W [K, C]),  do = dy * s,  dg = dy * o * s (1 - s),  s = sigmoid(g)
// One pass: dout, o, g read, do, dg written, dy stays in fp32 registers.  The contraction runs
// over W's rows, so its fragments are transposing LDS reads of 32-column tiles of W.
// ---------------------------------------------------------------------------------------
// Fragment (contraction over the tile's rows 16 s + 8 g ..) of column perm32(lane % 32) of a
// [rows][32] tile: ds_read_tr hands lane L the column that lane group L / 4 points at, so the
// groups 1 and 2 of every 16 columns trade places (perm32 swaps bits 2 and 3).
template <typename T, int SWZ = 0>
TRI_DEV typename Elem<T>::frag tr_perm_operand(const unsigned char* base, int row0, int lane) {
  using Tile = LdsTile<T, 32, SWZ>;
  const int L = lane & 15, quad = L & 3, sq = ((quad & 1) << 1) | (quad >> 1);
  const int col = 16 * ((lane >> 4) & 1) + 4 * sq;
  const auto lo = lds_tr4(reinterpret_cast<const T*>(base + Tile::off(row0 + (L >> 2), col * 2)));
  const auto hi = lds_tr4(reinterpret_cast<const T*>(base + Tile::off(row0 + 4 + (L >> 2), col * 2)));
  typename Elem<T>::frag f;
#pragma unroll
  for (int e = 0; e < 4; ++e) { f[e] = lo[e]; f[4 + e] = hi[e]; }
  return f;
}

// CH: 32-column chunks per workgroup at most
template <typename T, int KD, int CH>
__global__ __launch_bounds__(256) void linear_gate_bwd_kernel(const LinearGateBwdArgs a) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using Tile = LdsTile<T, 32>;
  constexpr int KS = KD / 16;
  constexpr int CHUNK_B = KD * Tile::ROWB;  // a 32-column chunk of W: [KD][32]
  extern __shared__ __attribute__((aligned(16))) unsigned char lin_smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cl = lane & 31, g = lane >> 5;
  int rb, grp;
  rows_remap(a.groups, rb, grp);
  const int64_t row0 = (int64_t)rb * 128 + wave * 32;
  if ((int64_t)rb * 128 >= a.rows) return;
  const int q0 = grp * a.chunks, nq = min(a.chunks, a.C / 32 - q0);
  const T* w = reinterpret_cast<const T*>(a.w);
  for (int q = 0; q < nq; ++q)
    Tile::template fill<KD, 4>(lin_smem + q * CHUNK_B, [&](int r) { return w + (int64_t)r * a.C + 32 * (q0 + q); }, wave, lane);

  // (rows past the end repeat the last one and are not stored)
  const int64_t row = row0 + cl, rr = min(row, a.rows - 1);
  const int64_t outer = outer_row(rr, a.plane, a.H, a.D);
  frag df[KS];
  const T* d = reinterpret_cast<const T*>(a.dout) + mapped_row(a.map, rr) * KD;
#pragma unroll
  for (int s = 0; s < KS; ++s) df[s] = *reinterpret_cast<const frag*>(d + 16 * s + 8 * g);
  // Everything this lane reads is asked for before the first product: a load issued behind a
  // chunk's stores would wait for them.
  vec gv[CH][2], ov[CH][2];
  int64_t oofs[CH][2];
#pragma unroll
  for (int q = 0; q < CH; ++q)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = 32 * min(q0 + q, a.C / 32 - 1) + 16 * half + 8 * g;
      oofs[q][half] = outer + outer_channel(k, a.plane.d, a.lgD);
      gv[q][half] = *reinterpret_cast<const vec*>(reinterpret_cast<const T*>(a.g) + rr * a.C + k);
      ov[q][half] = *reinterpret_cast<const vec*>(reinterpret_cast<const T*>(a.o) + oofs[q][half]);
    }
  wait_dma_known();
  __syncthreads();

#pragma unroll
  for (int q = 0; q < CH; ++q) {
    if (q >= nq) break;
    const unsigned char* tile = lin_smem + q * CHUNK_B;
    f32x16 acc = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = E::mfma(tr_perm_operand<T>(tile, 16 * s + 8 * g, lane), df[s], acc);
    if (row >= a.rows) continue;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      vec dov, dgv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float s, ds;
        gate_sigmoid<T>((float)gv[q][half][e], s, ds);
        const float dy = acc[8 * half + e];
        dov[e] = (T)(dy * s);
        dgv[e] = (T)(dy * (float)ov[q][half][e] * ds);
      }
      *reinterpret_cast<vec*>(reinterpret_cast<T*>(a.dox) + oofs[q][half]) = dov;
      *reinterpret_cast<vec*>(reinterpret_cast<T*>(a.dg) + row * a.C + 32 * (q0 + q) + 16 * half + 8 * g) = dgv;
    }
  }
}

// ---------------------------------------------------------------------------------------
// dx[r, :] = sum over layers p of dy_p[r, :] W_p: every dy_p is read once and dx is written once
// (the BLAS library runs one product per layer and autograd adds them up, which moves dx
// through memory nine times for five layers).  A workgroup owns 128 * RT rows and all KD
// columns, accumulated in fp32 over the layers.  The layers' contraction columns pass in chunks
// of 32, two chunks ahead in registers: the rows' fragments, and the same 32 rows of W_p, which go
// to LDS one step before their use (32-column tiles, read back transposed).  For layers whose weights do
// not fit LDS together, or whose columns are no whole chunks; the others take linear_dx_resident_kernel.
// ---------------------------------------------------------------------------------------
template <typename T, int KD, int RT>
__global__ __launch_bounds__(256) void linear_dx_kernel(const LinearDxArgs a) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using Tile = LdsTile<T, 32>;
  constexpr int KB = KD / 32;
  constexpr int BLOCK_B = 32 * Tile::ROWB;  // 32 contraction rows x 32 columns of dx
  constexpr int CHUNK_B = KB * BLOCK_B;
  constexpr int PIECES = 32 * KD / 8, WC = (PIECES + 255) / 256;  // 16-byte pieces of a chunk's weights, ... per lane
  __shared__ __attribute__((aligned(16))) unsigned char ws[3 * CHUNK_B];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cl = lane & 31, g = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * (128 * RT) + wave * (32 * RT);

  int total = 0;
  for (int p = 0; p < a.nlayers; ++p) total += (a.n[p] + 31) / 32;
  int64_t row[RT], rr[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    row[t] = row0 + 32 * t + cl;
    rr[t] = min(row[t], a.rows - 1);
  }
  // chunk q: registers and LDS buffer q % 3
  frag yf[3][RT][2];
  vec wr[3][WC];
  int lp = 0, lc = 0;  // layer and first column of the chunk the next load takes
  auto load = [&](frag (&f)[RT][2], vec (&w8)[WC]) __attribute__((always_inline)) {
    const int N = a.n[lp];
    const T* w = reinterpret_cast<const T*>(a.w[lp]);
    const T* dy = reinterpret_cast<const T*>(a.dy[lp]);
    const ChunkColumns cols(lc, N, a.hd[lp], a.rows);
    // (weight rows past the layer's last repeat it: the row fragments are zero there)
#pragma unroll
    for (int x = 0; x < WC; ++x) {
      const int q = x * 256 + tid;
      if (PIECES % 256 == 0 || q < PIECES) w8[x] = *reinterpret_cast<const vec*>(w + (int64_t)min(lc + q / (KD / 8), N - 1) * KD + 8 * (q % (KD / 8)));
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int in = 16 * s + 8 * g;
        vec v = {};
        if (lc + in < N) {
          const T* src = dy + cols.at(rr[t], in);
          if ((N % 8) == 0) {
            v = *reinterpret_cast<const vec*>(src);
          } else {
            // (all loads, then the columns past the layer's last cleared: a load behind a condition of its own
            // is waited for before the next)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[lc + in + e < N ? e : 0];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = lc + in + e < N ? v[e] : (T)0.0f;
          }
        }
        f[t][s] = v;
      }
    lc += 32;
    if (lc >= N) { ++lp; lc = 0; }
  };
  auto stage = [&](int buf, const vec (&w8)[WC]) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < WC; ++x) {
      const int q = x * 256 + tid, r = q / (KD / 8), col = 8 * (q % (KD / 8));
      if (PIECES % 256 == 0 || q < PIECES) *reinterpret_cast<vec*>(ws + buf * CHUNK_B + (col / 32) * BLOCK_B + Tile::off(r, (col % 32) * 2)) = w8[x];
    }
  };

  f32x16 acc[RT][KB];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) acc[t][kb] = zero16();

  load(yf[0], wr[0]);
  if (total > 1) load(yf[1], wr[1]);
  stage(0, wr[0]);
  lds_sync();
  auto step = [&](int q, auto which) __attribute__((always_inline)) {
    constexpr int buf = decltype(which)::value;
    if (q + 2 < total) load(yf[(buf + 2) % 3], wr[(buf + 2) % 3]);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const frag wf = tr_perm_operand<T>(ws + buf * CHUNK_B + kb * BLOCK_B, 16 * s + 8 * g, lane);
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t][kb] = E::mfma(wf, yf[buf][t][s], acc[t][kb]);
      }
    // (the buffer of chunk q + 1 was read in step q - 2, which every wave has left)
    if (q + 1 < total) stage((buf + 1) % 3, wr[(buf + 1) % 3]);
    lds_sync();
  };
  for (int q = 0; q < total; q += 3) {
    step(q, std::integral_constant<int, 0>{});
    if (q + 1 < total) step(q + 1, std::integral_constant<int, 1>{});
    if (q + 2 < total) step(q + 2, std::integral_constant<int, 2>{});
  }

  T* dx = reinterpret_cast<T*>(a.dx);
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    if (row[t] >= a.rows) continue;
    T* dst = dx + mapped_row(a.map, row[t]) * KD;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        vec v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (T)acc[t][kb][8 * half + e];
        *reinterpret_cast<vec*>(dst + 32 * kb + 16 * half + 8 * g) = v;
      }
  }
}

// The same with every layer's weights resident in LDS (see ResidentPlan): the row fragments of four
// chunks at a time go straight to registers, the next four in flight under the products.  No load
// stands behind a branch that some rounds do not take, but for the narrow layer's (see
// linear_fwd_resident_kernel).  Bound by HBM.  rows = 147456, K = 128, four layers of 128 outputs and one
// of 4, launched back to back: 56 -> 38 us, 5.0 TB/s (in the kernel above each of a narrow layer's columns was a
// load of its own that was waited for, and 577 workgroups shared 512 places).
constexpr int linear_dx_lds(int kd, int chunks) { return (chunks + 1) * (32 * kd * 2 + (int)sizeof(ChunkRow)); }

template <typename T, int KD>
__global__ __launch_bounds__(512, 2) void linear_dx_resident_kernel(const LinearDxArgs a, const ResidentPlan plan) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using Tile = LdsTile<T, 32>;
  typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));
  constexpr int KB = KD / 32, U = 4;
  constexpr int BLOCK_B = 32 * Tile::ROWB, CHUNK_B = KB * BLOCK_B;
  extern __shared__ __attribute__((aligned(16))) unsigned char lin_smem[];
  ChunkRow* const table = reinterpret_cast<ChunkRow*>(lin_smem + (plan.chunks + 1) * CHUNK_B);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cl = lane & 31, g = lane >> 5;
  int q0 = 0;
  for (int p = 0; p < a.nlayers; ++p) {
    const int N = a.n[p], hd = a.hd[p];
    for (int c0 = 0; c0 < N; c0 += 32) {
      const int q = p == plan.narrow ? plan.chunks : q0++;
      // (weight rows past a narrow layer's last repeat it: the row fragments are zero there)
      const T* w = reinterpret_cast<const T*>(a.w[p]);
      for (int gi = wave; gi < 2 * KB; gi += 8) {
        const int r = 16 * (gi & 1) + lane / 4, c = (lane % 4) ^ Tile::swz(r);
        const T* src = w + (int64_t)min(c0 + r, N - 1) * KD + 32 * (gi >> 1) + 8 * c;
        __builtin_amdgcn_global_load_lds((const TRI_G1 void*)src, (TRI_L3 void*)(lin_smem + q * CHUNK_B + gi * 1024), 16, 0, 0);
      }
      if (threadIdx.x == 0)
        table[q] = ChunkRow{(uint64_t)(reinterpret_cast<const T*>(a.dy[p]) + linear_offset(0, c0, N, hd, a.rows)), (uint32_t)((hd ? hd : N) * sizeof(T)), 0u};
    }
  }
  wait_dma_known();
  __syncthreads();

  const int tiles = (int)((a.rows + 31) / 32), quads = plan.chunks / U;
  auto row_at = [&](int k) { return min((int64_t)min(resident_tile(k, wave), tiles - 1) * 32 + cl, a.rows - 1); };
  const int nn = plan.narrow >= 0 ? a.n[plan.narrow] : 0;
  vec yf[2][U][2];
  u32x4s nf[2];
  // the quad the next load takes (past the last tile: its rows again, which nobody uses)
  int lk = 0, lq = 0;
  auto load = [&](vec (&f)[U][2], u32x4s& narrow) __attribute__((always_inline)) {
    const uint64_t row = (uint64_t)row_at(lk);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const ChunkRow at = table[U * lq + u];
      const auto* src = reinterpret_cast<TRI_G1 const vec*>(at.base + (row & 0xffffffffu) * at.pitch + 16 * g);
      f[u][0] = src[0];
      f[u][1] = src[2];
    }
    if (++lq < quads) return;
    lq = 0;
    ++lk;
    if (nn) {
      const ChunkRow at = table[plan.chunks];
      const auto* src = reinterpret_cast<TRI_G1 const uint32_t*>(at.base + (row & 0xffffffffu) * at.pitch);
#pragma unroll
      for (int e = 0; e < 4; ++e) narrow[e] = src[8 * g + 2 * e < nn ? 4 * g + e : 0];
    }
  };
  load(yf[0], nf[0]);

  f32x16 acc[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) acc[kb] = zero16();
  int k = 0, q = 0;  // the quad the next products take
  T* dx = reinterpret_cast<T*>(a.dx);
  auto step = [&](auto which) __attribute__((always_inline)) {
    constexpr int set = decltype(which)::value;
    load(yf[set ^ 1], nf[set ^ 1]);
    const unsigned char* tile = lin_smem + U * q * CHUNK_B;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
          acc[kb] = E::mfma(tr_perm_operand<T>(tile + u * CHUNK_B + kb * BLOCK_B, 16 * s + 8 * g, lane), __builtin_bit_cast(frag, yf[set][u][s]), acc[kb]);
    if (++q < quads) return;
    if (nn) {
      u32x4s v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = 8 * g + 2 * e < nn ? nf[set][e] : 0u;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        acc[kb] = E::mfma(tr_perm_operand<T>(lin_smem + plan.chunks * CHUNK_B + kb * BLOCK_B, 8 * g, lane), __builtin_bit_cast(frag, v), acc[kb]);
    }
    const int64_t row = (int64_t)resident_tile(k, wave) * 32 + cl;
    if (resident_tile(k, wave) < tiles && row < a.rows) {
      T* dst = dx + mapped_row(a.map, row) * KD;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          vec v;
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (T)acc[kb][8 * half + e];
          *reinterpret_cast<vec*>(dst + 32 * kb + 16 * half + 8 * g) = v;
        }
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) acc[kb] = zero16();
    q = 0;
    ++k;
  };
  while (resident_tile(k, wave) < tiles) {
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
  }
}

// ---------------------------------------------------------------------------------------
// dW_p[n, k] = sum over r of dy_p[r, n] x[r, k], and on request db_p[n] = sum over r of dy_p[r, n].
// The contraction runs over the long dimension and the result is tiny, which is the one shape of
// the block's linear layers that a BLAS library serves badly (one or two workgroups walk all the
// rows: 1.7 ms per layer at rows = 2^20, K = N = 128).  Here the rows are split into chunks,
// one workgroup per (chunk, group of four 32-output blocks of the layers): it streams its rows of
// dy and x through a ring of LDS stages of 64 rows (both operands have the contraction index as
// their memory row, so both are read back transposed, ds_read_tr), keeps its part of dW in fp32
// accumulators, and writes it as an fp32 partial; a second kernel adds the partials of all layers
// in a fixed order (deterministic, no atomics) and rounds once.
//
// Eight waves: waves 0-3 take the first 32 rows of a stage, 4-7 the other 32, wave w the outputs of
// block w % 4 and all K columns; the halves are added through LDS at the end.  One workgroup fills
// a CU (two at K <= 64), so a launch writes a third of the partials that three workgroups of four
// waves would.  A wave loads its own dy tile and a quarter of its half's x tile, straight into LDS:
// nothing that is in flight is in registers.  The ring is as deep as the blocks of the group leave room.
//
// A layer of up to 16 outputs that would open a group for itself (the four biases next to four
// layers of 128 outputs) rides in the first group, each of its waves taking one K block of it in
// four: as a group of its own it read all of x for 3 % of the work.
//
// Bound by HBM.  rows = 147456, K = 128, four layers of 128 outputs and one of 4: 80 -> 51 us, 3.9
// TB/s of dy, x and partials (three workgroups of four waves per CU with padded tiles filled through
// registers, the four outputs a group: 61 % of its LDS cycles were bank conflicts); gated, one layer: 42
// -> 33 us; the sum of the partials 10.5 -> 6.3 us, each.  One layer alone, 2^20 rows: K = 256, 128
// outputs 215 -> 160 us, K = 128 123 -> 104, 8 outputs 64 -> 55, 3 outputs 101 -> 82 (see kDwWords).
//
// kDwGated: x is o * sigmoid(g) (see linear_fwd); o and g land in LDS and each wave gates the pieces
// it loaded before the stage is handed over.  kDwGateBwd: the gate's backward (linear_gate_bwd) from the
// same stages, which hold all it reads: dy = dout W for the rows of the stage, W resident, do and dg
// stored, and the gated rows written over o for the weight gradient.  rows = 147456, K = 128, 128
// outputs, with the sum of the partials: 44 us, 65 as two launches.
//
// kDwWords: launches with a layer (but a riding one) whose rows of dy are no whole 16-byte pieces, see
// words_log2.  A kernel of its own: with the choice in the plain one every launch paid for it (K = 64, 4096
// rows, 128 outputs 19.9 us alone, 21.6 with it).  Loaded through registers instead, with a wait for
// everything in flight in every stage, 3 outputs at K = 128 and 2^20 rows took 141 us in place of 82, and four layers
// of 96 outputs and one of 3, 147456 rows, 84 in place of 56.
// ---------------------------------------------------------------------------------------
constexpr int kDwPlain = 0, kDwGated = 1, kDwGateBwd = 2, kDwWords = 3;
template <typename T, int KD, int MODE>
struct LinearDwShape {
  static constexpr bool GATED = MODE == kDwGated || MODE == kDwGateBwd, FUSED = MODE == kDwGateBwd;
  static constexpr int PER_CU = FUSED ? 1 : kLinearDwPerCu<KD>;
  static constexpr int XB = 32 * KD * (int)sizeof(T), YB = 32 * 32 * (int)sizeof(T);  // x tile of a half, dy tile of a wave
  static constexpr int XP = XB / 1024;           // 1 KiB loads of an x tile, shared by the four waves of the half
  static constexpr int XN = (XP + 3) / 4;        // ... per wave (a wave without one loads into `DUMP`)
  static constexpr int OFF_G = 2 * XB, OFF_Y = (GATED ? 4 : 2) * XB;
  static constexpr bool RIDER = !GATED && KD <= 128;  // (the gated layer comes alone)
  static constexpr int RB = 32 * kLinearDwRider * (int)sizeof(T);  // dy tile of a riding layer, of a half
  static constexpr int LDS = 160 * 1024 / PER_CU, DUMP = XP % 4 ? LDS - 1024 : LDS;
  // loads per wave and stage: of x, of dy (16 or, where its rows keep only 4-byte alignment, 4 bytes per lane)
  static constexpr int X_LOADS = (GATED ? 2 : 1) * XN, Y_LOADS = 2, Y4_LOADS = 8;
  static constexpr int MOST = 6;  // stages of a ring, at least two: four blocks with a riding layer, or of wide tiles
  static_assert(YB == kLinearDwTile && 2 * (OFF_Y + 8 * YB + (RIDER ? 2 * RB : 0)) + (FUSED ? 128 * KD * (int)sizeof(T) : 0) <= DUMP, "two stages");
  static_assert(MODE != kDwWords || 2 * (OFF_Y + 8 * kLinearDwWideTile) <= DUMP, "two stages of wide tiles");
};

// 16 (or 4) bytes per lane into LDS at dst + the lane's piece; unseen by the compiler (see StageRing)
TRI_DEV void dma16(uint32_t dst, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(dst), "v"(src) : "memory", "m0");
}
TRI_DEV void dma4(uint32_t dst, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(dst), "v"(src) : "memory", "m0");
}
// 2 bytes per lane, 4 bytes apart in LDS, the upper two of them zero
TRI_DEV void dma2(uint32_t dst, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, off" : : "s"(dst), "v"(src) : "memory", "m0");
}
// wait until at most n (wave-uniform) loads are in flight; the count is part of the instruction
template <int LO, int HI>
TRI_DEV void wait_loads(int n) {
  if constexpr (LO == HI) {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LO) : "memory");
  } else {
    constexpr int mid = (LO + HI + 1) / 2;
    if (n >= mid) wait_loads<mid, HI>(n);
    else wait_loads<LO, mid - 1>(n);
  }
}

// the two halves of a transposing operand read
template <typename T>
TRI_DEV typename Elem<T>::frag tr_pair(const unsigned char* p_lo, const unsigned char* p_hi) {
  const auto lo = lds_tr4(reinterpret_cast<const T*>(p_lo));
  const auto hi = lds_tr4(reinterpret_cast<const T*>(p_hi));
  typename Elem<T>::frag f;
#pragma unroll
  for (int e = 0; e < 4; ++e) { f[e] = lo[e]; f[4 + e] = hi[e]; }
  return f;
}

// Rows of dy of an odd number of outputs start at any 2 bytes: they are loaded one output per lane and lie in LDS as
// one word per output, the block's outputs rounded up to a power of two per row (the words past the
// layer's last hold its last again).  Blocks of a few outputs of any number that is not a multiple of 8 take the same way:
// fewer loads than 4 bytes at a time for all 32 columns.
TRI_DEV int words_log2(int outputs) { return 32 - __builtin_clz((uint32_t)max(min(outputs, 32), 2) - 1u); }

template <typename T, int KD, int MODE>
__global__ __launch_bounds__(512, (2 * LinearDwShape<T, KD, MODE>::PER_CU)) void linear_dw_kernel(const LinearDwArgs a) {
  using E = Elem<T>;
  using frag = typename E::frag;
  using vec = typename E::vec;
  using S = LinearDwShape<T, KD, MODE>;
  constexpr bool GATED = S::GATED, FUSED = S::FUSED;
  using XTile = LdsTile<T, KD>;
  using YTile = LdsTile<T, 32>;
  using RTile = LdsTile<T, kLinearDwRider>;
  constexpr int XN = S::XN;
  constexpr int KB = KD / 32, KE = (KB + 4) / 4;  // K blocks; ... and the bias sums of a riding layer, per wave
  extern __shared__ __attribute__((aligned(16))) unsigned char lin_smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int half = wave >> 2, wc = wave & 3;
  const int g = lane >> 5;
  int chunk, grp;
  rows_remap(a.groups, chunk, grp);
  if (chunk >= a.chunks) return;
  // this wave's block: layer p, outputs col0 .. (not live: there is none)
  int p = 0, col0 = 0, blocks_here = -4 * grp;  // (blocks_here: of this group)
  bool live = true;
  {
    int at = -1, left = 4 * grp + wc;
    for (int l = 0; l < a.nlayers; ++l) {
      if (l == a.rider) continue;
      const int blocks = (a.n[l] + 31) / 32;
      if (at < 0) { p = l; col0 = 32 * min(left, blocks - 1); }
      if (at < 0 && left < blocks) at = l;
      left -= blocks;
      blocks_here += blocks;
    }
    live = at >= 0;
  }
  blocks_here = min(blocks_here, 4);
  const int N = a.n[p];
  const bool rides = S::RIDER && a.rider >= 0 && grp == 0;
  const int64_t r_begin = (int64_t)chunk * a.rows_per_chunk;
  const int64_t r_end = min(a.rows, r_begin + a.rows_per_chunk);
  const int steps = (int)((r_end - r_begin + 63) / 64);
  // rows of dy that keep 4- or 2-byte alignment only: loaded 4 bytes at a time, or one output per lane (see words_log2)
  const bool words = MODE == kDwWords && N % 8 != 0 && (N % 2 != 0 || N - col0 <= kLinearDwRider);
  const bool even = MODE == kDwWords && N % 8 != 0 && !words;

  // where this lane's pieces of the tiles lie: tile row and address in row 0
  const T* yg = reinterpret_cast<const T*>(a.dy[p]);
  const int y_pitch = a.hd[p] ? a.hd[p] : N;
  int xr[XN], rr = 0;
  const T *xp[XN], *gp[XN], *rp = nullptr;
  bool own[XN];  // (wave-uniform)
#pragma unroll
  for (int x = 0; x < XN; ++x) {
    own[x] = 4 * x + wc < S::XP;
    const int piece = min(4 * x + wc, S::XP - 1) * 64 + lane;
    xr[x] = piece / XTile::CPR;
    const int col = 8 * ((piece % XTile::CPR) ^ XTile::swz(xr[x]));
    xp[x] = reinterpret_cast<const T*>(a.x) + (GATED ? outer_channel(col, a.plane.d, a.lgD) : col);
    gp[x] = GATED ? reinterpret_cast<const T*>(a.g) + col : nullptr;
  }
  // (the second 16 rows of a dy tile have the swizzle of the first)
  const int yr = lane / 4, ycol = col0 + 8 * ((lane % 4) ^ YTile::swz(yr));
  // (columns past the layer's last: the block's first again, their outputs are not stored)
  const T* yp = yg + linear_offset(0, ycol < N ? ycol : col0, N, a.hd[p], a.rows);
  const int rN = rides ? a.n[a.rider] : 0;
  const int r_pitch = rides && a.hd[a.rider] ? a.hd[a.rider] : rN;
  if (rides) {
    const int piece = wc * 64 + lane;  // of 4 bytes
    rr = piece / (kLinearDwRider / 2);
    const int in = piece % (kLinearDwRider / 2), col = 8 * ((in / 4) ^ RTile::swz(rr)) + 2 * (in % 4);
    rp = reinterpret_cast<const T*>(a.dy[a.rider]) + linear_offset(0, col < rN ? col : 0, rN, a.hd[a.rider], a.rows);
  }
  // a stage: the x tiles of the two halves (o, then g), the dy tiles of their blocks, those of a riding layer
  const int yb = MODE == kDwWords ? a.y_tile : S::YB;
  const int off_y = S::OFF_Y + (half * blocks_here + wc) * yb;
  const int off_r = S::OFF_Y + 2 * blocks_here * yb + half * S::RB;
  const int stage = S::OFF_Y + 2 * blocks_here * yb + (rides ? 2 * S::RB : 0);
  const int lw = words ? words_log2(N - col0) : 0;
  // (the gate's backward: W, [N][32] tiles of the K blocks, in front of the ring)
  const int ring = FUSED ? N * KD * (int)sizeof(T) : 0;
  const int depth = min((S::DUMP - ring) / stage, S::MOST), end = ring + depth * stage;
  const int in_flight = (depth - 2) * (S::X_LOADS + (!live ? 0 : words ? 1 << (lw - 1) : even ? S::Y4_LOADS : S::Y_LOADS) + (rides ? 1 : 0));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(TRI_L3 const unsigned char*)lin_smem;
  auto uni = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };

  // ask for stage s (rows past the end: the last one again) into the ring buffer at `boff`
  auto issue = [&](int s, uint32_t boff, auto words_tag) __attribute__((always_inline)) {
    constexpr bool WORDS = decltype(words_tag)::value;
    const int64_t first = r_begin + 64 * (int64_t)s + 32 * half, last = r_end - 1;
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const int64_t r = min(first + xr[x], last);
      const uint32_t at = own[x] ? boff + half * S::XB + (4 * x + wc) * 1024 : S::DUMP;
      if constexpr (GATED) {
        dma16(uni(lds0 + at), xp[x] + outer_row(r, a.plane, a.H, a.D));
        dma16(uni(lds0 + (own[x] ? at + S::OFF_G : at)), gp[x] + r * KD);
      } else {
        dma16(uni(lds0 + at), xp[x] + mapped_row(a.xmap, r) * KD);
      }
    }
    const uint32_t ybuf = boff + off_y;
    if (!live) {
      // (nobody reads its tile)
    } else if (!WORDS && even) {
      int ln = lane;
      asm volatile("" : "+v"(ln));  // (what follows from the lane is worked out here, not kept in registers)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int row = 4 * t + ln / 16, col = col0 + 8 * ((ln % 16 / 4) ^ YTile::swz(row)) + 2 * (ln % 4);
        dma4(uni(lds0 + ybuf + t * 256), yg + mapped_row(a.ymap, min(first + row, last)) * N + (col < N ? col : col0));
      }
    } else if (!WORDS) {
#pragma unroll
      for (int t = 0; t < 2; ++t) dma16(uni(lds0 + ybuf + t * 1024), yp + mapped_row(a.ymap, min(first + 16 * t + yr, last)) * y_pitch);
    } else {
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int col = min(col0 + (ln & ((1 << lw) - 1)), N - 1);
#pragma unroll 1
      for (int t = 0; t < 32; t += 64 >> lw) dma2(uni(lds0 + ybuf + (t << lw) * 4), yg + mapped_row(a.ymap, min(first + t + (ln >> lw), last)) * N + col);
    }
    if (rides) dma4(uni(lds0 + boff + off_r + wc * 256), rp + mapped_row(a.ymap, min(first + rr, last)) * r_pitch);
  };
  // what this wave loaded of stage s has landed: gate it, and clear rows past the end
  auto finish = [&](int s, uint32_t boff, auto words_tag) __attribute__((always_inline)) {
    constexpr bool WORDS = decltype(words_tag)::value;
    unsigned char* xbuf = lin_smem + boff + half * S::XB + lane * 16;
    if constexpr (GATED && !FUSED) {
#pragma unroll
      for (int x = 0; x < XN; ++x) {
        if (!own[x]) continue;
        vec* o = reinterpret_cast<vec*>(xbuf + (4 * x + wc) * 1024);
        *o = gated_piece<T>(*o, *reinterpret_cast<const vec*>(xbuf + S::OFF_G + (4 * x + wc) * 1024));
      }
    }
    const int64_t first = r_begin + 64 * (int64_t)s + 32 * half;
    if (first + 32 <= r_end) return;
    const vec none = {};
#pragma unroll
    for (int x = 0; x < XN; ++x)
      if (own[x] && first + xr[x] >= r_end) {
        *reinterpret_cast<vec*>(xbuf + (4 * x + wc) * 1024) = none;
        if constexpr (FUSED) *reinterpret_cast<vec*>(xbuf + S::OFF_G + (4 * x + wc) * 1024) = none;
      }
    if (live && WORDS) {
#pragma unroll 1
      for (int t = 0; t < 32; t += 64 >> lw)
        if (first + t + (lane >> lw) >= r_end) *reinterpret_cast<uint32_t*>(lin_smem + boff + off_y + ((t << lw) + lane) * 4) = 0u;
    } else if (live) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (first + 16 * t + yr >= r_end) *reinterpret_cast<vec*>(lin_smem + boff + off_y + t * 1024 + lane * 16) = none;
    }
    if (rides && first + rr >= r_end) *reinterpret_cast<uint32_t*>(lin_smem + boff + off_r + wc * 256 + lane * 4) = 0u;
  };

  f32x16 acc[KB], racc[KE];
#pragma unroll
  for (int i = 0; i < KB; ++i) acc[i] = zero16();
#pragma unroll
  for (int i = 0; i < KE; ++i) racc[i] = zero16();
  // the bias gradient, the column sums of dy, rides along as one more product: dy^T times ones
  const bool sums = a.off_b[p] >= 0, rsums = rides && a.off_b[a.rider < 0 ? 0 : a.rider] >= 0;
  const frag ones = E::osplat(1.0f);
  f32x16 bacc = zero16();

  OperandOffsets<T, KD> xo;
  OperandOffsets<T, 32> yo;
  xo.init(0, lane);
  yo.init(lane & 31, lane);
  // a riding layer: its own tile, and the K blocks of this wave: wc, wc + 4, .. (block KB: its column sums)
  const int r16lo = RTile::off(8 * g + ((lane & 15) >> 2), 8 * (lane & 3)), r16hi = RTile::off(8 * g + 4 + ((lane & 15) >> 2), 8 * (lane & 3));
  int rlo[KE], rhi[KE];
#pragma unroll
  for (int i = 0; i < KE; ++i) {
    const int row = 8 * g + ((lane & 15) >> 2), col = 32 * min(wc + 4 * i, KB - 1) + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    rlo[i] = XTile::off(row, col * 2);
    rhi[i] = XTile::off(row + 4, col * 2);
  }
  auto words_frag = [&](const unsigned char* yt, int s2) __attribute__((always_inline)) {
    typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const uint32_t* w = reinterpret_cast<const uint32_t*>(yt) + ((16 * s2 + 8 * (ln >> 5)) << lw) + (ln & 31 & ((1 << lw) - 1));
    u32x4s v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = w[(2 * e) << lw] | w[(2 * e + 1) << lw] << 16;
    return __builtin_bit_cast(frag, v);
  };
  auto compute = [&](uint32_t boff, auto words_tag) __attribute__((always_inline)) {
    const unsigned char *xt = lin_smem + boff + half * S::XB, *yt = lin_smem + boff + off_y;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      if (live) {
        // A: dy^T (output row n in the lane, 8 memory rows as contraction slots); B: x^T
        frag af;
        if constexpr (decltype(words_tag)::value) af = words_frag(yt, s2);
        else af = yo.transposed(yt, s2, 0);
        if (sums) bacc = E::mfma(af, ones, bacc);
#pragma unroll
        for (int i = 0; i < KB; ++i) acc[i] = E::mfma(af, xo.transposed(xt, s2, i), acc[i]);
      }
      if (rides) {
        // (16 outputs: lanes 16-31 hold them again and are not stored)
        const unsigned char* rt = lin_smem + boff + off_r + 16 * s2 * RTile::ROWB;
        const frag rf = tr_pair<T>(rt + r16lo, rt + r16hi);
#pragma unroll
        for (int i = 0; i < KE; ++i) {
          const unsigned char* xs = xt + 16 * s2 * XTile::ROWB;
          if (wc + 4 * i < KB) racc[i] = E::mfma(rf, tr_pair<T>(xs + rlo[i], xs + rhi[i]), racc[i]);
          else if (wc + 4 * i == KB && rsums) racc[i] = E::mfma(rf, ones, racc[i]);
        }
      }
    }
  };

  // the gate's backward of stage s: dy = dout W for this half's rows and K block wc, and with it do, dg and,
  // in place of o, the gated row
  auto gate_bwd = [&](int s, uint32_t boff) __attribute__((always_inline)) {
    if (wc >= KB) return;
    f32x16 dy = zero16();
    const unsigned char* wt = lin_smem + wc * N * YTile::ROWB;
    for (int q = 0; q < blocks_here; ++q) {
      const unsigned char* tile = lin_smem + boff + S::OFF_Y + (half * blocks_here + q) * yb;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) dy = E::mfma(tr_perm_operand<T>(wt, 32 * q + 16 * s2 + 8 * g, lane), yo.natural(tile, s2), dy);
    }
    const int64_t row = r_begin + 64 * (int64_t)s + 32 * half + (lane & 31);
    T* dox = reinterpret_cast<T*>(a.dox) + outer_row(row, a.plane, a.H, a.D) + 8 * g;
    T* dg = reinterpret_cast<T*>(a.dg) + row * KD + 32 * wc + 8 * g;
    unsigned char* xt = lin_smem + boff + half * S::XB;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      vec* const o = reinterpret_cast<vec*>(xt + XTile::off(lane & 31, 2 * (32 * wc + 16 * h2 + 8 * g)));
      const vec ov = *o, gv = *reinterpret_cast<const vec*>(reinterpret_cast<unsigned char*>(o) + S::OFF_G);
      vec yv, dov, dgv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float sg, ds;
        gate_sigmoid<T>((float)gv[e], sg, ds);
        yv[e] = (T)((float)ov[e] * sg);
        dov[e] = (T)(dy[8 * h2 + e] * sg);
        dgv[e] = (T)(dy[8 * h2 + e] * (float)ov[e] * ds);
      }
      *o = yv;
      if (row < r_end) {
        *reinterpret_cast<vec*>(dox + outer_channel(32 * wc + 16 * h2, a.plane.d, a.lgD)) = dov;
        *reinterpret_cast<vec*>(dg + 16 * h2) = dgv;
      }
    }
  };
  if constexpr (FUSED) {
    const T* w = reinterpret_cast<const T*>(a.gw);
    for (int gi = wave; gi < KB * (N / 16); gi += 8) {
      const int kb = gi / (N / 16), part = gi % (N / 16), r = 16 * part + lane / 4;
      dma16(uni(lds0 + gi * 1024), w + (int64_t)r * KD + 32 * kb + 8 * ((lane % 4) ^ YTile::swz(r)));
    }
  }

  auto walk = [&](auto words_tag) __attribute__((always_inline)) {
    for (int s = 0; s < min(depth - 1, steps); ++s) issue(s, ring + s * stage, words_tag);
    int now = ring, next = end - stage;  // ring buffers of stages s and s + depth - 1
    for (int s = 0; s < steps; ++s) {
      // stage s of this wave has landed once at most the stages s + 1 .. s + depth - 2 are in flight
      // (and the four stores of each of the depth - 1 stages before this one, which are younger than stage s: loads and
      // stores leave the counter in one order, see ring_sync; gate_bwd's pieces of a row are four stores of the widest kind, no
      // fewer instructions can make them)
      const int stores = FUSED && wc < KB ? 4 * min(s, depth - 1) : 0;
      wait_loads<0, 40>(s + depth - 1 > steps ? 0 : in_flight + stores);
      finish(s, now, words_tag);
      lds_sync();
      // (buffer `next` held stage s - 1, which every wave has read)
      if (s + depth - 1 < steps) issue(s + depth - 1, next, words_tag);
      if constexpr (FUSED) {
        gate_bwd(s, now);
        lds_sync();
      }
      compute(now, words_tag);
      now = now + stage == end ? ring : now + stage;
      next = next + stage == end ? ring : next + stage;
    }
  };
  // (a loop of its own for the waves whose dy lies in words: with the choice inside the loop 2^20 rows, K = 128, 3 outputs
  // take 92 us in place of 85)
  if (words) walk(std::integral_constant<bool, MODE == kDwWords>{});
  else walk(std::false_type{});

  // the second half's sums -> LDS -> added to the first half's
  auto fold = [&](f32x16* set, int count, int slot) __attribute__((always_inline)) {
    float* at = reinterpret_cast<float*>(lin_smem) + ((slot * 4 + wc) * 16) * 64 + lane;
#pragma unroll
    for (int i = 0; i < count; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float* f = at + (i * 4 * 16 + v) * 64;
        if (half) *f = set[i][v];
        else set[i][v] += *f;
      }
  };
  lds_sync();
  if (half) fold(acc, KB, 0);
  lds_sync();
  if (!half) fold(acc, KB, 0);
  lds_sync();
  if (half) {
    fold(&bacc, 1, 0);
    if (S::RIDER) fold(racc, KE, 1);
  }
  lds_sync();
  if (half) return;
  fold(&bacc, 1, 0);
  if (S::RIDER) fold(racc, KE, 1);

  // partial [chunk][layer's n][k]: the lane holds column k = 32 kb + lane % 32 and rows
  // n = 8 q + 4 g + e of the block
  float* part = a.part + (int64_t)chunk * a.total;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int in = 8 * (v / 4) + 4 * g + (v % 4), n = col0 + in;
    if (live && n < N) {
      // (every column of the sums' product holds the same values: lanes 0 and 32 store theirs)
      if (sums && (lane & 31) == 0) part[a.off_b[p] + n] = bacc[v];
#pragma unroll
      for (int i = 0; i < KB; ++i) part[a.off_w[p] + (int64_t)n * KD + 32 * i + (lane & 31)] = acc[i][v];
    }
    if (rides && in < rN) {
#pragma unroll
      for (int i = 0; i < KE; ++i) {
        if (wc + 4 * i == KB && rsums && (lane & 31) == 0) part[a.off_b[a.rider] + in] = racc[i][v];
        if (wc + 4 * i < KB) part[a.off_w[a.rider] + (int64_t)in * KD + 32 * (wc + 4 * i) + (lane & 31)] = racc[i][v];
      }
    }
  }
}

// dW, db = sum of the partials, rounded once.  A workgroup sums 32 elements: lane group c of 8
// adds the chunks c, c + 8, ... in increasing order, then the 8 sums are added in order of c
// (one fixed association, whatever the timing).  The elements of all layers are one list.
template <typename T>
__global__ __launch_bounds__(256) void linear_dw_reduce_kernel(const LinearDwArgs a) {
  __shared__ float sums[8][32];
  const int e = threadIdx.x & 31, c0 = threadIdx.x >> 5;
  const int64_t idx = (int64_t)blockIdx.x * 32 + e;
  float sum = 0.f;
  if (idx < a.total) {
#pragma unroll 4
    for (int c = c0; c < a.chunks; c += 8) sum += a.part[(int64_t)c * a.total + idx];
  }
  sums[c0][e] = sum;
  __syncthreads();
  if (c0 == 0 && idx < a.total) {
    float total = sums[0][e];
#pragma unroll
    for (int c = 1; c < 8; ++c) total += sums[c][e];
    for (int p = 0; p < a.nlayers; ++p) {
      const int64_t w = idx - a.off_w[p], b = idx - a.off_b[p];
      if (w >= 0 && w < (int64_t)a.n[p] * a.K) reinterpret_cast<T*>(a.dw[p])[w] = (T)total;
      if (a.off_b[p] >= 0 && b >= 0 && b < a.n[p]) reinterpret_cast<T*>(a.db[p])[b] = (T)total;
    }
  }
}

}  // namespace tri
