// Tile-level building blocks shared by the four kernels.
#pragma once
#include "tri_args.hpp"
#include "tri_common.hpp"

namespace tri {

// Workgroups are handed to the 8 XCDs round-robin by linear id, and each XCD has
// its own L2.  All blocks that share one pair row (same K/V rows) should land on
// one XCD: with gx blocks per row, linear id L = 8*slot + xcd is re-read as
//   x = slot % gx,  y = 8 * (slot / gx) + xcd
// The launcher pads the row count to a multiple of 8; y >= rows means "no work".
TRI_DEV void xcd_remap(int gx, int& x, int& y) {
  const int L = blockIdx.x + gx * blockIdx.y;
  const int xcd = L & 7, slot = L >> 3;
  x = slot % gx;
  y = 8 * (slot / gx) + xcd;
}

// ---------------------------------------------------------------------------
// Swizzled LDS tiles filled by direct global->LDS loads.
//
// A tile holds ROWS rows of D elements, unpadded; the 16-byte chunks of a row are
// stored XOR-swizzled by swz(row) so that the operand reads of a wave (16 rows at
// one logical chunk, or 4 rows x 32 bytes for the transposing read) spread over
// all banks.  global_load_lds writes lane l's 16 bytes at (wave-uniform LDS base)
// + 16*l, so the swizzle costs nothing: it only decides which global address a
// lane reads.  The loads use no registers and are tracked by vmcnt; the caller
// waits with wait_dma() before the barrier that publishes the tile.
// ---------------------------------------------------------------------------
#define TRI_G1 __attribute__((address_space(1)))
#define TRI_L3 __attribute__((address_space(3)))

TRI_DEV void wait_dma() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// The same wait as an instruction the compiler knows: what it waits for no longer counts as
// in flight when the compiler places its own waits (vmcnt = 0, the other counters at maximum).
TRI_DEV void wait_dma_known() {
  __builtin_amdgcn_s_waitcnt(0x0F70);
  asm volatile("" ::: "memory");
}

// The order every counted wait here relies on: vmcnt counts a wave's vector loads (direct loads into LDS
// among them) and its stores together, and both leave it in the order of issue, so that "at most n outstanding"
// means that everything but the newest n has completed.  (The compiler places its own waits on gfx950 by the
// same rule: a load, two stores, a use of the load give vmcnt(2).)
// Stage hand-over for a ring of LDS buffers: wait until at most the newest
// IN_FLIGHT loads of this wave are outstanding (everything issued before them
// has landed in LDS) and every LDS read of the wave
// has returned, then meet the other waves.  A plain barrier instruction: the
// fence of __syncthreads() would wait for every load in flight.
template <int IN_FLIGHT>
TRI_DEV void ring_sync() {
  static_assert(IN_FLIGHT >= 0 && IN_FLIGHT <= 63, "vmcnt has 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(IN_FLIGHT) : "memory");
}

// SWZ_ROWS: rows that share one swizzle value (0: as many as make 256 bytes, which is what
// 16-byte operand reads of 16 rows want; a tile that is written with 16-byte stores, one row
// per lane, and only read back transposed wants 2: measured, the stores then run without
// bank conflicts, and transposing reads take whole rows, so any per-row swizzle suits them).
// bytes of a row of D elements in LDS (fp32 rows lie there as their three bf16 parts, see SplitStream)
constexpr int lds_row_bytes(int D, int es) { return es == 4 ? 6 * D : D * es; }

template <typename T, int D, int SWZ_ROWS = 0>
struct LdsTile {
  static_assert(sizeof(T) == 2, "fp32 tiles are three tiles of bf16 parts");
  static constexpr int ROWB = D * (int)sizeof(T);  // bytes per row
  static constexpr int CPR = ROWB / 16;            // 16-byte chunks per row (power of two)
  static constexpr int RPB = SWZ_ROWS > 0 ? SWZ_ROWS : ((256 / ROWB) > 0 ? 256 / ROWB : 1);  // rows per swizzle value
  static constexpr int VEC = 16 / (int)sizeof(T);
  // Neighbouring swizzle values differ in the high chunk bits: a transposing read takes 4 rows x 64
  // bytes at once, and the rows that start at the same bank (every second one of 128 bytes, each of 256)
  // have to lie 64 bytes apart.  (With the plain row number as the value two or four of them met in a
  // bank, 25 to 30 % of the LDS cycles at d = 64: n = 512, h = 4, d = 128 dk/dv 970 -> 930 us, dq 616 ->
  // 598; n = 768, h = 8, d = 64 dk/dv 2.52 -> 2.48 ms, the others within 1 %.  As 5 x the value is one
  // instruction away from the row number; with the chunk bits rotated, which is as free of conflicts, a
  // step at n = 242, h = 8, d = 64 took 410 us, with 5 x 399, with the row number 399.)
  TRI_DEV static int swz(int r) {
    constexpr int B = CPR < 16 ? CPR : 16;  // (16 chunks are all banks)
    const unsigned x = (unsigned)r / RPB % B;  // (rows are not negative)
    return (int)(B <= 4 ? x : (x + (x << 2)) % B);  // (5 x: bits 2 and 3 take what bits 0 and 1 are)
  }
  // byte offset, from the tile base, of byte `o` of row r (o must not straddle a chunk)
  TRI_DEV static int off(int r, int o) { return (r * CPR + ((o >> 4) ^ swz(r))) * 16 + (o & 15); }
  template <typename V>
  TRI_DEV static V read(const unsigned char* base, int r, int elem) {
    return *reinterpret_cast<const V*>(base + off(r, elem * (int)sizeof(T)));
  }
  // Fill ROWS rows; row_ptr(r) gives the global address of row r (callers clamp r
  // into range instead of branching).  NW waves share the work.
  template <int ROWS, int NW, typename RowPtr>
  TRI_DEV static void fill(unsigned char* base, RowPtr row_ptr, int wave, int lane) {
    constexpr int GROUPS = ROWS * CPR / 64;
    static_assert(ROWS * CPR % 64 == 0, "tile must be a whole number of 1 KiB wave loads");
#pragma unroll
    for (int x = 0; x < (GROUPS + NW - 1) / NW; ++x) {
      const int gi = x * NW + wave;
      if (GROUPS % NW == 0 || gi < GROUPS) {
        const int p = gi * 64 + lane;
        const int r = p / CPR, c = (p % CPR) ^ swz(r);
        const T* src = row_ptr(r) + c * VEC;
        __builtin_amdgcn_global_load_lds((const TRI_G1 void*)src, (TRI_L3 void*)(base + gi * 1024), 16, 0, 0);
      }
    }
  }
};

// Lane-constant byte offsets of the operand reads of one wave.  Tiles start at
// rows that are multiples of 32 and MFMA steps move by 16 rows; neither changes
// the swizzle, so an operand read is (tile base + compile-time offset) + one of
// these registers.  fp32: every block of 32 rows is three such tiles of bf16 parts, one
// after the other, and an operand is read from all three.
template <typename T, int D, int SWZ_ROWS = 0>
struct OperandOffsets {
  using P = std::conditional_t<sizeof(T) == 4, __bf16, T>;
  using Tile = LdsTile<P, D, SWZ_ROWS>;
  using frag = typename Elem<T>::frag;
  using pfrag = typename Elem<P>::frag;
  static constexpr int KP = Elem<T>::KP;
  static constexpr int DS = D / (2 * KP);
  static constexpr int DM = (D + 31) / 32;
  static constexpr int PLANE = 32 * Tile::ROWB;  // between the parts of a block of fp32 rows
  int nat[DS], tlo[DM], thi[DM];
  int lane;
  // `row_in_tile`: the row of a 32-row tile this lane reads as a natural operand
  TRI_DEV void init(int row_in_tile, int lane_) {
    lane = lane_;
    const int g = lane >> 5, L = lane & 15, chalf = (lane >> 4) & 1;
#pragma unroll
    for (int s = 0; s < DS; ++s) nat[s] = Tile::off(row_in_tile, (2 * KP * s + KP * g) * (int)sizeof(P));
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) {
      const int col = 32 * mt + 16 * chalf + 4 * (L & 3);
      tlo[mt] = Tile::off(8 * g + (L >> 2), col * 2);
      thi[mt] = Tile::off(8 * g + 4 + (L >> 2), col * 2);
    }
  }
  // move every offset by a whole number of 32-row tiles (a wave's own part of a larger tile)
  TRI_DEV void shift(int bytes) {
#pragma unroll
    for (int s = 0; s < DS; ++s) nat[s] += bytes;
#pragma unroll
    for (int mt = 0; mt < DM; ++mt) { tlo[mt] += bytes; thi[mt] += bytes; }
  }
  // make the offsets opaque to the compiler: it then keeps them in registers as they
  // are instead of rebuilding them from another instance plus a constant
  TRI_DEV void pin() {
#pragma unroll
    for (int s = 0; s < DS; ++s) asm volatile("" : "+v"(nat[s]));
  }
  // Fold the address of the workgroup's LDS block into the offsets: natural_at() then
  // reads from absolute LDS addresses, one register plus an immediate per read.
  TRI_DEV void make_absolute(const unsigned char* lds_base) {
    const int b0 = (int)(uintptr_t)(TRI_L3 const unsigned char*)lds_base;
#pragma unroll
    for (int s = 0; s < DS; ++s) nat[s] += b0;
  }
  template <typename Read>
  static TRI_DEV frag parts(Read read) {
    if constexpr (sizeof(T) == 4) return frag{read(0), read(PLANE), read(2 * PLANE)};
    else return read(0);
  }
  // natural operand of the 32-row tile `byte_offset` bytes into the block (after make_absolute)
  TRI_DEV frag natural_at(int byte_offset, int s) const {
    return parts([&](int o) { return *reinterpret_cast<TRI_L3 const pfrag*>((uintptr_t)(uint32_t)(nat[s] + byte_offset + o)); });
  }
  // natural operand (head-dim index in-lane), MFMA step s, of the 32-row tile at `tile`
  TRI_DEV frag natural(const unsigned char* tile, int s) const {
    return parts([&](int o) { return *reinterpret_cast<const pfrag*>(tile + nat[s] + o); });
  }
  // transposed operand (row index in-lane): rows cidx(KP*step.., g), column 32*mt + lane%32
  TRI_DEV frag transposed(const unsigned char* tile, int step, int mt) const {
    if (D % 32 != 0 && 32 * mt + (lane & 31) >= D) return Elem<T>::zero();
    return transposed_all(tile, step, mt);
  }
  // The same without the branch: lanes whose column lies past the end of a row get bytes of the LDS behind it.  For operand rows whose
  // results nobody uses.
  TRI_DEV frag transposed_all(const unsigned char* tile, int step, int mt) const {
    return parts([&](int o) {
      const unsigned char* p = tile + 16 * step * Tile::ROWB + o;
      const auto lo = lds_tr4(reinterpret_cast<const P*>(p + tlo[mt]));
      const auto hi = lds_tr4(reinterpret_cast<const P*>(p + thi[mt]));
      pfrag f;
#pragma unroll
      for (int e = 0; e < 4; ++e) { f[e] = lo[e]; f[4 + e] = hi[e]; }
      return f;
    });
  }
};

// fp32 rows on their way to LDS: ROWS rows (whole blocks of 32) of D numbers, loaded into
// registers 16 bytes per lane and piece, and written as their three bf16 parts once the compute
// that reads the old contents is done.  The split is paid once per workgroup and row here, not
// once per wave and use (3.5 vector instructions a number).
template <int D, int ROWS, int NW>
struct SplitStream {
  using Tile = LdsTile<__bf16, D>;
  static constexpr int PLANE = 32 * Tile::ROWB;
  static constexpr int CH = D / 4, TOTAL = ROWS * CH, XN = (TOTAL + NW * 64 - 1) / (NW * 64);
  static constexpr bool WHOLE = TOTAL % (NW * 64) == 0;
  const float* p0[XN];
  uint32_t dst[XN];
  f32x4 x[XN];
  int tid;
  template <typename RowPtr>
  TRI_DEV void init(RowPtr row_ptr, int wave, int lane) {
    tid = wave * 64 + lane;
#pragma unroll
    for (int i = 0; i < XN; ++i) {
      const int p = min(i * NW * 64 + tid, TOTAL - 1), r = p / CH, c = p % CH;
      p0[i] = row_ptr(r) + 4 * c;
      dst[i] = (uint32_t)((r / 32) * 3 * PLANE + Tile::off(r % 32, 8 * c));
    }
  }
  // the tile, moved by `elem_offset` (wave-uniform) from the rows of init()
  TRI_DEV void load(int64_t elem_offset) {
#pragma unroll
    for (int i = 0; i < XN; ++i) x[i] = *reinterpret_cast<const f32x4*>(p0[i] + elem_offset);
  }
  // any rows
  template <typename RowPtr>
  TRI_DEV void load_rows(RowPtr row_ptr) {
#pragma unroll
    for (int i = 0; i < XN; ++i) {
      const int p = min(i * NW * 64 + tid, TOTAL - 1);
      x[i] = *reinterpret_cast<const f32x4*>(row_ptr(p / CH) + 4 * (p % CH));
    }
  }
  TRI_DEV void store(unsigned char* base) const {
#pragma unroll
    for (int i = 0; i < XN; ++i) {
      bf16x2 h[2], m[2], l[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) split_pair(x[i][2 * t], x[i][2 * t + 1], h[t], m[t], l[t]);
      if (!WHOLE && i * NW * 64 + tid >= TOTAL) continue;
      unsigned char* d = base + dst[i];
      *reinterpret_cast<bf16x4*>(d) = bf16x4{h[0][0], h[0][1], h[1][0], h[1][1]};
      *reinterpret_cast<bf16x4*>(d + PLANE) = bf16x4{m[0][0], m[0][1], m[1][0], m[1][1]};
      *reinterpret_cast<bf16x4*>(d + 2 * PLANE) = bf16x4{l[0][0], l[0][1], l[1][0], l[1][1]};
    }
  }
};

// A tile of ROWS rows that is re-filled stage after stage from rows that move
// along one tensor index: the per-lane source pointers are computed once for
// position 0 and a stage adds one wave-uniform element offset to them.
template <typename T, int D, int ROWS, int NW>
struct TileStream {
  using Tile = LdsTile<T, D>;  // (16-bit types; SplitStream for fp32)
  static constexpr int GROUPS = ROWS * Tile::CPR / 64;
  static constexpr int XN = (GROUPS + NW - 1) / NW;
  static_assert(ROWS * Tile::CPR % 64 == 0, "tile must be a whole number of 1 KiB wave loads");
  const T* p0[XN];
  template <typename RowPtr>
  TRI_DEV void init(RowPtr row_ptr, int wave, int lane) {
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const int gi = (GROUPS % NW == 0) ? x * NW + wave : min(x * NW + wave, GROUPS - 1);
      const int p = gi * 64 + lane;
      const int r = p / Tile::CPR, c = (p % Tile::CPR) ^ Tile::swz(r);
      p0[x] = row_ptr(r) + c * Tile::VEC;
    }
  }
  // EVERY = true: a wave whose share of the tile is empty repeats the tile's last
  // piece instead of skipping it, so that every wave issues exactly XN loads (a
  // fixed count is what lets a later s_waitcnt vmcnt(k) stand for "all but the
  // newest stages have landed")
  template <bool EVERY = false>
  TRI_DEV void issue(unsigned char* base, int64_t elem_offset, int wave) const {
    // the offset is wave-uniform: pin it to scalar registers so that a stage costs
    // one 64-bit add per load
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)elem_offset);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)elem_offset >> 32));
    elem_offset = (int64_t)(((uint64_t)hi << 32) | lo);
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const int gi = EVERY ? min(x * NW + wave, GROUPS - 1) : x * NW + wave;
      if (EVERY || GROUPS % NW == 0 || gi < GROUPS)
        __builtin_amdgcn_global_load_lds((const TRI_G1 void*)(p0[x] + elem_offset), (TRI_L3 void*)(base + gi * 1024), 16, 0, 0);
    }
  }
};

// A ring of 32-row stages in LDS: the same 32 positions of R pair rows of two tensors (K and V, or
// Q and dO) and the packed bias tile of each wave, filled by loads the compiler does not see: a
// load that it knows of makes every LDS read after it wait for that load, the read might be of the
// bytes in flight.  Every wave issues NLD loads per stage, so that a counted wait stands for "all but
// the newest stages have landed" (ring_sync).  A lane's source is a 32-bit byte offset from the
// stage's first row, and the scalar pointers move along the row by a constant step per stage.
constexpr int ring_stage_bytes(int D, int es, int NW, int R) { return 2 * R * 32 * D * es + NW * 2048; }
template <typename T, int D, int NW, int R, int NSTAGES>
struct StageRing {
  using Tile = LdsTile<T, D>;
  static constexpr int ROWB = Tile::ROWB;
  static constexpr int NS = NSTAGES;
  static constexpr int FSTAGE = ring_stage_bytes(D, (int)sizeof(T), NW, R);
  static constexpr int FOFF_V = R * 32 * ROWB, FOFF_B = 2 * R * 32 * ROWB;  // second tensor, bias tiles
  static constexpr int G = 2 * R * 32 * Tile::CPR / 64;  // 1 KiB wave loads per stage: first tensor, then second
  static_assert(G % NW == 0, "every wave issues the same number of loads");
  static constexpr int XN = G / NW;
  static constexpr int NLD = XN + 2;  // loads per wave and stage: its share of the rows, its bias tile
  uint32_t lofs[XN], lane16, lds0;
  int64_t kstep, vstep;
  int bstep;
  const T *kfill, *vfill, *bfill;
  uint32_t rowk, rowv;  // bytes between neighbouring rows
  int pos, last;        // the stage the pointers stand at, the last of the row
  int tail;             // rows of the last stage where it is ragged (0: n is a multiple of 32)

  // the 32-bit offsets reach the rows of a stage
  static TRI_DEV bool fits(const Str5& st) {
    return st.i >= 0 && st.j >= 0 && (uint64_t)(R - 1) * st.i + 31ull * st.j + D < (1ull << 31) / sizeof(T);
  }
  // bases of the batch and head, this wave's first bias tile and the elements from one to the next
  TRI_DEV void init(const Str5& sk, const Str5& sv, const T* kbh, const T* vbh, const T* bias_wave, int bias_step, int N, int i0, int wave, int lane,
                    const unsigned char* smem) {
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const int gi = x * NW + wave;
      const int p = (gi % (G / 2)) * 64 + lane;
      const int r_ = p / Tile::CPR, cc = (p % Tile::CPR) ^ Tile::swz(r_);
      const int64_t rr = min(i0 + r_ / 32, N - 1) - i0;
      const Str5& st = gi < G / 2 ? sk : sv;
      lofs[x] = (uint32_t)((rr * st.i + (int64_t)(r_ % 32) * st.j + cc * Tile::VEC) * (int64_t)sizeof(T));
    }
    lane16 = (uint32_t)lane * 16u;
    lds0 = (uint32_t)(uintptr_t)(TRI_L3 const unsigned char*)smem;
    kstep = 32 * sk.j;
    vstep = 32 * sv.j;
    bstep = bias_step;
    kfill = kbh + (int64_t)i0 * sk.i;
    vfill = vbh + (int64_t)i0 * sv.i;
    bfill = bias_wave;
    rowk = (uint32_t)sk.j * (uint32_t)sizeof(T);
    rowv = (uint32_t)sv.j * (uint32_t)sizeof(T);
    pos = 0;
    last = (N - 1) >> 5;
    tail = N & 31;
  }
  // Request the stage the pointers stand at into the ring buffer at `boff`, and move on unless
  // it is stage ns - 1: past the last stage a valid one is fetched again, which nobody uses.
  TRI_DEV void issue(int boff, int ns, int wave, int lane) {
    auto load_rows = [&](int x, uint32_t voff) __attribute__((always_inline)) {
      const int gi = x * NW + wave;
      const T* base = gi < G / 2 ? kfill : vfill;  // wave-uniform
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(boff + gi * 1024));
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(voff), "s"(base) : "memory", "m0");
    };
    if (tail != 0 && pos == last) {
      // the ragged last stage: rows past the end read the last one again
      asm volatile("" ::);  // (a real branch: nothing of this in the common path)
      int lane_now = lane;
      asm volatile("" : "+v"(lane_now));
#pragma unroll
      for (int x = 0; x < XN; ++x) {
        const int gi = x * NW + wave;
        const int key = ((gi % (G / 2)) * 64 + lane_now) / Tile::CPR & 31;
        // (row strides are below 2^24 bytes)
        load_rows(x, lofs[x] - __umul24((uint32_t)max(key - (tail - 1), 0), gi < G / 2 ? rowk : rowv));
      }
    } else {
#pragma unroll
      for (int x = 0; x < XN; ++x) load_rows(x, lofs[x]);
    }
    const uint32_t dstb = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(boff + FOFF_B + wave * 2048));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024" : : "s"(dstb), "v"(lane16), "s"(bfill) : "memory", "m0");
    // (the second load lands 1 KiB further: the instruction offset applies to both addresses)
    const bool more = pos + 1 < ns;
    kfill += more ? kstep : 0;
    vfill += more ? vstep : 0;
    bfill += more ? bstep : 0;
    pos += more ? 1 : 0;
  }
};

// 4-byte-per-lane variant for rows of floats (lse, delta): 64 floats per wave load
template <int COUNT, int NW, typename Ptr>
TRI_DEV void fill_floats(float* base, Ptr elem_ptr, int wave, int lane) {
  constexpr int GROUPS = COUNT / 64;
  static_assert(COUNT % 64 == 0, "whole wave loads only");
#pragma unroll
  for (int x = 0; x < (GROUPS + NW - 1) / NW; ++x) {
    const int gi = x * NW + wave;
    if (GROUPS % NW == 0 || gi < GROUPS)
      __builtin_amdgcn_global_load_lds((const TRI_G1 void*)elem_ptr(gi * 64 + lane), (TRI_L3 void*)(base + gi * 64), 4, 0, 0);
  }
}

// The same for COUNT floats that move along one index (lse, delta of a query tile).
template <int COUNT, int NW>
struct FloatStream {
  static constexpr int GROUPS = COUNT / 64;
  static constexpr int XN = (GROUPS + NW - 1) / NW;
  static_assert(COUNT % 64 == 0, "whole wave loads only");
  const float* p0[XN];
  template <typename Ptr>
  TRI_DEV void init(Ptr elem_ptr, int wave, int lane) {
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const int gi = (GROUPS % NW == 0) ? x * NW + wave : min(x * NW + wave, GROUPS - 1);
      p0[x] = elem_ptr(gi * 64 + lane);
    }
  }
  template <bool EVERY = false>
  TRI_DEV void issue(float* base, int64_t elem_offset, int wave) const {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)elem_offset);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)elem_offset >> 32));
    elem_offset = (int64_t)(((uint64_t)hi << 32) | lo);
#pragma unroll
    for (int x = 0; x < XN; ++x) {
      const int gi = EVERY ? min(x * NW + wave, GROUPS - 1) : x * NW + wave;
      if (EVERY || GROUPS % NW == 0 || gi < GROUPS)
        __builtin_amdgcn_global_load_lds((const TRI_G1 void*)(p0[x] + elem_offset), (TRI_L3 void*)(base + gi * 64), 4, 0, 0);
    }
  }
};

// The 16 bias values of one lane for tile (jt, kt), in the raw-score domain
// (times sqrt(d)) plus a per-lane additive term, from a packed bias array.
template <typename T>
TRI_DEV f32x16 bias_tile(const T* pack_bh, int NP, int jt, int kt, int lane, float sqrt_d, float add) {
  const T* p = pack_bh + ((((int64_t)jt * NP + kt) * 2) * 64 + lane) * 8;
  f32x16 s;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if constexpr (sizeof(T) == 2) {
      const typename Elem<T>::vec x = *reinterpret_cast<const typename Elem<T>::vec*>(p + r * 512);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[8 * r + e] = __builtin_fmaf((float)x[e], sqrt_d, add);
    } else {
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(p + r * 512);
      const f32x4 x1 = *reinterpret_cast<const f32x4*>(p + r * 512 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[8 * r + e] = __builtin_fmaf(x0[e], sqrt_d, add);
        s[8 * r + 4 + e] = __builtin_fmaf(x1[e], sqrt_d, add);
      }
    }
  }
  return s;
}

// acc + the products of eight consecutive numbers
template <typename T>
TRI_DEV float dot8(const T* x, const T* y, float acc) {
  using vec = typename Elem<T>::vec;
  constexpr int V = Elem<T>::VEC;
#pragma unroll
  for (int v = 0; v < 8 / V; ++v) {
    const vec xv = *reinterpret_cast<const vec*>(x + V * v), yv = *reinterpret_cast<const vec*>(y + V * v);
#pragma unroll
    for (int e = 0; e < V; ++e) acc += (float)xv[e] * (float)yv[e];
  }
  return acc;
}

// Which 32-key tiles matter to the R pair rows of a workgroup, as bitmaps over
// the key tiles, one 64-bit word per 64 tiles, built once into LDS:
//   live  = some row attends to some key of the tile (other tiles are skipped:
//           their probabilities are exactly zero),
//   plain = every row attends to every key of the tile (no mask work at all).
// The words of the 64-tile chunk in use are cached in scalar registers, so the
// per-stage queries are scalar bit operations.
// A 64-bit word that every lane holds, as a wave-uniform value (the two halves go through
// readfirstlane, whose result is a signed int: each half is widened as unsigned).
TRI_DEV uint64_t uniform_u64(uint64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | lo;
}

struct KeyTileMasks {
  const uint64_t* words;  // LDS: [nchunks] live, then [nchunks] plain
  int nchunks, ntiles, cur;
  uint64_t live, plain;

  static constexpr int lds_bytes(int nwords) { return 16 * ((nwords + 63) / 64); }

  // keep_row(r) = pointer to the keep words of row r.  Every wave calls this; the
  // caller synchronises the workgroup before the first query.  Bits of the last word that are
  // set in `past_end` (keys past the end of the row) do not keep its tile from being plain.
  template <int R, int NW, typename KeepRow>
  TRI_DEV void build(uint64_t* lds, KeepRow keep_row, int nwords, bool force_not_plain, int wave, int lane, uint32_t past_end = 0) {
    words = lds;
    ntiles = nwords;
    nchunks = (nwords + 63) / 64;
    cur = -1;
    live = plain = 0;
    for (int ch = wave; ch < nchunks; ch += NW) {
      const int w = ch * 64 + lane;
      uint32_t any = 0, all = 0xffffffffu;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t x = (w < nwords) ? keep_row(r)[w] : 0u;
        any |= x;
        all &= x | (w == nwords - 1 ? past_end : 0u);
      }
      const uint64_t lv = __ballot(any != 0);
      const uint64_t pl = force_not_plain ? 0 : __ballot(all == 0xffffffffu);
      if (lane == 0) {
        lds[ch] = lv;
        lds[nchunks + ch] = pl;
      }
    }
  }
  TRI_DEV void select(int ch) {
    if (ch == cur) return;
    cur = ch;
    const uint64_t lv = words[ch], pl = words[nchunks + ch];
    live = uniform_u64(lv);
    plain = uniform_u64(pl);
  }
  // first stage of KU tiles at or after tile t (t % KU == 0) with a live tile; ntiles if none
  template <int KU>
  TRI_DEV int next_live(int t) {
    while (t < ntiles) {
      select(t >> 6);
      const uint64_t m = live >> (t & 63);
      if (m != 0) {
        const int pos = __builtin_ctzll(m);
        return t + pos - pos % KU;
      }
      t = ((t >> 6) + 1) << 6;
    }
    return ntiles;
  }
  // one past the last key tile with an attended key, 0 if there is none (wave-uniform; reads
  // the bitmaps from LDS)
  TRI_DEV int last_live() const {
    int last = 0;
    for (int ch = 0; ch < nchunks; ++ch) {
      const uint64_t lv = words[ch];
      const uint64_t u = uniform_u64(lv);
      if (u != 0) last = 64 * ch + 64 - __builtin_clzll(u);
    }
    return last;
  }
  // every key tile is plain (wave-uniform; reads the bitmaps from LDS)
  TRI_DEV bool all_plain() const {
    bool all = true;
    for (int ch = 0; ch < nchunks; ++ch) {
      const int nt = min(64, ntiles - 64 * ch);
      const uint64_t want = nt == 64 ? ~0ull : ((1ull << nt) - 1);
      const uint64_t pl = words[nchunks + ch];
      const uint64_t u = uniform_u64(pl);
      all = all && (u & want) == want;
    }
    return all;
  }
  // every tile of the stage at tile t (in the chunk last selected) is plain
  template <int KU>
  TRI_DEV bool stage_plain(int t) const {
    constexpr uint64_t kMask = (1ull << KU) - 1;
    return ((plain >> (t & 63)) & kMask) == kMask;
  }
};

// Compile-time versions of a stage loop, chosen per workgroup: every row attends to
// every key (constant keys operand, no per-tile branch); some keys are masked but no
// row is fully masked (dead tiles skipped); anything.
constexpr int kPlain = 0, kMasked = 1, kGeneral = 2;

// Store a 32-row tile of an [n x D] output held transposed in registers
// (lane owns row `row`, values are columns 32*mt + 8*a4 + 4*g + 0..3), scaled.
template <typename T, int D, int DM>
TRI_DEV void store_rows(T* out_row, const f32x16* acc, float mul, int g) {
  using E = Elem<T>;
#pragma unroll
  for (int mt = 0; mt < DM; ++mt) {
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) {
      const int d0 = 32 * mt + 8 * a4 + 4 * g;
      if (d0 < D) {
        typename E::vec4 ov;
#pragma unroll
        for (int e = 0; e < 4; ++e) ov[e] = (T)(acc[mt][4 * a4 + e] * mul);
        *reinterpret_cast<typename E::vec4*>(out_row + d0) = ov;
      }
    }
  }
}

// The same store for 16-bit outputs with 16 bytes per lane: lane l and lane l ^ 32 own the
// two halves of every 8 columns of one row; they trade values (v_permlane32_swap) so that
// the lower lane ends up with columns 32*mt + 8*h + 0..7 and the upper lane with columns
// 32*mt + 16 + 8*h + 0..7, each whole.  Half as many store instructions, each of them
// writing whole 16-byte pieces.  Every lane of the wave takes part in the exchange;
// `active` says whether this lane's row is stored.
template <typename T, int D, int DM>
TRI_DEV void store_rows_wide(T* out_row, const f32x16* acc, float mul, int g, bool active) {
  static_assert(sizeof(T) == 2, "16-bit outputs");
  using E = Elem<T>;
  typedef uint32_t u32x2s __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int mt = 0; mt < DM; ++mt) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      typename E::vec4 lo4, hi4;  // this lane's columns 8h + 4g + 0..3 and 8(h+2) + 4g + 0..3
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo4[e] = (T)(acc[mt][4 * h + e] * mul);
        hi4[e] = (T)(acc[mt][4 * (h + 2) + e] * mul);
      }
      const u32x2s x = __builtin_bit_cast(u32x2s, lo4), y = __builtin_bit_cast(u32x2s, hi4);
      const auto r0 = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
      const u32x4s out = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
      const int d0 = 32 * mt + 16 * g + 8 * h;
      if (active && d0 < D) *reinterpret_cast<u32x4s*>(out_row + d0) = out;
    }
  }
}

// either of the two, by the element type
template <typename T, int D, int DM>
TRI_DEV void store_rows_any(T* out_row, const f32x16* acc, float mul, int g, bool active) {
  if constexpr (sizeof(T) == 2) {
    store_rows_wide<T, D, DM>(out_row, acc, mul, g, active);
  } else {
    if (active) store_rows<T, D, DM>(out_row, acc, mul, g);
  }
}

}  // namespace tri
