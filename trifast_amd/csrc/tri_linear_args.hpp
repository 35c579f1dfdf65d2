// Argument blocks and launchers of the linear-layer kernels (tri_linear.hpp), and the rules by
// which their work is split.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tri {

constexpr int kLinearLayers = 6;

// Division of x < 2^31 by a launch's constant d as a product: with 2^s the next power of two at or above d and
// mul = ceil(2^(31+s) / d) < 2^32, x / d = x mul >> 31 + s (the excess x (mul d - 2^(31+s)) / d stays below
// 2^(31+s) / d).  mul = 0: d = 1.
struct Divisor {
  uint32_t d, mul, shift;
};
inline Divisor make_divisor(uint32_t d) {
  if (d <= 1) return Divisor{d, 0, 0};
  uint32_t s = 1;
  while ((uint64_t(1) << s) < d) ++s;
  return Divisor{d, (uint32_t)(((uint64_t(1) << (31 + s)) + d - 1) / d), s - 1};
}

// Row order: d = 0, rows are taken as they lie; otherwise the tensor is in pair order (b, i, j), i, j < d,
// while the work runs over the pair-transposed order (ending node): row (b, i, j) of the work is
// row (b, j, i) of the tensor.  (rows < 2^31)
struct RowMap {
  Divisor by;
};
inline RowMap row_map(uint32_t n) { return RowMap{make_divisor(n)}; }

struct LinearFwdArgs {
  const void* x;                    // [rows, K] in the order of xmap
  const void* w[kLinearLayers];     // [n[p], K]
  const void* bias[kLinearLayers];  // [n[p]] or null
  void* y[kLinearLayers];           // [rows, n[p]] (see linear_offset), rows in the order of ymap
  int n[kLinearLayers];
  int hd[kLinearLayers];
  int nlayers;
  int64_t rows;
  int K;
  RowMap xmap, ymap;
  // gated source in place of x: o [b, H, n, n, D] (K = H D, plane = n^2) and g [rows, K]
  const void *o, *g;
  Divisor plane;
  int H, D, lgD;
  // filled by the launcher: 32-column chunks of all layers, chunks per workgroup, workgroups per row block
  int total_chunks, chunks, groups;
};

struct LinearGateBwdArgs {
  const void* dout;  // [rows, K] in the order of map
  const void* w;     // [K, C], C = H D
  const void* o;     // [b, H, n, n, D]
  const void* g;     // [rows, C]
  void* dox;         // like o
  void* dg;          // like g
  int64_t rows;
  Divisor plane;
  int K, C, H, D, lgD;
  RowMap map;
  int chunks, groups;  // filled by the launcher
};

struct LinearDxArgs {
  const void* dy[kLinearLayers];  // [rows, n[p]] (see linear_offset)
  const void* w[kLinearLayers];   // [n[p], K]
  int n[kLinearLayers];
  int hd[kLinearLayers];
  int nlayers;
  void* dx;                       // [rows, K] in the order of map
  int64_t rows;
  int K;
  RowMap map;
};

struct LinearDwArgs {
  const void* x;                    // [rows, K] in the order of xmap, or the gated source's o
  const void* dy[kLinearLayers];    // [rows, n[p]] (see linear_offset), rows in the order of ymap
  int n[kLinearLayers];
  int hd[kLinearLayers];
  void* dw[kLinearLayers];          // [n[p], K]
  void* db[kLinearLayers];          // [n[p]] or null
  int nlayers;
  float* part;                      // [chunks][total] partial sums
  int64_t off_w[kLinearLayers], off_b[kLinearLayers];  // of a layer's parts in a chunk's row; off_b < 0: no bias gradient
  int64_t total;
  int64_t rows, rows_per_chunk;     // (a multiple of 64)
  int chunks, groups, rider;        // (see linear_dw_groups)
  int y_tile;                       // (see linear_dw_y_tile)
  int K;
  RowMap xmap, ymap;
  const void* g;                    // gated source: g [rows, K]
  const void* gw;                   // the gate's backward too: W [n[0], K], and where do (like x) and dg (like g) go
  void *dox, *dg;
  Divisor plane;
  int H, D, lgD;
};

constexpr int kLinearDwRider = 16;  // outputs of a riding layer at most (see linear_dw_groups)
constexpr int kLinearDwTile = 2048, kLinearDwWideTile = 4096;

// LDS bytes of a block's tile of 32 rows of dy: 64 per row; those of an odd number of outputs lie there as one word
// per output, which beyond 16 of them is twice as much.
template <typename Int>
inline int linear_dw_y_tile(const Int* n, int nlayers) {
  for (int p = 0; p < nlayers; ++p)
    if (n[p] % 2 != 0 && n[p] > 16) return kLinearDwWideTile;
  return kLinearDwTile;
}

// How the weight-gradient kernel's outputs are split over workgroups: groups of four 32-output blocks,
// the layers' blocks one after the other.  A layer of one block that would be a group for itself
// rides in the first group instead (an even number of outputs: it is loaded 4 bytes at a time; up
// to 128 channels: the accumulators of one block and a part of another fill the registers at 256; next to
// tiles of the ordinary size: with wide ones two stages and its own would not fit LDS at 64 channels).
// Alone it rides in a group without blocks, so that four waves share the work of a stage in place of
// one (2^20 rows, K = 128, 8 outputs: 71 -> 55 us); of 8 or 16 outputs of up to 64 channels one wave
// keeps up (K = 64 39.9 us and 44.4, K = 32 36.8 and 42.2; of 4, which are loaded in words then, 49.9 and 44.3).
struct LinearDwGroups {
  int groups, rider;  // rider: layer, or -1
};
template <typename Int>
inline LinearDwGroups linear_dw_groups(const Int* n, int nlayers, int64_t k) {
  int64_t blocks = 0;
  int small = -1;
  for (int p = 0; p < nlayers; ++p) {
    blocks += (n[p] + 31) / 32;
    if (n[p] <= kLinearDwRider && n[p] % 2 == 0) small = p;
  }
  const bool rides = k <= 128 && linear_dw_y_tile(n, nlayers) == kLinearDwTile && small >= 0 && blocks % 4 == 1 && (blocks > 1 || k == 128 || n[small] % 8 != 0);
  return LinearDwGroups{blocks == 1 ? 1 : (int)((blocks - (rides ? 1 : 0) + 3) / 4), rides ? small : -1};
}
// Whether rows of dy of some layer (but the riding one) are not whole 16-byte pieces.
template <typename Int>
inline bool linear_dw_words(const Int* n, int nlayers, int rider) {
  for (int p = 0; p < nlayers; ++p)
    if (p != rider && n[p] % 8 != 0) return true;
  return false;
}
// Workgroups of eight waves per CU: two for narrow rows, where one step's latency shows next to the few
// bytes of a stage (2^20 rows, 8 or 64 outputs: K = 32 59 us with one, 41 to 46 with two, K = 64 61 to 63
// and 44 to 59).  At 128 and 256 the accumulators take more than a fourth of a SIMD's registers.
template <int64_t K>
constexpr int kLinearDwPerCu = K <= 64 ? 2 : 1;
// Rows of one chunk: the groups of a chunk run on one XCD of 32 CUs, so 8 * (resident workgroups of an
// XCD / groups) chunks are one full round; at least 256 rows (the partials of a chunk cost as much
// traffic as 128 rows).
inline int64_t linear_dw_rows_per_chunk(int64_t rows, int groups, int64_t k) {
  const int64_t slots = 32 * (k <= 64 ? kLinearDwPerCu<64> : kLinearDwPerCu<128>);
  const int64_t most = 8 * (slots / groups < 1 ? 1 : slots / groups);
  const int64_t per = ((rows + most - 1) / most + 63) / 64 * 64;
  return per < 256 ? 256 : per;
}

// One layer by itself is given room for the partials of chunks of at least 1024 rows, at most 768 of them.
inline int64_t linear_dw_chunks(int64_t rows) {
  const int64_t even = ((rows + 767) / 768 + 31) / 32 * 32, per = even < 1024 ? 1024 : even;
  return (rows + per - 1) / per;
}

// The gated output layer's weight gradient and the gate's backward in one launch: o, g and dout are read once
// for both.  K = 128, 128 outputs: 16384 rows 25.7 -> 23.8 us, 147456 65 -> 44, 2^20 452 -> 281; K = 64, 64 outputs:
// 16384 rows 20.2 -> 19.0, 147456 45.6 -> 36.9, 2^20 251 -> 173.  At K = 32 the weight gradient runs
// two workgroups per CU, which the gate's backward has no registers for (2^20 rows 125 -> 147); at K = 256 two
// stages and W do not fit LDS.
inline bool linear_dw_with_gate_bwd(int64_t k) { return k == 64 || k == 128; }

inline bool linear_fwd_k_ok(int64_t k) { return k == 32 || k == 64 || k == 128; }
inline bool linear_gated_k_ok(int64_t k) { return k == 32 || k == 64 || k == 128 || k == 256; }
// (the accumulators of 64 rows x K columns per wave stay in registers: K up to 128)
inline bool linear_dx_k_ok(int64_t k) { return k == 32 || k == 64 || k == 128; }
inline bool linear_dw_k_ok(int64_t k) { return k == 32 || k == 64 || k == 128 || k == 256; }

hipError_t linear_fwd_launch(LinearFwdArgs a, int dtype, hipStream_t st);
hipError_t linear_gate_bwd_launch(LinearGateBwdArgs a, int dtype, hipStream_t st);
hipError_t linear_dx_launch(const LinearDxArgs& a, int dtype, hipStream_t st);
hipError_t linear_dw_launch(const LinearDwArgs& a, int dtype, hipStream_t st);

}  // namespace tri
