// Linear-layer kernel instantiations and their launchers.
#include "tri_linear.hpp"

namespace tri {
namespace {

// How the outputs of a row block are split over workgroups: `most` 32-column chunks per workgroup
// at most (their weights share LDS), fewer while the launch has less than `wgs` workgroups: four per
// CU for the projections; one where the rows are gated first, which every workgroup of a row block
// does for itself (K = 128, 128 outputs, 25600 rows: 16.7 us with four, 11.4 with one; the gate's
// backward 15.2 and 11.3; the projections of 10000 rows 9.1 to 11.0 and 11.9).
void split_chunks(int64_t row_blocks, int total, int most, int wgs, int& chunks, int& groups) {
  int64_t per = row_blocks * total / wgs;
  per = per < 1 ? 1 : (per > most ? most : per);
  groups = (int)((total + per - 1) / per);
  chunks = (total + groups - 1) / groups;
  groups = (total + chunks - 1) / chunks;
}

// 256 rows per workgroup (two row tiles per wave share every weight fragment) once that fills the
// GPU twice over, 128 below
bool two_row_tiles(int64_t rows) { return rows >= 256 * 512; }

dim3 row_grid(int64_t rows, int per_block, int groups) {
  const int64_t blocks = ((rows + per_block - 1) / per_block + 7) / 8 * 8;
  return dim3((unsigned)(blocks * groups));
}

template <typename T, int KD, int RT, bool GATED>
hipError_t fwd_run(LinearFwdArgs a, hipStream_t st) {
  a.total_chunks = 0;
  for (int p = 0; p < a.nlayers; ++p) a.total_chunks += (a.n[p] + 31) / 32;
  constexpr int chunk_bytes = 32 * KD * (int)sizeof(T);
  const int64_t blocks = (a.rows + 128 * RT - 1) / (128 * RT);
  split_chunks(blocks, a.total_chunks, 40 * 1024 / chunk_bytes, GATED ? 256 : 1024, a.chunks, a.groups);
  return launch_dyn(linear_fwd_kernel<T, KD, RT, GATED>, row_grid(a.rows, 128 * RT, a.groups), dim3(256), a.chunks * (chunk_bytes + 32 * (int)sizeof(T)), st, a);
}

template <typename T, int KD>
hipError_t fwd_rows(const LinearFwdArgs& a, hipStream_t st) {
  if (a.o) return fwd_run<T, KD, 1, true>(a, st);
  if constexpr (KD <= 128) {
    // Five tiles of 32 rows per CU and more (K = 128, 17 chunks: 65536 rows 32 -> 28 us, 16384 14 -> 18).  Narrower
    // rows are as fast through the other kernel until the layers are many (K = 64, 33 chunks: 2^20
    // rows 584 -> 522 us, 65536 44 -> 46; 17 chunks: 2^20 rows 304 -> 295).
    const ResidentPlan plan = resident_plan(a);
    const int lds = linear_fwd_resident_lds(KD, plan.chunks);
    const bool gains = KD == 128 ? a.rows >= kResidentWgs * 32 * 5 : plan.chunks >= 32 && a.rows >= kResidentWgs * 32 * 32;
    if (plan.chunks && gains && a.rows < (int64_t(1) << 31) && lds <= kResidentLds)
      return launch_dyn(linear_fwd_resident_kernel<T, KD>, dim3(kResidentWgs), dim3(64 * kResidentWaves), lds, st, a, plan);
    return two_row_tiles(a.rows) ? fwd_run<T, KD, 2, false>(a, st) : fwd_run<T, KD, 1, false>(a, st);
  }
  else return hipErrorInvalidConfiguration;
}

template <typename T>
hipError_t fwd_k(const LinearFwdArgs& a, hipStream_t st) {
  switch (a.K) {
    case 32: return fwd_rows<T, 32>(a, st);
    case 64: return fwd_rows<T, 64>(a, st);
    case 128: return fwd_rows<T, 128>(a, st);
    case 256: return fwd_rows<T, 256>(a, st);
  }
  return hipErrorInvalidConfiguration;
}

template <typename T, int KD>
hipError_t gate_bwd_run(LinearGateBwdArgs a, hipStream_t st) {
  constexpr int chunk_bytes = KD * 32 * (int)sizeof(T), kMost = 4;
  const int64_t blocks = (a.rows + 127) / 128;
  split_chunks(blocks, a.C / 32, kMost, 256, a.chunks, a.groups);
  return launch_dyn(linear_gate_bwd_kernel<T, KD, kMost>, row_grid(a.rows, 128, a.groups), dim3(256), a.chunks * chunk_bytes, st, a);
}

template <typename T>
hipError_t gate_bwd_k(const LinearGateBwdArgs& a, hipStream_t st) {
  switch (a.K) {
    case 32: return gate_bwd_run<T, 32>(a, st);
    case 64: return gate_bwd_run<T, 64>(a, st);
    case 128: return gate_bwd_run<T, 128>(a, st);
  }
  return hipErrorInvalidConfiguration;
}

template <typename T, int KD>
hipError_t dx_run(const LinearDxArgs& a, hipStream_t st) {
  // (wherever the weights fit, from the smallest sizes on: K = 128, 17 chunks, 500 rows 15.6 -> 11.0 us, 2^20
  // 320 -> 276; K = 64 13.5 -> 8.6 and 253 -> 243; K = 32 12.6 -> 7.6 and 221 -> 225)
  const ResidentPlan plan = resident_plan(a);
  const int lds = linear_dx_lds(KD, plan.chunks);
  if (plan.chunks && a.rows < (int64_t(1) << 31) && lds <= kResidentLds)
    return launch_dyn(linear_dx_resident_kernel<T, KD>, dim3(kResidentWgs), dim3(64 * kResidentWaves), lds, st, a, plan);
  const dim3 block(256);
  if (two_row_tiles(a.rows)) hipLaunchKernelGGL((linear_dx_kernel<T, KD, 2>), dim3((unsigned)((a.rows + 255) / 256)), block, 0, st, a);
  else hipLaunchKernelGGL((linear_dx_kernel<T, KD, 1>), dim3((unsigned)((a.rows + 127) / 128)), block, 0, st, a);
  return hipGetLastError();
}

template <typename T>
hipError_t dx_k(const LinearDxArgs& a, hipStream_t st) {
  switch (a.K) {
    case 32: return dx_run<T, 32>(a, st);
    case 64: return dx_run<T, 64>(a, st);
    case 128: return dx_run<T, 128>(a, st);
  }
  return hipErrorInvalidConfiguration;
}

template <typename T, int KD>
hipError_t dw_run(const LinearDwArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((a.chunks + 7) / 8 * 8 * a.groups));
  hipError_t e;
  if (!a.g && linear_dw_words(a.n, a.nlayers, a.rider)) {
    e = launch_dyn(linear_dw_kernel<T, KD, kDwWords>, grid, dim3(512), LinearDwShape<T, KD, kDwWords>::LDS, st, a);
  } else if (!a.g) {
    e = launch_dyn(linear_dw_kernel<T, KD, kDwPlain>, grid, dim3(512), LinearDwShape<T, KD, kDwPlain>::LDS, st, a);
  } else if (!a.gw) {
    e = launch_dyn(linear_dw_kernel<T, KD, kDwGated>, grid, dim3(512), LinearDwShape<T, KD, kDwGated>::LDS, st, a);
  } else {
    if constexpr (KD == 64 || KD == 128) e = launch_dyn(linear_dw_kernel<T, KD, kDwGateBwd>, grid, dim3(512), LinearDwShape<T, KD, kDwGateBwd>::LDS, st, a);
    else return hipErrorInvalidConfiguration;
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((linear_dw_reduce_kernel<T>), dim3((unsigned)((a.total + 31) / 32)), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <typename T>
hipError_t dw_k(const LinearDwArgs& a, hipStream_t st) {
  switch (a.K) {
    case 32: return dw_run<T, 32>(a, st);
    case 64: return dw_run<T, 64>(a, st);
    case 128: return dw_run<T, 128>(a, st);
    case 256: return dw_run<T, 256>(a, st);
  }
  return hipErrorInvalidConfiguration;
}

}  // namespace

hipError_t linear_fwd_launch(LinearFwdArgs a, int dtype, hipStream_t st) { return dtype == kBF16 ? fwd_k<__bf16>(a, st) : fwd_k<_Float16>(a, st); }
hipError_t linear_gate_bwd_launch(LinearGateBwdArgs a, int dtype, hipStream_t st) { return dtype == kBF16 ? gate_bwd_k<__bf16>(a, st) : gate_bwd_k<_Float16>(a, st); }
hipError_t linear_dx_launch(const LinearDxArgs& a, int dtype, hipStream_t st) { return dtype == kBF16 ? dx_k<__bf16>(a, st) : dx_k<_Float16>(a, st); }
hipError_t linear_dw_launch(const LinearDwArgs& a, int dtype, hipStream_t st) { return dtype == kBF16 ? dw_k<__bf16>(a, st) : dw_k<_Float16>(a, st); }

}  // namespace tri
