// How many waves take a pair row in the row-resident backward of short rows (up to 512 keys, head dims 16 and 32): the kernel of
// tri_bwd_row_short.hpp with one wave or two, or the four waves of tri_bwd_row.hpp.  Plain C++, so that the rule can be checked where there is no GPU.
#pragma once
#include <cstdint>

namespace tri {

enum class RowForm { kOneWave, kTwoWaves, kFourWaves };

// nwords: key tiles of a row; per_xcd: rows of the launch per XCD (32 compute units).  A compute unit takes four rows of one wave side by side, two
// of two waves, two of four waves (one above 256 keys).  One wave of up to eight key tiles costs the least per row but takes a row for longest: launches
// that leave SIMDs without a wave, and those whose last round of 128 rows per XCD is nearly empty, spread a row over more.
//
// This kernel alone, bf16, h heads.  Few rows, d = 32, us, one wave / two / four: 9 rows per XCD (h = 1, n = 70) 13.3 / 12.9 / 12.6, 27 (h = 3, n = 70)
// 13.6 / 13.2 / 12.8, 32 (h = 2, n = 128) 15.8 / 13.9 / 14.0, 35 (h = 4, n = 70) 14.0 / 13.6 / 14.9, 64 (h = 4, n = 128) 18.3 / 16.5 / 18.3, 65 (h = 5,
// n = 100) 18.4 / 23.9 / 24.3; one wave / four: six key tiles 43 (h = 2, n = 170) 26.4 / 22.2, 66 (h = 3) 28.4 / 31.4, seven 75 (h = 3, n = 200) 33.9 / 34.1, eight 64
// (h = 2, n = 256) 38.6 / 29.7, 87 (h = 3, n = 230) 41.4 / 38.9, 96 (n = 256) 41.0 / 39.9, 128 (h = 4) 45.4 / 48.1.
// More than one round, four waves over one wave at d = 16 and 32 by rows per XCD: five key tiles 140 1.02 1.02, 260 1.10 1.04; six 129 0.88 0.86, 154 0.92
// 0.94, 168 1.01 1.01, 240 1.20 1.14, 264 0.98 0.96, 301 1.03 1.02; seven 140 0.83 0.85, 175 0.91 0.91, 200 1.01 0.99, 250 1.07 1.05, 280 0.88 0.90,
// 325 1.01 0.99, 364 1.08 1.00, 400 0.89 0.87, 450 1.01 0.93, 600 1.00 0.95; eight 115 1.04 1.05, 145 0.74 0.78, 192 0.84 0.84, 256 0.99 1.00, 288
// 0.80 0.83, 384 0.96 0.94, 512 0.96 0.90, 768 0.93 0.92.  Above 256 keys four waves over two: 9 to 16 key tiles 1.03 to 1.38, but for 11 and 12 with
// 83 rows 0.97 0.96 and 96 0.98 0.99 (144 1.05 1.07).
constexpr RowForm bwd_row_form(int nwords, int d, int64_t per_xcd) {
  const int64_t last_round = (per_xcd - 1) % 128 + 1;
  if (nwords <= 2) return RowForm::kOneWave;
  if (nwords <= 4) return per_xcd <= 32 ? RowForm::kFourWaves : per_xcd <= 64 ? RowForm::kTwoWaves : RowForm::kOneWave;
  if (nwords <= 8) {
    const bool few = per_xcd <= (nwords == 8 ? 96 : 64);
    const bool nearly_empty = per_xcd > 128 && (nwords == 8 || (nwords == 7 && (last_round <= 64 || (d == 32 && per_xcd > 384))) || (nwords == 6 && last_round <= 32));
    return few || nearly_empty ? RowForm::kFourWaves : RowForm::kOneWave;
  }
  return (nwords == 11 || nwords == 12) && per_xcd > 64 && per_xcd <= 96 ? RowForm::kFourWaves : RowForm::kTwoWaves;
}

}  // namespace tri
