// The coefficient rows that the many-density synthesis reads, step by step: (l, m) with l running
// inside m, one row per harmonic (m = 0: q; m > 0: cos at q, sin at q + 1), qbytes apart.
#pragma once

namespace napmo {

// Loads run ahead of the products, whole groups of steps at a time, so they go on past the last
// harmonic: from there on (and for the sin row that m = 0 does not have) they repeat the last row.
// The clamp is what keeps them inside the table: a buffer load's range check does not have to
// count its scalar offset.
struct SynthRows {
  int l = 0, m = 0, row = 0;

  constexpr int cos_row(int last) const { return row < last ? row : last; }
  constexpr int sin_row(int qbytes, int last) const { return row + qbytes < last ? row + qbytes : last; }
  constexpr void next(int lmax, int qbytes) {
    row += m ? 2 * qbytes : qbytes;
    const bool end = l == lmax;
    m += end ? 1 : 0;
    l = end ? m : l + 1;
  }
};

}  // namespace napmo
