// Where the float64 logistic passes read the row-major X[N][D] of a posterior:
// integer functions without device code, so that a host program can evaluate them
// over every width and remainder (they have to stay inside the row, and inside
// the last row of X).
#pragma once

#include <stdint.h>

#include <type_traits>

namespace gjx {
namespace logistic {

// f(integral_constant<NB>) with the number of 16-feature tiles of a posterior of D
// features, 16 (NB - 1) < D <= 16 NB: the passes limit the columns of the last tile
// only, so every tile before it has to lie inside the row.
template <int MAXD, class F>
__attribute__((always_inline)) constexpr void by_width(int D, F f) {
  static_assert(MAXD == 64 || MAXD == 128, "feature capacity 64 or 128");
  if constexpr (MAXD == 64) {
    if (D <= 16) f(std::integral_constant<int, 1>{});
    else if (D <= 32) f(std::integral_constant<int, 2>{});
    else if (D <= 48) f(std::integral_constant<int, 3>{});
    else f(std::integral_constant<int, 4>{});
  } else {
    if (D <= 80) f(std::integral_constant<int, 5>{});
    else if (D <= 96) f(std::integral_constant<int, 6>{});
    else if (D <= 112) f(std::integral_constant<int, 7>{});
    else f(std::integral_constant<int, 8>{});
  }
}

// Bytes from row n0 to row n0 + r, given as rowb = 8 r D (r < 16); rows past N - 1 become row N - 1.
constexpr uint32_t row_bytes(uint32_t rowb, int n0, int N, int D) {
  const int left = N - n0 - 1 < 15 ? N - n0 - 1 : 15;
  const uint32_t last = 8u * (uint32_t)(left * D);
  return rowb < last ? rowb : last;
}

// Bytes from a row's start to feature f of the last of NB tiles (f < 16); features
// past D - 1 become feature D - 1.
constexpr uint32_t last_tile_bytes(int NB, int f, int D) {
  const int c = 16 * (NB - 1) + f;
  return 8u * (uint32_t)(c < D - 1 ? c : D - 1);
}

// Feature of K step s in lane group g of the quadratic-form pass (s even: that and the next are neighbours)
constexpr int quad_feature(int s, int g) { return 8 * (s / 2) + 2 * g + s % 2; }

}  // namespace logistic
}  // namespace gjx
