// The two codebook tables, generated at compile time (qs_codebook.hip puts
// them into __constant__ memory; no initialisation call on any device).  Plain
// C++: compiles on the host too.
#pragma once

namespace qs {

// ----------------------------------------------------------------------------
// Codebook tables, built by constexpr code so that no initialisation call is
// needed on any device.
//
// E8P abs table (quipsharp/codebooks/e8p.py:64-89): rows 0..226 are every abs
// pattern over {1/2,3/2,5/2,7/2}^8 with squared norm <= 10 in ascending
// lexicographic order; rows 227..255 are the 29 norm^2 = 12 padding rows of the
// QuIP# paper (Appendix C.1) in the reference's order; finally each row whose
// coordinate sum is odd has its last coordinate negated.
// ----------------------------------------------------------------------------
struct Table8 {
  float v[256][8];
};

namespace detail {
// k[i] is the half-integer index (value k + 1/2); budget bounds sum k(k+1).
constexpr void e8p_enum(Table8& t, int& n, int pos, int budget, int* k) {
  if (pos == 8) {
    for (int i = 0; i < 8; ++i) t.v[n][i] = (float)k[i] + 0.5f;
    ++n;
    return;
  }
  for (int v = 0; v < 4; ++v) {
    int c = v * (v + 1);
    if (c > budget) break;
    k[pos] = v;
    e8p_enum(t, n, pos + 1, budget - c, k);
  }
}
// Padding rows, each digit a numerator over 2.
constexpr const char* kPad29[29] = {
    "31113333", "13113333", "11313333", "11133333", "33313311", "33313131",
    "33311331", "33313113", "33311313", "33311133", "33133311", "33133131",
    "33131331", "33133113", "33131313", "33131133", "31333311", "31333131",
    "31331331", "31333113", "31331313", "13331133", "13333311", "13333131",
    "13331331", "13333113", "13331313", "11331333", "33113331"};

// Integer / half-integer shells of E8 in itertools.product order (last
// coordinate fastest).  vals are doubled integers (value = vals/2).
constexpr void e8_shell(Table8& t, int& n, int cap, const int* vals, int nv, int pos,
                        int norm4_left, int sum2, int* cur) {
  if (n >= cap) return;
  if (pos == 8) {
    if (norm4_left != 0) return;
    if ((sum2 / 2) % 2 != 0) return;  // coordinate sum must be even
    for (int i = 0; i < 8; ++i) t.v[n][i] = (float)cur[i] * 0.5f;
    ++n;
    return;
  }
  for (int j = 0; j < nv && n < cap; ++j) {
    int v = vals[j];
    int sq = v * v;
    if (sq > norm4_left) continue;
    cur[pos] = v;
    e8_shell(t, n, cap, vals, nv, pos + 1, norm4_left - sq, sum2 + v, cur);
  }
}
}  // namespace detail

constexpr Table8 make_e8p_table() {
  Table8 t{};
  int n = 0;
  int k[8] = {};
  detail::e8p_enum(t, n, 0, 8, k);
  for (int r = 0; r < 29; ++r, ++n)
    for (int i = 0; i < 8; ++i) t.v[n][i] = (float)(detail::kPad29[r][i] - '0') * 0.5f;
  for (int r = 0; r < 256; ++r) {
    int s2 = 0;
    for (int i = 0; i < 8; ++i) s2 += (int)(t.v[r][i] * 2.0f);
    if ((s2 / 2) % 2 != 0) t.v[r][7] = -t.v[r][7];
  }
  return t;
}

// E8 one-bit table (quipsharp/codebooks/e8_1bit.py:26-70): zero, the 112
// integer and 128 half-integer norm^2 = 2 vectors, then the first 15 integer
// norm^2 = 4 vectors, each group in cartesian-product order.
constexpr Table8 make_e81_table() {
  Table8 t{};
  int n = 1;  // row 0 stays zero
  int cur[8] = {};
  const int ints1[3] = {-2, 0, 2};                  // {-1,0,1} doubled
  const int halves[4] = {-3, -1, 1, 3};             // {-3/2,...,3/2} doubled
  const int ints2[5] = {-4, -2, 0, 2, 4};           // {-2,...,2} doubled
  detail::e8_shell(t, n, 256, ints1, 3, 0, 8, 0, cur);   // norm^2 2 -> doubled norm 8
  detail::e8_shell(t, n, 256, halves, 4, 0, 8, 0, cur);
  int cap = n + 15;
  detail::e8_shell(t, n, cap, ints2, 5, 0, 16, 0, cur);  // norm^2 4 -> 16
  return t;
}

constexpr Table8 kE8PHost = make_e8p_table();
constexpr Table8 kE81Host = make_e81_table();

}  // namespace qs
