// Nearest-codeword search of one vector in one lane, without visiting the
// tables' 512 (E8P) or 256 (E8 one-bit) candidates.
//
// E8P.  At a shift, with magnitudes a_i = |x_i +- 1/4|, a table row with
// entries T has the distance sum (a_i - T_i)^2, plus 4 min a_i T_i where its
// signing has the wrong parity (quipsharp/codebooks/e8p.py:104-128, the greedy
// repair).  Rows 0 .. 226 are every arrangement of seven multisets of entries:
// all 1/2 with j = 0 .. 4 entries of 3/2, or with one 5/2 and up to one 3/2
// (64 rows).  By the rearrangement inequality the best row of a multiset gives
// the large entries to the large magnitudes, penalty included (the least
// product is then 1/2 times the least magnitude), and any other row of the
// multiset is worse by at least twice the least gap between two neighbours in
// the sorted magnitudes where its entries differ.  So sorting the eight
// magnitudes gives the best row of seven multisets and a lower bound for every
// other row; the 29 rows with five entries of 3/2 (not every arrangement is in
// the table) are evaluated one by one through the sum of their three other
// magnitudes.  About 350 operations per shift instead of 256 x ~25.
//
// E8 one-bit (quipsharp/codebooks/e8_1bit.py:66-83): zero, the 112 rows of two
// +-1 (the two largest magnitudes), the 128 rows of +-1/2 with an even number
// of minus signs (the signs of x, the least magnitude flipped where their
// number is odd), and the 15 rows of norm 4 one by one.
//
// These distances are not rounded as the reference rounds them, so the answer
// counts only when the best and the second-best candidate are further apart
// than both roundings together (`certain`); the caller evaluates every
// candidate in the reference's arithmetic otherwise (ties, near-ties and
// non-finite inputs).  Compiles on the host too (tests/test_e8_search.py).
#pragma once

#include <stdint.h>
#include <string.h>

#include <utility>

#include "qs_tables.h"

#ifdef __HIP__
#define QS_HD __host__ __device__ __forceinline__
#define QS_UNROLL _Pragma("unroll")
#else
#define QS_HD inline
#define QS_UNROLL
#endif

namespace qs {

// ---- lookup tables -------------------------------------------------------
// An E8P row as a pattern: two bits per coordinate, entry - 1/2 (0, 1 or 2).
// The last coordinate's sign is negative where the number of 1s is odd.
constexpr int kE8PSel = 349;  // [0, 256): mask of the 3/2 entries; 256 + 8 u + v: 5/2 at u, 3/2 at v (u = v: none);
                              // 320 + i: row 227 + i
struct E8Luts {
  uint32_t sel[kE8PSel + 3];  // row | pattern << 8
  uint32_t pat[256];          // pattern of a row
  uint32_t one[256];          // E8 one-bit row: four bits per coordinate, 2 value + 8
  uint32_t pair[256];         // E8 one-bit row of two +-1: [i][j][x_i > 0][x_j > 0], i < j
  uint32_t low[32];           // E8P row 227 + i: its three coordinates of 1/2, a byte each (i < 29)
};

// Coordinates of row 227 + i that hold 1/2 (there are three).
constexpr int e8p_low(int i, int n) {
  int c = 0;
  for (int k = 0; k < 8; ++k) {
    const float v = kE8PHost.v[227 + i][k];
    if (v == 0.5f || v == -0.5f) {
      if (c == n) return k;
      ++c;
    }
  }
  return -1;
}

constexpr E8Luts make_e8_luts() {
  E8Luts t{};
  for (int r = 0; r < 256; ++r) {
    uint32_t pat = 0, mask = 0;
    int two = -1, one = -1;
    for (int i = 0; i < 8; ++i) {
      const float v = kE8PHost.v[r][i];
      const int k = (int)(v < 0 ? -v : v);
      pat |= (uint32_t)k << (2 * i);
      if (k == 1) mask |= 1u << i, one = i;
      if (k == 2) two = i;
    }
    t.pat[r] = pat;
    const int at = r >= 227 ? 320 + r - 227 : two < 0 ? (int)mask : 256 + 8 * two + (one < 0 ? two : one);
    t.sel[at] = (uint32_t)r | (pat << 8);
  }
  for (int r = 0; r < 256; ++r) {
    uint32_t w = 0;
    int n = 0, at[8] = {}, pos[8] = {};
    for (int i = 0; i < 8; ++i) {
      const int two = (int)(kE81Host.v[r][i] * 2.0f);
      w |= (uint32_t)(two + 8) << (4 * i);
      if (two == 2 || two == -2) at[n] = i, pos[n] = two > 0, ++n;
    }
    t.one[r] = w;
    if (r >= 1 && r <= 112) t.pair[at[0] * 32 + at[1] * 4 + pos[0] * 2 + pos[1]] = (uint32_t)r;
  }
  for (int i = 0; i < 29; ++i)
    t.low[i] = (uint32_t)(e8p_low(i, 0) | e8p_low(i, 1) << 8 | e8p_low(i, 2) << 16);
  return t;
}

QS_HD uint32_t as_bits(float f) { return __builtin_bit_cast(uint32_t, f); }
QS_HD float as_value(uint32_t u) { return __builtin_bit_cast(float, u); }
QS_HD float min2(float a, float b) { return __builtin_fminf(a, b); }
QS_HD uint32_t umin2(uint32_t a, uint32_t b) { return a < b ? a : b; }
QS_HD uint32_t umax2(uint32_t a, uint32_t b) { return a > b ? a : b; }

// The two least values of a running set (m1 <= m2).
QS_HD void take(float& m1, float& m2, float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  m2 = __builtin_amdgcn_fmed3f(m1, m2, v);
#else
  m2 = min2(m2, __builtin_fmaxf(m1, v));
#endif
  m1 = min2(m1, v);
}
QS_HD void take(float& m1, float& m2, uint32_t& sel, float v, uint32_t s) {
  sel = v < m1 ? s : sel;
  take(m1, m2, v);
}

// Magnitudes with their coordinate in the three low bits (8e-7 relative), in
// descending order: Batcher's 19 exchanges, on the bits (positive floats order
// as integers).
QS_HD void sort8(uint32_t (&k)[8]) {
  auto cx = [&](int i, int j) {
    const uint32_t hi = umax2(k[i], k[j]), lo = umin2(k[i], k[j]);
    k[i] = hi;
    k[j] = lo;
  };
  cx(0, 1); cx(2, 3); cx(4, 5); cx(6, 7);
  cx(0, 2); cx(1, 3); cx(4, 6); cx(5, 7);
  cx(1, 2); cx(5, 6);
  cx(0, 4); cx(1, 5); cx(2, 6); cx(3, 7);
  cx(2, 4); cx(3, 5);
  cx(1, 2); cx(3, 4); cx(5, 6);
}

// ---- E8P -----------------------------------------------------------------
struct E8Best {
  float best, second;  // least and second-least distance found
  float slack;         // the two are decided where they differ by more
  uint32_t sel;        // E8P: index into E8Luts::sel; E8 one-bit: the row
};

// The 29 rows with five entries of 3/2: twice the sum of the other three
// magnitudes over the least such sum of any three, plus the parity repair;
// least and second least, the row's number in the five low bits (31 ulp of
// what is left after that subtraction).
QS_HD void take_five(uint32_t& q1, uint32_t& q2, uint32_t v) {
  q2 = umin2(q2, umax2(q1, v));
  q1 = umin2(q1, v);
}
QS_HD uint32_t five_value(float a, float b, float c, float floor3, float cap, float odd2, uint32_t i) {
  const float over = (a + b + c) - floor3;
  const float least = min2(min2(a, b), min2(c, cap));
  return (as_bits(__builtin_fmaf(odd2, least, 2.0f * over)) & ~31u) | i;
}
struct AllFives {  // in one lane
  template <int... I>
  QS_HD void each(const float (&a)[8], float floor3, float cap, float odd2, uint32_t& q1, uint32_t& q2,
                  std::integer_sequence<int, I...>) const {
    (take_five(q1, q2, five_value(a[e8p_low(I, 0)], a[e8p_low(I, 1)], a[e8p_low(I, 2)], floor3, cap, odd2, I)), ...);
  }
  QS_HD void operator()(const float (&a)[8], float floor3, float cap, float odd2, uint32_t& q1,
                        uint32_t& q2) const {
    each(a, floor3, cap, odd2, q1, q2, std::make_integer_sequence<int, 29>());
  }
};

// The best row for x shifted by `shift` (+1/4: shift bit 0, -1/4: bit 1);
// fives(a, floor3, cap, odd2, q1, q2) leaves the least two values of the 29 rows.
template <class Fives>
QS_HD E8Best e8p_search(const float (&x)[8], float shift, const Fives& fives) {
  float a[8], s0 = 0.0f, sum = 0.0f;
  uint32_t k[8], sx = 0;
  QS_UNROLL for (int i = 0; i < 8; ++i) {
    const float xs = x[i] + shift;
    sx ^= as_bits(xs);
    a[i] = __builtin_fabsf(xs);
    k[i] = (as_bits(a[i]) & ~7u) | (uint32_t)i;
    const float d = a[i] - 0.5f;
    s0 = __builtin_fmaf(d, d, s0);
    sum += a[i];
  }
  const bool odd_even = sx >> 31;                    // an even number of 3/2 entries: the last entry is positive
  const bool odd_odd = odd_even != (a[7] != 0.0f);   // odd: negative (a product of zero never flips)
  sort8(k);
  float A[8];
  QS_UNROLL for (int i = 0; i < 8; ++i) A[i] = as_value(k[i]);
  const float pe = odd_even ? 2.0f * A[7] : 0.0f, po = odd_odd ? 2.0f * A[7] : 0.0f;
  const float g1 = A[0] - A[1], g2 = A[1] - A[2], g3 = A[2] - A[3], g4 = A[3] - A[4];
  // values relative to s0, the distance of the row of 1/2s
  float m1 = pe, m2 = __builtin_huge_valf();
  uint32_t sel = 0, mask = 0;
  float f = 0.0f;
  const float gap[4] = {g1, g2, g3, g4};
  QS_UNROLL for (int j = 0; j < 4; ++j) {
    f += 2.0f - 2.0f * A[j];
    mask |= 1u << (k[j] & 7);
    const float v = f + (j & 1 ? pe : po);
    take(m1, m2, sel, v, mask);
    m2 = min2(m2, __builtin_fmaf(2.0f, gap[j], v));
  }
  const uint32_t u = k[0] & 7, w = k[1] & 7;
  const float t = 6.0f - 4.0f * A[0];
  const float p0 = t + pe, p1 = t + (2.0f - 2.0f * A[1]) + po;
  take(m1, m2, sel, p0, 256 + 9 * u);
  m2 = min2(m2, __builtin_fmaf(4.0f, g1, p0));
  take(m1, m2, sel, p1, 256 + 8 * u + w);
  m2 = min2(m2, __builtin_fmaf(2.0f, min2(g1, g2), p1));
  uint32_t q1 = ~0u, q2 = ~0u;
  // a little below the least sum of three, so that no value is negative
  const float floor3 = __builtin_fmaf(-1e-5f, A[0], A[5] + A[6] + A[7]) - 1e-30f;
  fives(a, floor3, 3.0f * A[7], odd_odd ? 2.0f : 0.0f, q1, q2);
  const float base = 10.0f - 2.0f * (sum - floor3);
  take(m1, m2, sel, base + as_value(q1), 320 + (q1 & 31));
  m2 = min2(m2, base + as_value(q2));
  E8Best b;
  b.best = s0 + m1;
  b.second = s0 + m2;
  // Error of one candidate, this search's and the reference's rounding
  // together: keys 8.4e-6 A_0 (10 A_0 at 7 ulp), ~12 roundings at up to
  // 8 + 8 A_0, s0's nine and the reference's 24 at up to s0 + 2 A_0: 1.8e-5 A_0
  // + 1.3e-6 s0 + 6e-6; of the 29 rows 31 ulp of their value too.  Two
  // candidates; the caller adds the slacks of both shifts (whose A_0 differ by
  // up to 1/2).
  b.slack = __builtin_fmaf(8e-6f, as_value(q1),
                           __builtin_fmaf(2e-6f, s0, __builtin_fmaf(1.9e-5f, A[0], 1.2e-5f)));
  b.sel = sel;
  return b;
}

// Both shifts: shift bit in sb.
QS_HD E8Best e8p_search2(const float (&x)[8], int& sb, bool& certain) {
  const E8Best p = e8p_search(x, 0.25f, AllFives()), m = e8p_search(x, -0.25f, AllFives());
  const bool first = p.best <= m.best;
  sb = first ? 0 : 1;
  E8Best r = first ? p : m;
  r.second = min2(r.second, first ? m.best : p.best);
  r.slack = p.slack + m.slack;
  certain = r.second - r.best > r.slack;  // false for NaN
  return r;
}

// ---- E8 one-bit ----------------------------------------------------------
template <int R, int I>
QS_HD void e81_term(const float (&x)[8], float& dot) {
  constexpr float t = kE81Host.v[R][I];
  if constexpr (t == 1.0f) dot += x[I];
  else if constexpr (t == -1.0f) dot -= x[I];
  else if constexpr (t != 0.0f) dot = __builtin_fmaf(t, x[I], dot);
}
template <int R>
QS_HD void e81_four(const float (&x)[8], float& m1, float& m2, uint32_t& sel) {
  float dot = 0.0f;
  e81_term<R, 0>(x, dot); e81_term<R, 1>(x, dot); e81_term<R, 2>(x, dot); e81_term<R, 3>(x, dot);
  e81_term<R, 4>(x, dot); e81_term<R, 5>(x, dot); e81_term<R, 6>(x, dot); e81_term<R, 7>(x, dot);
  take(m1, m2, sel, __builtin_fmaf(-2.0f, dot, 4.0f), R);
}
template <int... I>
QS_HD void e81_fours(const float (&x)[8], float& m1, float& m2, uint32_t& sel, std::integer_sequence<int, I...>) {
  (e81_four<241 + I>(x, m1, m2, sel), ...);
}

// The best row for x; sel: the row, or 256 + index into E8Luts::pair.
QS_HD E8Best e81_search(const float (&x)[8], bool& certain) {
  uint32_t k[8], sx = 0, bits = 0, pos = 0;
  float sum = 0.0f, x2 = 0.0f;
  QS_UNROLL for (int i = 0; i < 8; ++i) {
    const uint32_t u = as_bits(x[i]), neg = u >> 31;
    sx ^= u;
    pos |= (neg ^ 1u) << i;
    if (i < 7) bits |= (neg ^ 1u) << (6 - i);
    const float b = __builtin_fabsf(x[i]);
    k[i] = (as_bits(b) & ~7u) | (uint32_t)i;
    sum += b;
    x2 = __builtin_fmaf(b, b, x2);
  }
  sort8(k);
  float A[8];
  QS_UNROLL for (int i = 0; i < 8; ++i) A[i] = as_value(k[i]);
  // values relative to |x|^2, the distance of the zero row
  float m1 = 0.0f, m2 = __builtin_huge_valf();
  uint32_t sel = 0;
  const uint32_t u = k[0] & 7, w = k[1] & 7;
  const uint32_t i = umin2(u, w), j = umax2(u, w);
  const float v2 = 2.0f - 2.0f * (A[0] + A[1]);
  take(m1, m2, sel, v2, 256 + i * 32 + j * 4 + ((pos >> i) & 1) * 2 + ((pos >> j) & 1));
  m2 = min2(m2, v2 + min2(2.0f * (A[1] - A[2]), 4.0f * A[1]));
  const bool odd = sx >> 31;
  const float vh = 2.0f - sum + (odd ? 2.0f * A[7] : 0.0f);
  const uint32_t last = k[7] & 7;
  const uint32_t flip = odd && last < 7 ? 64u >> last : 0u;
  take(m1, m2, sel, vh, 113 + (bits ^ flip));
  m2 = min2(m2, vh + 2.0f * (odd ? A[6] - A[7] : A[6] + A[7]));
  e81_fours(x, m1, m2, sel, std::make_integer_sequence<int, 15>());
  E8Best b;
  b.best = x2 + m1;
  b.second = x2 + m2;
  // two candidates, each 8.4e-6 A_0 (keys at 7 ulp, ~10 roundings at up to
  // 4 + 8 A_0) + 1.2e-6 |x|^2 (both sums) + 2e-6
  b.slack = __builtin_fmaf(4e-6f, x2, __builtin_fmaf(3e-5f, A[0], 8e-6f));
  b.sel = sel;
  certain = b.second - b.best > b.slack;
  return b;
}

}  // namespace qs
