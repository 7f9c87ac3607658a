// Input and output transforms of a long batch of rows (prefill), one row per
// wave and no exchange between waves.
//
// T = M (x) H_256 over the index 256 c + t (M = K_p (x) H_{L/256}, S = n / 256
// <= 128 chunks).  A wave holds 16 rows of M (output slices 16 k .. 16 k + 15)
// and one activation row: M first, on the matrix cores, then H_256.
//  * Operand: lane (q, r16) loads chunks c = 32 kb + 8 q + i (i < 8) at columns
//    t = 128 th + 8 r16 .. + 7, 16 bytes each, and transposes the 8 x 8 block in
//    registers (one v_perm_b32 per pair): the fragment of column set u (t = 128
//    th + 8 r16 + u) has c contiguous, as the MFMA's k index wants it.
//  * Result (the row's operand as MFMA operand A, M as B): lane (q, r16) holds
//    slice r16 at t = 128 th + 32 q + 8 j + u, j < 4, u < 8, so that H_256 is
//    six stages in registers (bits of u, j and th) and two across the four rows
//    of lanes.  Those two swap a register bit with the lane bit as they go
//    (v_permlane16_swap / 32_swap of two registers, then their sum and
//    difference: three instructions for two values), which leaves lane row q at
//    t = 128 th + 32 j + 8 q + u: eight consecutive columns in registers, one
//    16-byte word.  (fp32 partial sums: four columns per lane, t = 64 x + 4 r16
//    + u, by the same scheme.)
// So there is no LDS traffic but M's fragments and the signs, no barrier in the
// loop, and a CU has eight independent rows in flight.  The per-row kernels of
// the short batches (qs_linear_batched.hip, qs_linear_big.hip) spread one row
// over 16 waves with three barriers, which is the shorter chain for a few rows
// but leaves a CU waiting when there are many.
// Rows longer than 16 chunks are read once per group of 16 slices.  On the input
// side the work-groups of a row tile run on one XCD, whose L2 serves the repeats;
// on the output side, with four bytes an element, one work-group takes all the
// groups of a row.
//
// Measured (bf16, sum over a layer's launches, per-row kernels -> this):
//   input, Llama-2-7B   130 rows 35 -> 37 us, 200 39 -> 37, 512 66 -> 45, 2000 212 -> 116
//   input, Qwen3-32B    130 rows 63 -> 53 us, 200 85 -> 57, 512 217 -> 112, 2000 721 -> 282
//   output beyond 12288 (Llama-3-8B gate + up) 130 rows 29 -> ~46 us, 320 57 -> ~42, 2000 360 -> ~150
//   output up to 12288 (Llama-2-7B) 512 rows 62 -> 86 us, 2000 201 -> 231: not taken
//   input, one linear alone (its whole call, 2 bits): 4096 x 4096 160 rows 34.5 -> 36.3, 256 39.6 -> 40.8, 320 39.3
//     -> 40.7, 512 45.4 -> 44.5; 1024 x 1024 256 rows 20.4 -> 21.9, 320 23.9 -> 23.6; 4096 x 11008 200 rows 51.1 ->
//     52.5, 256 54.0 -> 52.8; 4096 x 14336 160 rows 55.7 -> 54.6; 4096 to 3 x 4096 200 rows 52.7 -> 53.3, 256 55.0 -> 53.9
// (up to 256 rows the per-row kernel has every row in work at once), so the
// input runs here from kRowsInMin rows, beyond 12288 from kRowsInMinLong, and the
// output from kRowsOutMin rows beyond 12288.  The output kernel reads the fp32 partial sums once per group
// of 16 slices and splits them each time; up to 12288 qs_linear_batched.hip's
// by_kernel reads them once.  Groups of a row in one work-group instead of one
// each (the layer's calls, 2 bits): Qwen2.5-7B 2000 rows 1382 -> 1333 us, 4000
// 2585 -> 2454, Qwen3-32B 2000 2618 -> 2573, Llama-3-8B 4000 2097 -> 2078.
#include "qs_forward_dev.h"
#include "qs_linear_dev.h"

namespace qs {
namespace {

constexpr int kRowsThreads = 256;
constexpr int kRowsWaves = kRowsThreads / 64;  // rows per tile
constexpr int kRowsMaxS = 128;
// Longest fp32 rows.  Beyond them shorter batches run xin_kernel, which is fp32
// throughout: error against 64 bits at 160 rows of 18944 2.082e-4 there, 2.091e-4
// with two bf16 planes here (25600: 2.084e-4 and 2.097e-4).  fp16 rows, whose M is
// two fp16 planes, have xin_kernel's error at every length (18944: 2.080e-4 both).
constexpr int64_t kRowsMaxFp32 = 16384;
constexpr int kRowsMStr = kRowsMaxS + 8;  // 16-bit words per row of M in LDS
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t perm_lo(uint32_t hi, uint32_t lo) {  // low halves: lo in bits 0-15
  return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}
__device__ __forceinline__ uint32_t perm_hi(uint32_t hi, uint32_t lo) {
  return __builtin_amdgcn_perm(hi, lo, 0x07060302u);
}

// Rows 16 k .. 16 k + 15 of M (zero past S) as two 16-bit planes whose sum is
// the entry to 16 bits or more: truncated bf16, or fp16 for F16.
template <bool F16, int NT = kRowsThreads>
__device__ __forceinline__ void build_m16(uint16_t* Mh, uint16_t* Ml, int k, int S, int Spad, int lsh, int p,
                                          const float* K, int tid) {
  for (int e = tid; e < 16 * Spad; e += NT) {
    const int rr = e / Spad, c = e - rr * Spad;
    const int r = 16 * k + rr;
    const float v = r < S && c < S ? mmat(r, c, lsh, p, K) : 0.0f;
    uint16_t hi, lo;
    if constexpr (F16) {
      const _Float16 h = (_Float16)v;
      hi = __builtin_bit_cast(uint16_t, h);
      lo = __builtin_bit_cast(uint16_t, (_Float16)(v - (float)h));
    } else {
      const uint32_t u = __float_as_uint(v) & 0xFFFF0000u;
      hi = (uint16_t)(u >> 16);
      lo = (uint16_t)(__float_as_uint(v - __uint_as_float(u)) >> 16);
    }
    Mh[rr * kRowsMStr + c] = hi;
    Ml[rr * kRowsMStr + c] = lo;
  }
}

// H_256 of a lane's slice, its 16 / U x U x 4 elements v[x][u][j].  In: t = 16 U x
// + 4 U q + U j + u; out: j and q have changed places, t = 16 U x + 4 U j + U q
// + u.
template <int U>
__device__ __forceinline__ void h256_rows(floatx4 (&v)[16 / U][U]) {
  constexpr int X = 16 / U;
#pragma unroll
  for (int x = 0; x < X; ++x) {
#pragma unroll
    for (int h = 1; h < U; h <<= 1)
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (!(u & h)) {
          const floatx4 a = v[x][u], b = v[x][u + h];
          v[x][u] = a + b;
          v[x][u + h] = a - b;
        }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const floatx4 a = v[x][u];
      const float s0 = a[0] + a[1], d0 = a[0] - a[1], s1 = a[2] + a[3], d1 = a[2] - a[3];
      float w[4] = {s0 + s1, d0 + d1, s0 - s1, d0 - d1};  // both bits of j done
      // the low bit of q on lane bit 4, which takes the low bit of j
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(w[i]), __float_as_uint(w[i + 1]), false, false);
        const float c = __uint_as_float(p[0]), d = __uint_as_float(p[1]);
        w[i] = c + d;
        w[i + 1] = c - d;
      }
      // the high bit of q on lane bit 5, which takes the high bit of j
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(w[i]), __float_as_uint(w[i + 2]), false, false);
        const float c = __uint_as_float(p[0]), d = __uint_as_float(p[1]);
        w[i] = c + d;
        w[i + 2] = c - d;
      }
      v[x][u] = (floatx4){w[0], w[1], w[2], w[3]};
    }
  }
#pragma unroll
  for (int h = 1; h < X; h <<= 1)
#pragma unroll
    for (int x = 0; x < X; ++x)
      if (!(x & h)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const floatx4 a = v[x][u], b = v[x + h][u];
          v[x][u] = a + b;
          v[x + h][u] = a - b;
        }
      }
}

// Which job, slice group and first row tile a work-group takes.
struct RowsSlot {
  int wg0, ngrp, per;  // first work-group, slice groups, work-groups per slice group (a multiple of 32)
};
__device__ __forceinline__ void rows_place(int local, const RowsSlot& s, int& k, int& turn) {
  k = local / s.per;
  turn = local - k * s.per;
}
// First row of a turn's tile: the four tiles of 16 rows, whose words share
// cache lines in the operand, take turns 8 apart (one XCD).
__device__ __forceinline__ int rows_first(int turn) {
  return kRowsWaves * ((turn & ~31) + 4 * (turn & 7) + ((turn >> 3) & 3));
}

// ---------------------------------------------------------------------------
// input transform
// ---------------------------------------------------------------------------
struct WxJob {
  RowsSlot at;
  const float* sv;  // fp32 signs or packed bits
  _Float16* x2h;
  _Float16* sg;
  float* xmul;
};
struct WxArgs {
  const void* x;
  int64_t ldx;
  int B, S, lsh, pn, njobs;
  const float* Kn;
  float scale;
  WxJob job[QS_MAX_GROUP];
};
constexpr int kOutStr = 32 * kRowsWaves + 1;  // words per slice of a tile (one more: distinct banks)
struct WxLds {
  uint16_t Mh[16 * kRowsMStr], Ml[16 * kRowsMStr];
  int plain;                       // every sign is +-1
  uint32_t sign[kRowsMaxS * 32];   // 8 elements: element 2 j in bit 15 - j, 2 j + 1 in bit 31 - j
  uint4 out[16 * kOutStr];         // a tile's operand words: [slice][word of the slice][row]
};

// Four consecutive activations (8 or 16 bytes, aligned), exact in fp32.
template <int XT>
__device__ __forceinline__ float4 load_x4(const void* x, int64_t at) {
  if constexpr (XT == 2) return *reinterpret_cast<const float4*>(static_cast<const float*>(x) + at);
  const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(x) + at);
  if constexpr (XT == 0)
    return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16),
                       __uint_as_float(w.y & 0xFFFF0000u));
  const half2v a = __builtin_bit_cast(half2v, w.x), b = __builtin_bit_cast(half2v, w.y);
  return make_float4((float)a[0], (float)a[1], (float)b[0], (float)b[1]);
}

// How sv meets the activations: 16-bit ones times +-1 are MFMA operands as they
// are; fp32 ones, and the products with other multipliers, enter as two bf16
// planes (truncated, and the remainder rounded), 16 bits or more as in the
// per-row kernels.  Error against 64 bits, bf16 rows of 3584 with multipliers of
// 1.03 .. 2.33: 3.3e-3 as one bf16 plane, 2.1e-4 (the fp16 operand's) as two.
enum class Mul { kExact, kSign, kFactor };

// The rows of a work-group.  A function for each kind of multiplier, so that
// none takes the others' registers (in one loop the 16-bit rows spilled 50).
// XT: 0 bf16, 1 fp16, 2 fp32 activations; LO: M has a second plane (an odd factor).
template <int XT, Mul MUL, bool LO>
__device__ __forceinline__ void wx_rows(const WxArgs& A, const WxJob& J, WxLds& D, int k, int turn) {
  constexpr bool kExact = MUL == Mul::kExact;
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r16 = lane & 15;
  const LaneX lx = lane_x_init();
  const int S = A.S, nkb = (S + 31) >> 5;
  build_m16<kExact && XT == 1>(D.Mh, D.Ml, k, S, 32 * nkb, A.lsh, A.pn, A.Kn, tid);
  __syncthreads();
  // the operand block of (row b, k-step kb, half th), requested one block ahead
  // (the next row's first one during the last block of a row): with two waves
  // per SIMD nothing else covers the loads
  uint4 nx[8];
  auto request = [&](int b, int kb, int th) __attribute__((always_inline)) {
    if constexpr (kExact) {
      const uint16_t* src = static_cast<const uint16_t*>(A.x) + (int64_t)b * A.ldx + 128 * th + 8 * r16;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int c = 32 * kb + 8 * q + i;
        nx[i] = *reinterpret_cast<const uint4*>(src + 256 * (c < S ? c : S - 1));
      }
    }
  };
  const int row = tid >> 6;
  const int turns = (A.B + 32 * kRowsWaves - 1) / (32 * kRowsWaves) * 32;
  auto row_of = [&](int t) { return rows_first(t) + row < A.B ? rows_first(t) + row : A.B - 1; };
  if (turn < turns) request(row_of(turn), 0, 0);

  for (; turn < turns; turn += J.at.per) {
    const int first = rows_first(turn);
    if (first >= A.B) continue;  // the same in every wave
    // rows past the end repeat the last one and are not stored
    const int b = row_of(turn), next = turn + J.at.per < turns ? row_of(turn + J.at.per) : b;
    floatx4 acc[2][8];
#pragma unroll
    for (int th = 0; th < 2; ++th)
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[th][u] = (floatx4){0.f, 0.f, 0.f, 0.f};
    float ss = 0.0f;
    for (int kb = 0; kb < nkb; ++kb) {
      const int c0 = 32 * kb + 8 * q;
      const uint4 ah = *reinterpret_cast<const uint4*>(D.Mh + r16 * kRowsMStr + c0);
      const uint4 al = *reinterpret_cast<const uint4*>(D.Ml + r16 * kRowsMStr + c0);
#pragma unroll
      for (int th = 0; th < 2; ++th) {
        if constexpr (kExact) {
          uint32_t d[8][4];
#pragma unroll
          for (int i = 0; i < 8; ++i) d[i][0] = nx[i].x, d[i][1] = nx[i].y, d[i][2] = nx[i].z, d[i][3] = nx[i].w;
          if (th == 0) request(b, kb, 1);
          else if (kb + 1 < nkb) request(b, kb + 1, 0);
          else request(next, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int c = c0 + i;
            const int at = 32 * (c < S ? c : S - 1) + 16 * th + r16;
            const uint32_t w = D.sign[at];
#pragma unroll
            for (int j = 0; j < 4; ++j) d[i][j] ^= (w << j) & 0x80008000u;
            if (32 * kb + 32 > S && c >= S) d[i][0] = d[i][1] = d[i][2] = d[i][3] = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              if constexpr (XT == 0) {
                const bf16x2_t h = __builtin_bit_cast(bf16x2_t, d[i][j]);
                ss = __builtin_amdgcn_fdot2_f32_bf16(h, h, ss, false);
              } else {
                const half2v h = __builtin_bit_cast(half2v, d[i][j]);
                ss = __builtin_amdgcn_fdot2(h, h, ss, false);
              }
            }
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            uint4 f;
            if (u & 1)
              f = make_uint4(perm_hi(d[1][u >> 1], d[0][u >> 1]), perm_hi(d[3][u >> 1], d[2][u >> 1]),
                             perm_hi(d[5][u >> 1], d[4][u >> 1]), perm_hi(d[7][u >> 1], d[6][u >> 1]));
            else
              f = make_uint4(perm_lo(d[1][u >> 1], d[0][u >> 1]), perm_lo(d[3][u >> 1], d[2][u >> 1]),
                             perm_lo(d[5][u >> 1], d[4][u >> 1]), perm_lo(d[7][u >> 1], d[6][u >> 1]));
            if constexpr (XT == 0) {
              const bf16x8 xf = __builtin_bit_cast(bf16x8, f);
              acc[th][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, __builtin_bit_cast(bf16x8, ah), acc[th][u], 0, 0, 0);
              if constexpr (LO)
                acc[th][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, __builtin_bit_cast(bf16x8, al), acc[th][u], 0, 0, 0);
            } else {
              const half8 xf = __builtin_bit_cast(half8, f);
              acc[th][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf, __builtin_bit_cast(half8, ah), acc[th][u], 0, 0, 0);
              if constexpr (LO)
                acc[th][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf, __builtin_bit_cast(half8, al), acc[th][u], 0, 0, 0);
            }
          }
        } else {  // four columns at a time
          const int64_t src = (int64_t)b * A.ldx + 128 * th + 8 * r16;
#pragma unroll
          for (int uh = 0; uh < 2; ++uh) {
            uint32_t fh[4][4], fl[4][4];  // [u][pair of chunks]
#pragma unroll
            for (int i2 = 0; i2 < 4; ++i2) {
              float v[2][4];
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                const int c = c0 + 2 * i2 + i, cc = c < S ? c : S - 1;
                const float4 f = load_x4<XT>(A.x, src + 256 * cc + 4 * uh);
                const int at = 32 * cc + 16 * th + r16;
                v[i][0] = f.x, v[i][1] = f.y, v[i][2] = f.z, v[i][3] = f.w;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                  const int e = 4 * uh + u;
                  if constexpr (MUL == Mul::kSign)
                    v[i][u] = __uint_as_float(__float_as_uint(v[i][u]) ^
                                              ((D.sign[at] << ((e & 1 ? 0 : 16) + (e >> 1))) & 0x80000000u));
                  else
                    v[i][u] = v[i][u] * J.sv[8 * at + e];
                  if (c >= S) v[i][u] = 0.0f;
                  ss = __builtin_fmaf(v[i][u], v[i][u], ss);
                }
              }
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const uint32_t a = __float_as_uint(v[0][u]), c = __float_as_uint(v[1][u]);
                fh[u][i2] = perm_hi(c, a);
                fl[u][i2] = f32x2_to_bf16x2(v[0][u] - __uint_as_float(a & 0xFFFF0000u),
                                            v[1][u] - __uint_as_float(c & 0xFFFF0000u));
              }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const bf16x8 h = __builtin_bit_cast(bf16x8, make_uint4(fh[u][0], fh[u][1], fh[u][2], fh[u][3]));
              const bf16x8 l = __builtin_bit_cast(bf16x8, make_uint4(fl[u][0], fl[u][1], fl[u][2], fl[u][3]));
              floatx4& t = acc[th][4 * uh + u];
              t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, __builtin_bit_cast(bf16x8, ah), t, 0, 0, 0);
              if constexpr (LO) t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, __builtin_bit_cast(bf16x8, al), t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, __builtin_bit_cast(bf16x8, ah), t, 0, 0, 0);
            }
          }
        }
      }
    }
    const int e = operand_exponent(wave_sum(ss, lx));
    const float mul = ldexpf(A.scale, -e);
    if (k == 0 && lane == 0) J.xmul[b] = ldexpf(1.0f, e);
    h256_rows<8>(acc);
    const int s = 16 * k + r16;
    // The tile's words pass through LDS so that a store covers four rows' words
    // (64 bytes) instead of one row's 16: stored from here they took a third of
    // the kernel's time.
    __syncthreads();  // the previous tile's words have been read
    uint32_t sums[4];
#pragma unroll
    for (int t67 = 0; t67 < 4; ++t67) {
      half2v pair;
#pragma unroll
      for (int t5 = 0; t5 < 2; ++t5) {
        const int th = t67 >> 1, j = t5 + 2 * (t67 & 1);
        half2v h[4];
        float sum = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          h[u] = __builtin_convertvector((f32x2_t){acc[th][2 * u][j] * mul, acc[th][2 * u + 1][j] * mul}, half2v);
          sum = __builtin_amdgcn_fdot2(h[u], (half2v){(_Float16)1.0f, (_Float16)1.0f}, sum, false);
        }
        D.out[r16 * kOutStr + ((q + 4 * t5) * 4 + t67) * kRowsWaves + row] =
            make_uint4(__builtin_bit_cast(uint32_t, h[0]), __builtin_bit_cast(uint32_t, h[1]),
                       __builtin_bit_cast(uint32_t, h[2]), __builtin_bit_cast(uint32_t, h[3]));
        pair[t5] = (_Float16)sum * (_Float16)0.25f;
      }
      sums[t67] = __builtin_bit_cast(uint32_t, pair);
    }
    // group sums: lane row q holds groups q and q + 4 of every 64 columns; swapped
    // so that it holds the eight groups of 64-column quarter q, one word
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const auto p = __builtin_amdgcn_permlane16_swap(sums[i], sums[i + 1], false, false);
      sums[i] = p[0], sums[i + 1] = p[1];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto p = __builtin_amdgcn_permlane32_swap(sums[i], sums[i + 2], false, false);
      sums[i] = p[0], sums[i + 2] = p[1];
    }
    if (s < S && first + row < A.B)
      *reinterpret_cast<uint4*>(J.sg + sg_frag_index(b, 32 * s + 8 * q, S)) =
          make_uint4(perm_lo(sums[1], sums[0]), perm_lo(sums[3], sums[2]), perm_hi(sums[1], sums[0]),
                     perm_hi(sums[3], sums[2]));
    __syncthreads();
    _Float16* xo = J.x2h + frag_index(first, 256 * 16 * k, S);
#pragma unroll
    for (int i = 0; i < 16 * 32 * kRowsWaves / kRowsThreads; ++i) {
      const int n = tid + kRowsThreads * i, sl = n / (32 * kRowsWaves), w = n % (32 * kRowsWaves);
      if (16 * k + sl < S && first + w % kRowsWaves < A.B)
        *reinterpret_cast<uint4*>(xo + (sl * 512 + (w / kRowsWaves) * 16 + w % kRowsWaves) * 8) = D.out[sl * kOutStr + w];
    }
  }
}

// SB: sv is packed sign bits.
template <int XT, bool SB, bool LO>
__global__ __launch_bounds__(kRowsThreads, 2) void wx_kernel(WxArgs A) {
  __shared__ WxLds D;
  const int tid = threadIdx.x;
  int g = 0;
#pragma unroll
  for (int j = 1; j < QS_MAX_GROUP; ++j)
    if (j < A.njobs && (int)blockIdx.x >= A.job[j].at.wg0) g = j;
  const WxJob J = A.job[g];
  const int S = A.S;
  int k, turn;
  rows_place((int)blockIdx.x - J.at.wg0, J.at, k, turn);

  if (tid == 0) D.plain = 1;
  __syncthreads();
  for (int i = tid; i < 32 * S; i += kRowsThreads) {
    uint32_t w = 0;
    if constexpr (SB) {
      const uint32_t b = reinterpret_cast<const uint8_t*>(J.sv)[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) w |= ((b >> (2 * j)) & 1u) << (15 - j) | ((b >> (2 * j + 1)) & 1u) << (31 - j);
    } else {
      const float4 lo = reinterpret_cast<const float4*>(J.sv)[2 * i], hi = reinterpret_cast<const float4*>(J.sv)[2 * i + 1];
      const float s[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      bool one = true;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        one = one && fabsf(s[e]) == 1.0f;
        w |= (__float_as_uint(s[e]) >> 31) << ((e & 1 ? 31 : 15) - (e >> 1));
      }
      if (!one) D.plain = 0;
    }
    D.sign[i] = w;
  }
  __syncthreads();
  const bool plain = SB || __builtin_amdgcn_readfirstlane(D.plain) != 0;
  if (plain) wx_rows<XT, XT == 2 ? Mul::kSign : Mul::kExact, LO>(A, J, D, k, turn);
  else if constexpr (!SB) wx_rows<XT, Mul::kFactor, LO>(A, J, D, k, turn);
}

// ---------------------------------------------------------------------------
// output transform
// ---------------------------------------------------------------------------
// A work-group's 8 waves take turns at the pairs of its rows and groups of 16
// slices, so that the groups of one row are in work at one time and its partial
// sums, which every group needs whole, come from memory once and then from the
// L1 and L2.  (Work-groups with one group each drifted apart: five groups of a
// 18944 wide row fetched 3 GB instead of 0.6.)  M of all the groups is in LDS,
// and the signs as bits; signs that are not +-1 and the bias are read as needed.
constexpr int kWyThreads = 512;
constexpr int kWyWaves = kWyThreads / 64;
constexpr int kMaxGroups16 = kRowsMaxS / 16;
struct WyJob {
  int wg0, per;      // first work-group, work-groups
  const float* y1p;  // [SG][B][m]
  int SG, m, S, lsh, pm, ngrp;
  const float* Km;
  float scale;       // of the transform, times the layer's
  const float* xmul;
  const float* su;
  const float* bias;
  void* y;
  int64_t ldy;
  int wide;          // y rows start on 16 bytes
  int bias_wide;     // the bias starts on 16 bytes
};
struct WyArgs {
  int B, y_dtype, njobs;
  WyJob job[QS_MAX_GROUP];
};
constexpr int kYStr = 256 + 8;  // outputs per slice of a row (16-byte words of two rows in distinct banks)
struct WyLds {
  uint32_t sign[kRowsMaxS * 8];  // bit t % 32 of word t / 32: column t is negative
  uint16_t out[kWyWaves][16 * kYStr];
  uint16_t M[kMaxGroups16][2][16 * kRowsMStr];  // as many groups as the launch has
};
constexpr size_t wy_lds(int groups) {
  return sizeof(WyLds) - (size_t)(kMaxGroups16 - groups) * 2 * 16 * kRowsMStr * sizeof(uint16_t);
}
constexpr int kWyMaxLds = (int)wy_lds(kMaxGroups16);
static_assert(kWyMaxLds <= 160 * 1024, "LDS budget");

// LO: a job's M has a second plane.
template <bool SB, bool LO>
__global__ __launch_bounds__(kWyThreads) void wy_kernel(WyArgs A) {
  extern __shared__ __attribute__((aligned(16))) char wy_sm[];
  WyLds& D = *reinterpret_cast<WyLds*>(wy_sm);
  __shared__ int odd_sign;
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r16 = lane & 15;
  int g = 0;
#pragma unroll
  for (int j = 1; j < QS_MAX_GROUP; ++j)
    if (j < A.njobs && (int)blockIdx.x >= A.job[j].wg0) g = j;
  const WyJob J = A.job[g];
  const int S = J.S, nkb = (S + 31) >> 5;
  const int wg = (int)blockIdx.x - J.wg0;
  for (int k = 0; k < J.ngrp; ++k)
    build_m16<false, kWyThreads>(D.M[k][0], D.M[k][1], k, S, 32 * nkb, J.lsh, J.pm, J.Km, tid);
  if (tid == 0) odd_sign = 0;
  __syncthreads();
  bool odd = false;
  for (int i = tid; i < 8 * S; i += kWyThreads) {
    uint32_t w = 0;
    if constexpr (SB) {
      w = reinterpret_cast<const uint32_t*>(J.su)[i];
    } else {
      for (int t = 0; t < 32; ++t) {
        const float f = J.su[32 * i + t];
        odd = odd || fabsf(f) != 1.0f;
        w |= (f < 0.0f ? 1u : 0u) << t;
      }
    }
    D.sign[i] = w;
  }
  if (odd) odd_sign = 1;
  __syncthreads();
  const bool plain = SB || odd_sign == 0;
  // columns 64 x + 4 r16 .. + 3 of the eight chunks of k-step kb (256 consecutive
  // bytes per 16 lanes), requested one block ahead
  float4 nx[8];
  auto request = [&](int b, int kb, int x, int sg) __attribute__((always_inline)) {
    const float* src = J.y1p + ((int64_t)sg * A.B + b) * J.m + 4 * r16 + 64 * x;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = 32 * kb + 8 * q + i;
      nx[i] = *reinterpret_cast<const float4*>(src + 256 * (c < S ? c : S - 1));
    }
  };
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int turns = (A.B - wg + J.per - 1) / J.per * J.ngrp;
  if (wave < turns) request(wg + wave / J.ngrp * J.per, 0, 0, 0);

  for (int turn = wave; turn < turns; turn += kWyWaves) {  // no barrier follows
    const int i0 = turn / J.ngrp, k = turn - i0 * J.ngrp, b = wg + i0 * J.per;
    const int next = turn + kWyWaves < turns ? wg + (turn + kWyWaves) / J.ngrp * J.per : b;
    floatx4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[x][u] = (floatx4){0.f, 0.f, 0.f, 0.f};
    for (int kb = 0; kb < nkb; ++kb) {
      const int c0 = 32 * kb + 8 * q;
      const bf16x8 ah = *reinterpret_cast<const bf16x8*>(D.M[k][0] + r16 * kRowsMStr + c0);
      const bf16x8 al = *reinterpret_cast<const bf16x8*>(D.M[k][1] + r16 * kRowsMStr + c0);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        float4 z[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) z[i] = nx[i];
        for (int sg = 1; sg < J.SG; ++sg) {
          request(b, kb, x, sg);
#pragma unroll
          for (int i = 0; i < 8; ++i) z[i].x += nx[i].x, z[i].y += nx[i].y, z[i].z += nx[i].z, z[i].w += nx[i].w;
        }
        if (x < 3) request(b, kb, x + 1, 0);
        else if (kb + 1 < nkb) request(b, kb + 1, 0, 0);
        else request(next, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t fh[4][4], fl[4][4];
#pragma unroll
        for (int i2 = 0; i2 < 4; ++i2) {
          const float v0[4] = {z[2 * i2].x, z[2 * i2].y, z[2 * i2].z, z[2 * i2].w};
          const float v1[4] = {z[2 * i2 + 1].x, z[2 * i2 + 1].y, z[2 * i2 + 1].z, z[2 * i2 + 1].w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            // chunks past S (repeats of the last one) meet zero columns of M
            const uint32_t a = __float_as_uint(v0[u]), c = __float_as_uint(v1[u]);
            fh[u][i2] = perm_hi(c, a);
            fl[u][i2] = perm_hi(__float_as_uint(v1[u] - __uint_as_float(c & 0xFFFF0000u)),
                                __float_as_uint(v0[u] - __uint_as_float(a & 0xFFFF0000u)));
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bf16x8 h = __builtin_bit_cast(bf16x8, make_uint4(fh[u][0], fh[u][1], fh[u][2], fh[u][3]));
          const bf16x8 l = __builtin_bit_cast(bf16x8, make_uint4(fl[u][0], fl[u][1], fl[u][2], fl[u][3]));
          floatx4& t = acc[x][u];
          t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, ah, t, 0, 0, 0);
          t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, ah, t, 0, 0, 0);
          if constexpr (LO) t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, al, t, 0, 0, 0);
        }
      }
    }
    h256_rows<4>(acc);
    const float mul = J.scale * J.xmul[b];
    const int s = 16 * k + r16;
    uint16_t* stage = D.out[wave];
    const int col = 256 * (s < S ? s : S - 1);  // slices past S: computed, never stored
#pragma unroll
    for (int x = 0; x < 4; ++x) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t0 = 64 * x + 16 * j + 4 * q;
        const uint32_t neg = D.sign[(col + t0) >> 5] >> (t0 & 31);
        float4 su = make_float4(neg & 1 ? -1.0f : 1.0f, neg & 2 ? -1.0f : 1.0f, neg & 4 ? -1.0f : 1.0f,
                                neg & 8 ? -1.0f : 1.0f);
        if (!plain) su = *reinterpret_cast<const float4*>(J.su + col + t0);
        float4 bi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (J.bias) {
          const float* p = J.bias + col + t0;
          bi = J.bias_wide ? *reinterpret_cast<const float4*>(p) : make_float4(p[0], p[1], p[2], p[3]);
        }
        const float o[4] = {acc[x][0][j] * mul * su.x + bi.x, acc[x][1][j] * mul * su.y + bi.y,
                            acc[x][2][j] * mul * su.z + bi.z, acc[x][3][j] * mul * su.w + bi.w};
        if (A.y_dtype == QS_DTYPE_F32) {
          if (s >= S) continue;
          float* p = static_cast<float*>(J.y) + (int64_t)b * J.ldy + 256 * s + t0;
          if (J.wide) {
            *reinterpret_cast<float4*>(p) = make_float4(o[0], o[1], o[2], o[3]);
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) p[u] = o[u];
          }
        } else {
          uint2 w;
          if (A.y_dtype == QS_DTYPE_F16) {
            w.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){o[0], o[1]}, half2v));
            w.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){o[2], o[3]}, half2v));
          } else {
            w.x = f32x2_to_bf16x2(o[0], o[1]);
            w.y = f32x2_to_bf16x2(o[2], o[3]);
          }
          *reinterpret_cast<uint2*>(stage + r16 * kYStr + t0) = w;
        }
      }
    }
    if (A.y_dtype == QS_DTYPE_F32) continue;
    // 16-bit outputs through the wave's own LDS rows: a store then writes two
    // whole slices (512 bytes each) instead of 64 bytes of 16
    uint16_t* yo = static_cast<uint16_t*>(J.y) + (int64_t)b * J.ldy + 4096 * k;
    if (J.wide) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int sl = 2 * i + (lane >> 5), t0 = 8 * (lane & 31);
        const uint4 w = *reinterpret_cast<const uint4*>(stage + sl * kYStr + t0);
        if (16 * k + sl < S) *reinterpret_cast<uint4*>(yo + 256 * sl + t0) = w;
      }
    } else {
#pragma unroll 4
      for (int i = 0; i < 64; ++i) {
        const int sl = i >> 2, t0 = 64 * (i & 3) + lane;
        if (16 * k + sl < S) yo[256 * sl + t0] = stage[sl * kYStr + t0];
      }
    }
  }
}

// Work-groups per slice group: two per CU over all jobs and groups (what fits by
// registers), at most one per row tile, a multiple of 32 (a row tile's
// work-groups on one XCD).
int rows_per_group(int B, int total_groups, int ncu) {
  const int tiles = (B + kRowsWaves - 1) / kRowsWaves;
  int per = 2 * ncu / total_groups;
  if (per > tiles) per = tiles;
  per = (per + 31) / 32 * 32;
  return per;
}

}  // namespace

bool rows_transform_fits(int64_t len, int p) {
  return len % 256 == 0 && len / 256 <= kRowsMaxS && len / p >= 256 && p >= 1 && p <= QS_MAX_KRON;
}
bool rows_input_fits(const BatchedPass& P) {
  const size_t es = P.x_dtype == QS_DTYPE_F32 ? 4 : 2;
  if (P.x_dtype == QS_DTYPE_F32 && P.n > kRowsMaxFp32) return false;
  const int64_t rows = chunk_transform_fits(P.n, P.pn) ? kRowsInMin : kRowsInMinLong;
  return P.frag && P.B >= rows && rows_transform_fits(P.n, P.pn) && (reinterpret_cast<uintptr_t>(P.x) & 15) == 0 &&
         P.ldx * es % 16 == 0 && (reinterpret_cast<uintptr_t>(P.sv) & (P.sbits ? 3 : 15)) == 0;
}
bool rows_output_fits(const BatchedPass& P) {
  return P.B >= kRowsOutMin && !chunk_transform_fits(P.m, P.pm) && rows_transform_fits(P.m, P.pm) && (reinterpret_cast<uintptr_t>(P.y1p) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(P.su) & (P.sbits ? 3 : 15)) == 0;
}

int launch_wx(const BatchedPass* P, int count, hipStream_t stream) {
  QS_REQUIRE(count >= 1 && count <= QS_MAX_GROUP, "input transform: 1..%d linears", QS_MAX_GROUP);
  WxArgs A{};
  A.x = P[0].x;
  A.ldx = P[0].ldx;
  A.B = P[0].B;
  A.S = (int)(P[0].n / 256);
  A.pn = P[0].pn;
  A.lsh = log2_exact(P[0].n / P[0].pn / 256);
  A.njobs = count;
  A.Kn = P[0].Kn;
  A.scale = inv_sqrt_len(P[0].n / P[0].pn);
  const int ngrp = (A.S + 15) / 16, per = rows_per_group(A.B, count * ngrp, P[0].ncu);
  for (int g = 0; g < count; ++g) {
    QS_REQUIRE(rows_input_fits(P[g]) && P[g].x == P[0].x && P[g].n == P[0].n && P[g].B == A.B &&
                   P[g].sbits == P[0].sbits,
               "input transform: linears of one input");
    A.job[g] = WxJob{{g * ngrp * per, ngrp, per}, P[g].sv, P[g].x2h, P[g].sg, P[g].xmul};
  }
  const dim3 grid((unsigned)(count * ngrp * per)), block(kRowsThreads);
  const int xt = P[0].x_dtype == QS_DTYPE_BF16 ? 0 : P[0].x_dtype == QS_DTYPE_F16 ? 1 : 2;
  auto launch = [&](auto dt, auto bits, auto lo) {
    hipLaunchKernelGGL((wx_kernel<decltype(dt)::value, decltype(bits)::value, decltype(lo)::value>), grid, block, 0,
                       stream, A);
  };
  auto by_lo = [&](auto dt, auto bits) {
    if (A.pn > 1) launch(dt, bits, std::true_type());
    else launch(dt, bits, std::false_type());
  };
  auto by_bits = [&](auto dt) {
    if (P[0].sbits) by_lo(dt, std::true_type());
    else by_lo(dt, std::false_type());
  };
  if (xt == 0) by_bits(std::integral_constant<int, 0>());
  else if (xt == 1) by_bits(std::integral_constant<int, 1>());
  else by_bits(std::integral_constant<int, 2>());
  QS_LAUNCHED("wx_kernel");
  return QS_OK;
}

int launch_wy(const BatchedPass* P, int count, hipStream_t stream) {
  QS_REQUIRE(count >= 1 && count <= QS_MAX_GROUP, "output transform: 1..%d linears", QS_MAX_GROUP);
  WyArgs A{};
  A.B = P[0].B;
  A.y_dtype = P[0].y_dtype;
  A.njobs = count;
  int groups = 0;
  bool odd = false;  // a job without an odd factor has a zero second plane
  for (int g = 0; g < count; ++g) groups += (int)((P[g].m / 256 + 15) / 16), odd = odd || P[g].pm > 1;
  int wg = 0, most = 1;
  for (int g = 0; g < count; ++g) {
    const BatchedPass& Q = P[g];
    QS_REQUIRE(rows_output_fits(Q) && Q.B == A.B && Q.y_dtype == A.y_dtype && Q.sbits == P[0].sbits,
               "output transform: m %lld (p %d) or mixed rows / dtype / sign format", (long long)Q.m, Q.pm);
    const size_t es = Q.y_dtype == QS_DTYPE_F32 ? 4 : 2;
    const int S = (int)(Q.m / 256), ngrp = (S + 15) / 16;
    // one work-group per CU (by its LDS), dealt by the linears' sizes
    int per = P[0].ncu * ngrp / groups;
    per = per < 1 ? 1 : per > A.B ? A.B : per;
    A.job[g] = WyJob{wg,
                     per,
                     Q.y1p,
                     Q.SG,
                     (int)Q.m,
                     S,
                     log2_exact(Q.m / Q.pm / 256),
                     Q.pm,
                     ngrp,
                     Q.Km,
                     inv_sqrt_len(Q.m / Q.pm) * Q.layer_scale,
                     Q.xmul,
                     Q.su,
                     Q.bias,
                     Q.y,
                     Q.ldy,
                     (reinterpret_cast<uintptr_t>(Q.y) & 15) == 0 && Q.ldy * es % 16 == 0,
                     (reinterpret_cast<uintptr_t>(Q.bias) & 15) == 0};
    wg += per;
    most = ngrp > most ? ngrp : most;
  }
  const size_t lds = wy_lds(most);
  auto launch = [&](auto kernel) {
    // the most that any call takes: a limit of its own could be another thread's next launch's
    QS_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kWyMaxLds));
    hipLaunchKernelGGL(kernel, dim3((unsigned)wg), dim3(kWyThreads), lds, stream, A);
    return (int)QS_OK;
  };
  const int rc = P[0].sbits ? (odd ? launch(wy_kernel<true, true>) : launch(wy_kernel<true, false>))
                            : (odd ? launch(wy_kernel<false, true>) : launch(wy_kernel<false, false>));
  if (rc) return rc;
  QS_LAUNCHED("wy_kernel");
  return QS_OK;
}

}  // namespace qs
