// E8P / E8 1-bit / residual-VQ encode and decode on gfx950, plus the fused
// BlockLDLQ rounding step and the code repacker for the forward kernels.
//
// Bit-exactness: the encoder returns the candidate that the reference's fp32
// CPU arithmetic (quipsharp/codebooks/e8p.py:104-162) puts first.  Every
// product, difference and square is there a separately rounded IEEE operation
// (this file is compiled with -ffp-contract=off), the eight squares are summed
// left to right, flips are strict "< 0", the parity repair goes to the first
// coordinate of least |product|, and the winner is the lexicographic minimum
// of (distance, shift bit, table row).  A vector whose winner the search of
// qs_e8_search.h can tell from the runner-up by more than all roundings is
// decided there; the others (of Gaussian vectors four in ten thousand; ties and
// non-finite values among them) have every candidate evaluated in that
// arithmetic by the whole wave.  The winner's signs, code and values are
// formed in the reference's arithmetic either way.
#include "qs_common.h"
#include "qs_e8_search.h"

namespace qs {
namespace {

__constant__ Table8 kE8P = make_e8p_table();
__constant__ Table8 kE81 = make_e81_table();

__constant__ E8Luts kLuts = make_e8_luts();

constexpr int kEncThreads = 256;  // one vector per lane

struct StageCfg {
  int n;
  int kind[QS_MAX_STAGES];
  float scale[QS_MAX_STAGES];
};

struct EncodeArgs {
  // target = base (+ delta (@ dinv))
  const float* base;
  int64_t ldbase;
  const float* delta;  // [nvec][8] or NULL
  const float* dinv;   // [8][8] or NULL
  // outputs
  float* vals;
  int64_t ldvals;
  const float* w;      // residual output: resid = w - vals
  int64_t ldw;
  float* resid;
  int64_t ldresid;
  void* codes;
  int code_bytes;
  int64_t code_stage_stride;
  int64_t code_stride;
  int64_t nvec;
  float in_div, out_mul;
  StageCfg st;
};

__device__ __forceinline__ void store_code(void* codes, int code_bytes, int64_t off, uint32_t c) {
  if (code_bytes == 2) static_cast<uint16_t*>(codes)[off] = (uint16_t)c;
  else if (code_bytes == 4) static_cast<int32_t*>(codes)[off] = (int32_t)c;
  else static_cast<int64_t*>(codes)[off] = (int64_t)c;
}

__device__ __forceinline__ uint32_t load_code(const void* codes, int code_bytes, int64_t off) {
  if (code_bytes == 2) return static_cast<const uint16_t*>(codes)[off];
  if (code_bytes == 4) return (uint32_t) static_cast<const int32_t*>(codes)[off];
  return (uint32_t) static_cast<const int64_t*>(codes)[off];
}

// Eight consecutive floats: two 16-byte accesses where the address allows it.
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  if ((reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = p[i];
  }
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
  if ((reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = v[i];
  }
}

// Distance of the shifted input (|xs| = a, parity bit `odd` for this row) to
// the best even-parity signing of table row t (absolute values T).
__device__ __forceinline__ float e8p_row_d2(const float a[8], const float T[8], bool odd) {
  float sq[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float d = a[i] - T[i];
    sq[i] = d * d;
  }
  if (odd) {
    float best = a[0] * T[0];
    int j = 0;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      float p = a[i] * T[i];
      if (p < best) { best = p; j = i; }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i == j) {
        float d = a[i] + T[i];
        sq[i] = d * d;
      }
    }
  }
  float d2 = sq[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) d2 = d2 + sq[i];
  return d2;
}

// res += dl . dinv (dinv 8 x 8, row-major), or res += dl without dinv.
__device__ __forceinline__ void add_delta(float (&res)[8], const float (&dl)[8], const float* dinv) {
  if (dinv) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float acc = dl[0] * dinv[i];
#pragma unroll
      for (int j = 1; j < 8; ++j) acc = __builtin_fmaf(dl[j], dinv[j * 8 + i], acc);
      res[i] = res[i] + acc;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) res[i] = res[i] + dl[i];
  }
}

// The target of vector vv: base (+ delta, or + delta . dinv), divided by
// in_div.
__device__ __forceinline__ void encode_target(const EncodeArgs& A, int64_t vv, float (&res)[8]) {
  load8(A.base + vv * A.ldbase, res);
  if (A.delta) {
    float dl[8];
    load8(A.delta + vv * 8, dl);
    add_delta(res, dl, A.dinv);
  }
  if (A.in_div != 1.0f) {
#pragma unroll
    for (int i = 0; i < 8; ++i) res[i] = res[i] / A.in_div;
  }
}

__device__ __forceinline__ void load_luts(E8Luts& L, int tid, int threads) {
  for (int i = tid; i < (int)(sizeof(E8Luts) / 4); i += threads)
    reinterpret_cast<uint32_t*>(&L)[i] = reinterpret_cast<const uint32_t*>(&kLuts)[i];
}

__device__ __forceinline__ void e8p_entries(uint32_t pat, float (&T)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) T[i] = (float)((pat >> (2 * i)) & 3u) + 0.5f;
}
__device__ __forceinline__ void e81_value(const E8Luts& L, uint32_t row, float (&q)[8]) {
  const uint32_t w = L.one[row];
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = (float)(int)((w >> (4 * i)) & 15u) * 0.5f - 4.0f;  // exact
}

// Least value over the wave, in every lane.
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = umin2(v, (uint32_t)__shfl_xor((int)v, off));
  return v;
}

// Every candidate of the table for x (the same in every lane), in the
// reference's arithmetic: lane l evaluates rows l + 64 k (k < 4), at both
// shifts for E8P.  Returns the row | shift bit << 8 of least (distance, shift
// bit, row); a distance's bits order as its value, NaN last.  U: rows of a lane
// in flight at once (all four where a vector's latency counts and registers
// do not).
template <int U>
__device__ __forceinline__ uint32_t wave_all_candidates(int kind, const float (&x)[8], int lane, const E8Luts& L) {
  uint32_t best = ~0u, at = 0;
  if (kind == QS_STAGE_E8P) {
#pragma unroll 1
    for (int sb = 0; sb < 2; ++sb) {
      float a[8];
      uint32_t sx = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float xs = sb == 0 ? x[i] + 0.25f : x[i] - 0.25f;
        a[i] = fabsf(xs);
        sx ^= __float_as_uint(xs) >> 31;
      }
      const bool p_pos = sx & 1, p_neg = p_pos ^ (a[7] != 0.0f);
#pragma unroll U
      for (int k = 0; k < 4; ++k) {
        const uint32_t pat = L.pat[lane + 64 * k];
        float T[8];
        e8p_entries(pat, T);
        const uint32_t d2 = __float_as_uint(e8p_row_d2(a, T, __popc(pat & 0x5555u) & 1 ? p_neg : p_pos));
        if (d2 < best) best = d2, at = (uint32_t)sb << 8 | (uint32_t)(lane + 64 * k);
      }
    }
  } else {
#pragma unroll U
    for (int k = 0; k < 4; ++k) {
      float q[8], d2 = 0.0f;
      e81_value(L, lane + 64 * k, q);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = x[i] - q[i];
        d2 = i == 0 ? d * d : d2 + d * d;
      }
      const uint32_t u = __float_as_uint(d2);
      if (u < best) best = u, at = (uint32_t)(lane + 64 * k);
    }
  }
  return wave_min(best == wave_min(best) ? at : ~0u);
}

// The value of lane src (wave-uniform) in every lane.
__device__ __forceinline__ float lane_value(float v, int src) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), src));
}

// The lanes of `todo` whose search was not certain: each one's candidates
// evaluated by the whole wave.  GROUP lanes hold one vector (all of them take
// its answer; `todo` has the first lane of each).  sel: row | pattern << 8, sb:
// the shift bit (E8P); sel: the row (E8 one-bit).
template <int GROUP>
__device__ __forceinline__ void settle(unsigned long long todo, int kind, const float (&x)[8], int lane,
                                       const E8Luts& L, uint32_t& sel, int& sb) {
  while (todo) {
    const int src = __ffsll((unsigned long long)todo) - 1;
    todo &= todo - 1;
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = lane_value(x[i], src);
    const uint32_t w = wave_all_candidates<GROUP == 1 ? 1 : 4>(kind, y, lane, L), r = w & 0xFF;
    if (lane / GROUP == src / GROUP) {
      sel = kind == QS_STAGE_E8P ? r | (L.pat[r] << 8) : r;
      sb = (int)(w >> 8);
    }
  }
}

// Packs the code of the E8P row `sel` (row | pattern << 8, E8Luts) at shift bit
// sb for input x (e8p.py:116-123, 165-171) and writes the decoded codeword to q.
__device__ __forceinline__ uint32_t e8p_finish(const float (&x)[8], int sb, uint32_t sel, float (&q)[8]) {
  const uint32_t pat = sel >> 8;
  float T[8], prod[8];
  uint32_t flips = 0;
  e8p_entries(pat, T);
  if (__popc(pat & 0x5555u) & 1) T[7] = -T[7];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float xs = sb == 0 ? x[i] + 0.25f : x[i] - 0.25f;
    prod[i] = xs * T[i];
    flips |= (prod[i] < 0.0f ? 1u : 0u) << i;
  }
  float best = fabsf(prod[0]);
  uint32_t j = 1;
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    const float p = fabsf(prod[i]);
    if (p < best) { best = p; j = 1u << i; }
  }
  if (__popc(flips) & 1) flips ^= j;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = (flips >> i) & 1 ? -T[i] : T[i];
    q[i] = sb == 0 ? v - 0.25f : v + 0.25f;
  }
  const uint32_t sign7 = __brev(flips) >> 25;  // bit 6 - i: coordinate i
  return ((sel & 0xFF) << 8) | (sign7 << 1) | (uint32_t)sb;
}

// One vector per lane.  A wave runs ~800 vector operations for its 64 vectors
// (the sorted search of qs_e8_search.h at both shifts, then the winner's signs
// and values), where evaluating the 512 candidates took ~13,000.  2^20 vectors,
// 2 bits: 914 -> 40 us (the 75 MB in and out take 15 at the copy rate).  A call
// of nothing but ties, such as 2^17 zero vectors, is slower than with every
// candidate in one lane: 92 -> 217 us.
__global__ __launch_bounds__(kEncThreads) void rvq_encode_kernel(EncodeArgs A) {
  __shared__ E8Luts L;
  load_luts(L, threadIdx.x, kEncThreads);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t v = (int64_t)blockIdx.x * kEncThreads + threadIdx.x;
  const bool valid = v < A.nvec;
  float res[8], tot[8];
  encode_target(A, valid ? v : 0, res);
#pragma unroll
  for (int i = 0; i < 8; ++i) tot[i] = 0.0f;
  for (int s = 0; s < A.st.n; ++s) {
    const float sc = A.st.scale[s];
    const int kind = A.st.kind[s];
    float x[8], q[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = sc == 1.0f ? res[i] : res[i] / sc;
    uint32_t code;
    bool certain;
    if (kind == QS_STAGE_E8P) {
      int sb;
      const E8Best b = e8p_search2(x, sb, certain);
      uint32_t sel = L.sel[b.sel];
      settle<1>(__ballot(valid && !certain), kind, x, lane, L, sel, sb);
      code = e8p_finish(x, sb, sel, q);
    } else {
      const E8Best b = e81_search(x, certain);
      int sb = 0;
      code = b.sel < 256 ? b.sel : L.pair[b.sel - 256];
      settle<1>(__ballot(valid && !certain), kind, x, lane, L, code, sb);
      e81_value(L, code, q);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float qs = q[i] * sc;
      tot[i] = tot[i] + qs;
      res[i] = res[i] - qs;
    }
    if (valid && A.codes) store_code(A.codes, A.code_bytes, s * A.code_stage_stride + v * A.code_stride, code);
  }
  if (A.out_mul != 1.0f) {
#pragma unroll
    for (int i = 0; i < 8; ++i) tot[i] = tot[i] * A.out_mul;
  }
  if (!valid) return;
  if (A.vals) store8(A.vals + v * A.ldvals, tot);
  if (A.resid) {
    float wv[8];
    load8(A.w + v * A.ldw, wv);
#pragma unroll
    for (int i = 0; i < 8; ++i) wv[i] = wv[i] - tot[i];
    store8(A.resid + v * A.ldresid, wv);
  }
}

// ---------------------------------------------------------------------------
// A vector in 16 lanes, for the serial chain of BlockLDLQ: the time of one
// rounding counts, not how many fit the GPU.  Lanes 0..7 and 8..15 hold its
// coordinates and search the two shifts of an E8P stage at the same time, the
// 29 rows split over the eight lanes of a shift.
// ---------------------------------------------------------------------------
// A lane's value through a data-parallel-primitive pattern (rows of 16 lanes).
template <int CTRL, class V>
__device__ __forceinline__ V row_dpp(V v) {
  const int i = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xF, 0xF, true));
}
constexpr int kRowRor8 = 0x128, kRowRor4 = 0x124, kHalfMirror = 0x141, kQuadXor2 = 0x4E, kQuadXor1 = 0xB1;
constexpr int kRowLane = 0x150;
// Lanes 0..7 of each 16, in all of them.
__device__ __forceinline__ void row_lanes8(float v, float (&o)[8]) {
  o[0] = row_dpp<kRowLane + 0>(v), o[1] = row_dpp<kRowLane + 1>(v), o[2] = row_dpp<kRowLane + 2>(v);
  o[3] = row_dpp<kRowLane + 3>(v), o[4] = row_dpp<kRowLane + 4>(v), o[5] = row_dpp<kRowLane + 5>(v);
  o[6] = row_dpp<kRowLane + 6>(v), o[7] = row_dpp<kRowLane + 7>(v);
}
__device__ __forceinline__ float pick8(const float (&v)[8], int j) {
  const float v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3], v4 = v[4], v5 = v[5], v6 = v[6], v7 = v[7];
  const bool b0 = j & 1, b1 = j & 2, b2 = j & 4;
  const float c0 = b0 ? v1 : v0, c1 = b0 ? v3 : v2, c2 = b0 ? v5 : v4, c3 = b0 ? v7 : v6;
  const float d0 = b1 ? c1 : c0, d1 = b1 ? c3 : c2;
  return b2 ? d1 : d0;
}

// Lane t of eight: rows 4 t .. 4 t + 3 of the 29.
struct RowFives {
  int at[12];  // lanes (x 4) of the rows' coordinates
  int first;
  float aj;    // this lane's own magnitude
  __device__ __forceinline__ void lanes(const E8Luts& L, int lane) {
    first = 4 * (lane & 7);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t w = L.low[first + u];
#pragma unroll
      for (int n = 0; n < 3; ++n) at[3 * u + n] = 4 * ((lane & 56) | (int)((w >> (8 * n)) & 7));
    }
  }
  __device__ __forceinline__ void operator()(const float (&)[8], float floor3, float cap, float odd2, uint32_t& q1,
                                             uint32_t& q2) const {
    const int own = __builtin_bit_cast(int, aj);
    float c[12];
#pragma unroll
    for (int n = 0; n < 12; ++n) c[n] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(at[n], own));
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t v = five_value(c[3 * u], c[3 * u + 1], c[3 * u + 2], floor3, cap, odd2, (uint32_t)(first + u));
      take_five(q1, q2, first + u < 29 ? v : ~0u);
    }
    least2<kQuadXor1>(q1, q2);
    least2<kQuadXor2>(q1, q2);
    least2<kHalfMirror>(q1, q2);
  }
  template <int CTRL>
  __device__ __forceinline__ static void least2(uint32_t& q1, uint32_t& q2) {
    const uint32_t p1 = row_dpp<CTRL>(q1), p2 = row_dpp<CTRL>(q2);
    q2 = umin2(umin2(q2, p2), umax2(q1, p1));
    q1 = umin2(q1, p1);
  }
};

// e8p_finish with the coordinates in the row's lanes: xj is this lane's.
__device__ __forceinline__ uint32_t row_finish(float xj, int sb, uint32_t sel, int lane, float& qj) {
  const int j = lane & 7, row0 = lane & 48;
  const uint32_t pat = sel >> 8;
  float T = (float)((pat >> (2 * j)) & 3u) + 0.5f;
  if (j == 7 && (__popc(pat & 0x5555u) & 1)) T = -T;
  const float prod = (sb == 0 ? xj + 0.25f : xj - 0.25f) * T;
  const float p = fabsf(prod);
  auto bits = [&](bool b) { return (uint32_t)(__ballot(b) >> row0) & 0xFFu; };  // of coordinates 0..7
  uint32_t flips = bits(prod < 0.0f);
  float m = min2(p, row_dpp<kQuadXor1>(p));
  m = min2(m, row_dpp<kQuadXor2>(m));
  m = min2(m, row_dpp<kHalfMirror>(m));
  const uint32_t least = bits(p == m), nan = bits(p != p);
  // the first least product; coordinate 0 where its product is NaN
  const uint32_t repair = (nan & 1) || least == 0 ? 1u : least & (0u - least);
  if (__popc(flips) & 1) flips ^= repair;
  const float v = (flips >> j) & 1 ? -T : T;
  qj = sb == 0 ? v - 0.25f : v + 0.25f;
  return ((sel & 0xFF) << 8) | ((__brev(flips) >> 25) << 1) | (uint32_t)sb;
}

// A stage's kind and scale by selection: indexing the argument block loads
// from memory in the loop.
__device__ __forceinline__ int st_kind(const StageCfg& st, int s) {
  const int a = st.kind[0], b = st.kind[1], c = st.kind[2], d = st.kind[3];
  return s == 0 ? a : s == 1 ? b : s == 2 ? c : d;
}
__device__ __forceinline__ float st_scale(const StageCfg& st, int s) {
  const float a = st.scale[0], b = st.scale[1], c = st.scale[2], d = st.scale[3];
  return s == 0 ? a : s == 1 ? b : s == 2 ? c : d;
}

// One stage for coordinate j = lane & 7 of the residual `res` and the sum
// `tot`; returns the code.
__device__ __forceinline__ uint32_t row_stage(int kind, float sc, float& res, float& tot, bool valid, int lane,
                                              const E8Luts& L, RowFives& fives) {
  const float xj = sc == 1.0f ? res : res / sc;
  float x[8], qj;
  row_lanes8(xj, x);
  const unsigned long long rows = 0x0001000100010001ull;
  uint32_t code;
  int sb = 0;
  if (kind == QS_STAGE_E8P) {
    const bool second = lane & 8;
    const float shift = second ? -0.25f : 0.25f;
    fives.aj = fabsf(xj + shift);
    const E8Best mine = e8p_search(x, shift, fives);
    const float ob = row_dpp<kRowRor8>(mine.best), os = row_dpp<kRowRor8>(mine.second);
    const float ok = row_dpp<kRowRor8>(mine.slack);
    const uint32_t osel = row_dpp<kRowRor8>(mine.sel);
    const float b0 = second ? ob : mine.best, b1 = second ? mine.best : ob;
    const bool first = b0 <= b1;
    const bool own = first != second;
    const float runner = min2(own ? mine.second : os, first ? b1 : b0);
    const bool certain = runner - (first ? b0 : b1) > mine.slack + ok;
    uint32_t sel = L.sel[own ? mine.sel : osel];
    sb = first ? 0 : 1;
    settle<16>(__ballot(!certain && valid) & rows, kind, x, lane, L, sel, sb);
    code = row_finish(xj, sb, sel, lane, qj);
  } else {
    bool certain;
    const E8Best b = e81_search(x, certain);
    code = b.sel < 256 ? b.sel : L.pair[b.sel - 256];
    settle<16>(__ballot(!certain && valid) & rows, kind, x, lane, L, code, sb);
    qj = (float)(int)((L.one[code] >> (4 * (lane & 7))) & 15u) * 0.5f - 4.0f;
  }
  const float qs = qj * sc;
  tot = tot + qs;
  res = res - qs;
  return code;
}

// rvq_encode_kernel for the rounding step of one block of BlockLDLQ (and other
// short calls): 16 lanes to a vector.  4096 vectors 7.2 us, one vector per lane
// 11.5, a wave per vector with the 512 candidates over its lanes 10.1.
// One round of its 64-thread work-groups on the GPU; more vectors fill it at one
// per lane, which takes a tenth of the operations.
constexpr int64_t kRowEncodeMax = 16384;
__global__ __launch_bounds__(64) void rvq_encode_row_kernel(EncodeArgs A) {
  __shared__ E8Luts L;
  const int lane = threadIdx.x, j = lane & 7;
  const int64_t row = (int64_t)blockIdx.x * 4 + (lane >> 4);
  const bool valid = row < A.nvec;
  const int64_t v = valid ? row : A.nvec - 1;
  float res = A.base[v * A.ldbase + j], tot = 0.0f;
  if (A.delta) {
    float dl[8];
    row_lanes8(A.delta[v * 8 + j], dl);
    if (A.dinv) {
      float acc = dl[0] * A.dinv[j];
#pragma unroll
      for (int i = 1; i < 8; ++i) acc = __builtin_fmaf(dl[i], A.dinv[8 * i + j], acc);
      res = res + acc;
    } else {
      res = res + pick8(dl, j);
    }
  }
  if (A.in_div != 1.0f) res = res / A.in_div;
  const float wv = A.resid ? A.w[v * A.ldw + j] : 0.0f;
  load_luts(L, lane, 64);
  __syncthreads();
  RowFives fives;
  fives.lanes(L, lane);
  for (int s = 0; s < A.st.n; ++s) {
    const uint32_t code = row_stage(st_kind(A.st, s), st_scale(A.st, s), res, tot, valid, lane, L, fives);
    if (valid && (lane & 15) == 0 && A.codes)
      store_code(A.codes, A.code_bytes, s * A.code_stage_stride + v * A.code_stride, code);
  }
  if (A.out_mul != 1.0f) tot = tot * A.out_mul;
  if (!valid || (lane & 8)) return;
  if (A.vals) A.vals[v * A.ldvals + j] = tot;
  if (A.resid) A.resid[v * A.ldresid + j] = wv - tot;
}

// ---------------------------------------------------------------------------
// A chunk of up to 16 blocks c0 .. c0 + nb - 1 of the BlockLDLQ refinement
// pass, in descending order, in one launch, 16 lanes to a row: for block k
//   delta = p[row][8 (k - c0) ..] + E[row][chunk columns] . H[chunk rows][block k]
//   target = wq[row][block k] + delta . dinv[k]
// then the stages, wq and E of block k rewritten.  Lane l keeps the chunk's
// columns l + 16 i of E in registers.
//
// A row's blocks are one serial chain (the rounding of a block feeds the next),
// so a launch takes 16 times a block's latency whatever the rows, and a 4096-row
// layer leaves each SIMD one wave of four rows.  So the loop touches no global
// memory: H's chunk (64 KiB, in the order in which a block's lanes read it, 16
// bytes apart), dinv and the rows' p, w and wq are read into LDS first, and wq,
// E and the codes leave from there at the end (a store in the loop made the
// next block's loads wait for it).  4096 rows, 2 bits: a wave per row with the
// 512 candidates spread over its lanes 207 us per launch; this search with
// loads and stores in the loop 43 us; as it is 37 us (9 of them to fill LDS and
// write back, then 1.6 a block, ~780 instructions of one wave).
//
// The sums are those of a wave per row with columns c and c + 64 in lane c: the
// pair first, then the halves 32, 16, 8, 4, 2 and 1 apart.
// ---------------------------------------------------------------------------
constexpr int kChunkBlocks = 16;
constexpr int kChunkCols = 8 * kChunkBlocks;
constexpr int kChunkLd = kChunkCols + 8;  // a row's stride in LDS: four rows' blocks in distinct banks
struct ChunkArgs {
  const float* w;
  int64_t ldw;
  float* wq;
  int64_t ldwq;
  float* e;
  int64_t lde;
  const float* p;  // [m][8 nb]: the product of E with H's block columns outside the chunk
  int64_t ldp;
  const float* h;  // H's rows of the chunk (row c0 8 of H), ldh per row
  int64_t ldh;
  const float* dinv;  // [T][8][8]
  int c0, nb;
  int64_t m;
  void* codes;
  int code_bytes;
  int64_t code_stage_stride, code_stride;
  StageCfg st;
};
struct ChunkLds {
  float4 h[kChunkBlocks * 8 * 2 * 16];  // [block][i][half][l]: row l + 16 i, columns 4 half .. + 3 of the block
  E8Luts L;
  float dinv[kChunkBlocks * 64];
};
constexpr size_t chunk_lds(int rows) { return sizeof(ChunkLds) + (size_t)rows * 3 * kChunkLd * sizeof(float); }
constexpr int kChunkMaxRows = 32;  // of a work-group
constexpr int kChunkMaxLds = (int)chunk_lds(kChunkMaxRows);
static_assert(kChunkMaxLds <= 160 * 1024, "LDS budget");

__global__ __launch_bounds__(16 * kChunkMaxRows) void ldlq_chunk_kernel(ChunkArgs A) {
  extern __shared__ char sm[];
  ChunkLds& S = *reinterpret_cast<ChunkLds*>(sm);
  float* rows = reinterpret_cast<float*>(sm + sizeof(ChunkLds));  // per row: p (then codes), w (then E), wq
  const int tid = threadIdx.x, threads = blockDim.x;
  const int lane = tid & 63, l = tid & 15, j = tid & 7;
  const int R = threads >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  const int here = A.m - row0 < R ? (int)(A.m - row0) : R;  // rows of this work-group
  const bool valid = (tid >> 4) < here;
  const int nb = A.nb, wc = 8 * nb, col0 = 8 * A.c0;

  float ec[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = l + 16 * i;
    ec[i] = valid && c < wc ? A.e[(row0 + (tid >> 4)) * A.lde + col0 + c] : 0.0f;
  }
  const bool wide = (reinterpret_cast<uintptr_t>(A.h + col0) & 15) == 0 && (A.ldh & 3) == 0;
  auto load4 = [&](const float* src) {
    return wide ? *reinterpret_cast<const float4*>(src) : make_float4(src[0], src[1], src[2], src[3]);
  };
#pragma unroll 8
  for (int t = tid; t < kChunkCols * kChunkCols / 4; t += threads) {
    const int r = t >> 5, c4 = t & 31;
    float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // outside the chunk
    if (r < wc && c4 < 2 * nb) f = load4(A.h + (int64_t)r * A.ldh + col0 + 4 * c4);
    S.h[(((c4 >> 1) * 8 + (r >> 4)) * 2 + (c4 & 1)) * 16 + (r & 15)] = f;
  }
  load_luts(S.L, tid, threads);
  for (int t = tid; t < 64 * nb; t += threads) S.dinv[t] = A.dinv[64 * (int64_t)A.c0 + t];
#pragma unroll 4
  for (int t = tid; t < R * kChunkCols; t += threads) {
    const int r = t >> 7, c = t & 127;
    float* o = rows + r * 3 * kChunkLd + c;
    const bool in = r < here && c < wc;
    o[0] = in ? A.p[(row0 + r) * A.ldp + c] : 0.0f;
    o[kChunkLd] = in ? A.w[(row0 + r) * A.ldw + col0 + c] : 0.0f;
    o[2 * kChunkLd] = in ? A.wq[(row0 + r) * A.ldwq + col0 + c] : 0.0f;
  }
  __syncthreads();
  RowFives fives;
  fives.lanes(S.L, lane);

  float* mine = rows + (tid >> 4) * 3 * kChunkLd;
  // what a block reads from LDS, requested before the rounding of the block
  // before it (left to the compiler, the 16 reads of H waited one by one)
  float4 hv[16];
  float n_p, n_w, n_base, n_dinv[8];
  auto fetch = [&](int kk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) hv[i] = S.h[(kk * 16 + i) * 16 + l];
    n_p = mine[8 * kk + j];
    n_w = mine[kChunkLd + 8 * kk + j];
    n_base = mine[2 * kChunkLd + 8 * kk + j];
#pragma unroll
    for (int t = 0; t < 8; ++t) n_dinv[t] = S.dinv[64 * kk + 8 * t + j];
  };
  fetch(nb - 1);
  for (int kk = nb - 1; kk >= 0; --kk) {
    float s[4][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float h[8] = {hv[2 * i].x,     hv[2 * i].y,     hv[2 * i].z,     hv[2 * i].w,
                          hv[2 * i + 1].x, hv[2 * i + 1].y, hv[2 * i + 1].z, hv[2 * i + 1].w};
#pragma unroll
      for (int t = 0; t < 8; ++t) s[i & 3][t] = __builtin_fmaf(ec[i], h[t], i < 4 ? 0.0f : s[i & 3][t]);
    }
    const int at = 8 * kk + j;
    float f[8], pl[8], add = 0.0f;
    row_lanes8(n_p, pl);
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = (s[0][t] + s[2][t]) + (s[1][t] + s[3][t]);
    // eight sums side by side, a step of all of them before the next
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = f[t] + row_dpp<kRowRor8>(f[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = f[t] + row_dpp<kRowRor4>(f[t]);  // repeats every 8 lanes by now: lane ^ 4
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = f[t] + row_dpp<kQuadXor2>(f[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = f[t] + row_dpp<kQuadXor1>(f[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const float dl = pl[t] + f[t];
      add = t == 0 ? dl * n_dinv[0] : __builtin_fmaf(dl, n_dinv[t], add);
    }
    const float wv = n_w, base = n_base;
    __builtin_amdgcn_sched_barrier(0);
    if (kk > 0) fetch(kk - 1);
    __builtin_amdgcn_sched_barrier(0);
    float res = base + add, tot = 0.0f;
    for (int st = 0; st < A.st.n; ++st) {
      const uint32_t code = row_stage(st_kind(A.st, st), st_scale(A.st, st), res, tot, valid, lane, S.L, fives);
      if (l == 0) mine[8 * kk + st] = __uint_as_float(code);
    }
    const float r = wv - tot;
    if (l < 8) {
      mine[kChunkLd + at] = r;
      mine[2 * kChunkLd + at] = tot;
    }
    // column 8 kk + j into the lane and register that keep it
#pragma unroll
    for (int i = 0; i < 8; ++i) ec[i] = (kk >> 1) == i && (l >> 3) == (kk & 1) ? r : ec[i];
  }
  __syncthreads();
  for (int t = tid; t < here * kChunkCols; t += threads) {
    const int r = t >> 7, c = t & 127;
    if (c >= wc) continue;
    const float* o = rows + r * 3 * kChunkLd + c;
    A.e[(row0 + r) * A.lde + col0 + c] = o[kChunkLd];
    A.wq[(row0 + r) * A.ldwq + col0 + c] = o[2 * kChunkLd];
  }
  if (A.codes)
    for (int t = tid; t < here * nb * A.st.n; t += threads) {
      const int s = t / (here * nb), u = t - s * (here * nb), r = u / nb, k = u - r * nb;
      store_code(A.codes, A.code_bytes, s * A.code_stage_stride + (row0 + r) * A.code_stride + A.c0 + k,
                 __float_as_uint(rows[r * 3 * kChunkLd + 8 * k + s]));
    }
}

int launch_encode(EncodeArgs& A, hipStream_t stream) {
  if (A.nvec == 0) return QS_OK;
  if (A.nvec <= kRowEncodeMax) {
    hipLaunchKernelGGL(rvq_encode_row_kernel, dim3((unsigned)((A.nvec + 3) / 4)), dim3(64), 0, stream, A);
    QS_LAUNCHED("rvq_encode_row_kernel");
    return QS_OK;
  }
  const int64_t blocks = (A.nvec + kEncThreads - 1) / kEncThreads;
  QS_REQUIRE(blocks < (1ll << 31), "too many vectors: %lld", (long long)A.nvec);
  hipLaunchKernelGGL(rvq_encode_kernel, dim3((unsigned)blocks), dim3(kEncThreads), 0, stream, A);
  QS_LAUNCHED("rvq_encode_kernel");
  return QS_OK;
}

int fill_stages(StageCfg& st, int nstages, const int* kinds, const float* scales) {
  QS_REQUIRE(nstages >= 1 && nstages <= QS_MAX_STAGES, "nstages must be in [1, %d], got %d",
             QS_MAX_STAGES, nstages);
  QS_REQUIRE(kinds && scales, "kinds and scales must be host arrays");
  st.n = nstages;
  for (int s = 0; s < nstages; ++s) {
    QS_REQUIRE(kinds[s] == QS_STAGE_E8P || kinds[s] == QS_STAGE_E8_1BIT, "bad stage kind %d", kinds[s]);
    QS_REQUIRE(scales[s] != 0.0f, "stage scale must be non-zero");
    st.kind[s] = kinds[s];
    st.scale[s] = scales[s];
  }
  return QS_OK;
}

// ---------------------------------------------------------------------------
// decode
// ---------------------------------------------------------------------------
struct DecodeArgs {
  const void* codes;
  int code_bytes;
  int64_t stage_stride;
  int64_t nvec;
  StageCfg st;
  float out_scale;
  float* out;
};

__device__ __forceinline__ void e8p_decode(uint32_t c, float v[8]) {
  const int a = (c >> 8) & 0xFF;
  uint32_t par = 0;
  const float sh = (c & 1) ? 0.25f : -0.25f;
#pragma unroll
  for (int i = 0; i < 7; ++i) {
    uint32_t f = (c >> (7 - i)) & 1;
    par ^= f;
    float t = kE8P.v[a][i];
    v[i] = (f ? -t : t) + sh;
  }
  float t7 = kE8P.v[a][7];
  v[7] = (par ? -t7 : t7) + sh;
}

__global__ __launch_bounds__(256) void rvq_decode_kernel(DecodeArgs A) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= A.nvec) return;
  float tot[8];
  for (int s = 0; s < A.st.n; ++s) {
    uint32_t c = load_code(A.codes, A.code_bytes, s * A.stage_stride + k);
    float v[8];
    if (A.st.kind[s] == QS_STAGE_E8P) {
      e8p_decode(c & 0xFFFF, v);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = kE81.v[c & 0xFF][i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float vs = v[i] * A.st.scale[s];
      tot[i] = s == 0 ? vs : tot[i] + vs;
    }
  }
  float4* o = reinterpret_cast<float4*>(A.out + k * 8);
  o[0] = make_float4(tot[0] * A.out_scale, tot[1] * A.out_scale, tot[2] * A.out_scale, tot[3] * A.out_scale);
  o[1] = make_float4(tot[4] * A.out_scale, tot[5] * A.out_scale, tot[6] * A.out_scale, tot[7] * A.out_scale);
}

// ---------------------------------------------------------------------------
// repack for the forward kernels
// ---------------------------------------------------------------------------
// Kernel form of an E8P code: [f1 f2 f3 q | abs_idx | f4 f5 f6 | shift], where
// f_i is the flip of coordinate i and q = f0^f1^f2^f3.  Then (e >> 4) indexes
// the table of signed coordinates 0..3 and ((e >> 1) & 0xFFF) the table of
// signed coordinates 4..7 (coordinate 7's flip is q^f4^f5^f6, the parity of
// the seven stored flips).
__device__ __forceinline__ uint32_t kernel_form(uint32_t c) {
  const uint32_t a = (c >> 8) & 0xFF;
  const uint32_t f0 = (c >> 7) & 1, f1 = (c >> 6) & 1, f2 = (c >> 5) & 1, f3 = (c >> 4) & 1;
  const uint32_t f4 = (c >> 3) & 1, f5 = (c >> 2) & 1, f6 = (c >> 1) & 1, sh = c & 1;
  const uint32_t q = f0 ^ f1 ^ f2 ^ f3;
  return (f1 << 15) | (f2 << 14) | (f3 << 13) | (q << 12) | (a << 4) | (f4 << 3) | (f5 << 2) |
         (f6 << 1) | sh;
}

struct PackArgs {
  const void* codes;
  int code_bytes;
  int64_t m, T;
  int kind;
  int layout;
  void* out;
};

__global__ __launch_bounds__(256) void pack_kernel(PackArgs A) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= A.m * A.T) return;
  const int64_t r = k / A.T, t = k % A.T;
  uint32_t c = load_code(A.codes, A.code_bytes, k);
  int64_t o = k;
  if (A.layout == QS_LAYOUT_TILED) {
    const int64_t S = A.T / 32;
    const int64_t rb = r >> 4, rr = r & 15, sl = t >> 5, tt = t & 31;
    const int64_t lane = (tt >> 3) * 16 + rr;
    o = ((rb * S + sl) * 64 + lane) * 8 + (tt & 7);
  }
  if (A.kind == QS_STAGE_E8P) {
    static_cast<uint16_t*>(A.out)[o] =
        (uint16_t)(A.layout == QS_LAYOUT_TILED ? kernel_form(c & 0xFFFF) : (c & 0xFFFF));
  } else {
    static_cast<uint8_t*>(A.out)[o] = (uint8_t)(c & 0xFF);
  }
}

__global__ __launch_bounds__(256) void div_kernel(const float* in, float* out, int64_t n, float d) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = in[i] / d;
}

}  // namespace
}  // namespace qs

using namespace qs;

extern "C" int qs_div_f32(const float* in, float* out, int64_t count, float divisor, qs_stream_t stream) {
  QS_REQUIRE(count >= 0, "count must be >= 0");
  QS_REQUIRE(divisor != 0.0f, "divisor must be non-zero");
  if (count == 0) return QS_OK;
  QS_REQUIRE(in && out, "null pointer");
  QS_REQUIRE((count + 255) / 256 < (1ll << 31), "count too large");
  hipLaunchKernelGGL(div_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, as_stream(stream), in, out,
                     count, divisor);
  QS_LAUNCHED("div_kernel");
  return QS_OK;
}

extern "C" int qs_e8p_abs_table(float* out_host) {
  QS_REQUIRE(out_host, "null output");
  for (int r = 0; r < 256; ++r)
    for (int i = 0; i < 8; ++i) out_host[r * 8 + i] = kE8PHost.v[r][i];
  return QS_OK;
}

extern "C" int qs_e81_table(float* out_host) {
  QS_REQUIRE(out_host, "null output");
  for (int r = 0; r < 256; ++r)
    for (int i = 0; i < 8; ++i) out_host[r * 8 + i] = kE81Host.v[r][i];
  return QS_OK;
}

extern "C" int qs_rvq_encode(const float* x, int64_t ldx, int64_t nvec, int nstages, const int* kinds,
                             const float* scales, float in_div, float out_mul, float* vals, int64_t ldv,
                             void* codes, int code_bytes, int64_t code_stage_stride, int64_t code_stride,
                             qs_stream_t stream) {
  QS_REQUIRE(nvec >= 0, "nvec must be >= 0");
  QS_REQUIRE(nvec == 0 || x, "null input");
  QS_REQUIRE(ldx >= 8 && (!vals || ldv >= 8), "row strides must be >= 8");
  QS_REQUIRE(!codes || code_bytes == 2 || code_bytes == 4 || code_bytes == 8, "code_bytes must be 2, 4 or 8");
  EncodeArgs A{};
  int rc = fill_stages(A.st, nstages, kinds, scales);
  if (rc) return rc;
  A.base = x;
  A.ldbase = ldx;
  A.vals = vals;
  A.ldvals = ldv;
  A.codes = codes;
  A.code_bytes = code_bytes;
  A.code_stage_stride = code_stage_stride;
  A.code_stride = code_stride;
  A.nvec = nvec;
  A.in_div = in_div;
  A.out_mul = out_mul;
  QS_REQUIRE(in_div != 0.0f, "in_div must be non-zero");
  return launch_encode(A, as_stream(stream));
}

extern "C" int qs_ldlq_step(const float* base, int64_t ldbase, const float* delta, const float* dinv,
                            const float* w, int64_t ldw, float* wq, int64_t ldwq, float* resid,
                            int64_t ldresid, int64_t m, int nstages, const int* kinds, const float* scales,
                            void* codes, int code_bytes, int64_t code_stage_stride, int64_t code_stride,
                            qs_stream_t stream) {
  QS_REQUIRE(m >= 0, "m must be >= 0");
  QS_REQUIRE(m == 0 || (base && delta && wq), "base, delta and wq are required");
  QS_REQUIRE(!resid || w, "resid needs w");
  QS_REQUIRE(ldbase >= 8 && ldwq >= 8 && (!resid || (ldw >= 8 && ldresid >= 8)), "row strides must be >= 8");
  QS_REQUIRE(!codes || code_bytes == 2 || code_bytes == 4 || code_bytes == 8, "code_bytes must be 2, 4 or 8");
  EncodeArgs A{};
  int rc = fill_stages(A.st, nstages, kinds, scales);
  if (rc) return rc;
  A.base = base;
  A.ldbase = ldbase;
  A.delta = delta;
  A.dinv = dinv;
  A.vals = wq;
  A.ldvals = ldwq;
  A.w = w;
  A.ldw = ldw;
  A.resid = resid;
  A.ldresid = ldresid;
  A.codes = codes;
  A.code_bytes = code_bytes;
  A.code_stage_stride = code_stage_stride;
  A.code_stride = code_stride;
  A.nvec = m;
  A.in_div = 1.0f;
  A.out_mul = 1.0f;
  return launch_encode(A, as_stream(stream));
}

extern "C" int qs_ldlq_chunk(const float* w, int64_t ldw, float* wq, int64_t ldwq, float* e, int64_t lde,
                             const float* p, int64_t ldp, const float* h, int64_t ldh, const float* dinv, int c0,
                             int nb, int64_t m, int nstages, const int* kinds, const float* scales, void* codes,
                             int code_bytes, int64_t code_stage_stride, int64_t code_stride, qs_stream_t stream) {
  QS_REQUIRE(m >= 0 && nb >= 1 && nb <= kChunkBlocks && c0 >= 0, "m %lld, nb %d (1..%d), c0 %d", (long long)m, nb,
             kChunkBlocks, c0);
  QS_REQUIRE(m == 0 || (w && wq && e && p && h && dinv), "w, wq, e, p, h and dinv are required");
  QS_REQUIRE(ldw >= 8 * (c0 + nb) && ldwq >= 8 * (c0 + nb) && lde >= 8 * (c0 + nb) && ldp >= 8 * nb &&
                 ldh >= 8 * (c0 + nb),
             "row strides too small");
  QS_REQUIRE(!codes || code_bytes == 2 || code_bytes == 4 || code_bytes == 8, "code_bytes must be 2, 4 or 8");
  ChunkArgs A{};
  int rc = fill_stages(A.st, nstages, kinds, scales);
  if (rc) return rc;
  if (m == 0) return QS_OK;
  QS_REQUIRE(m / 16 < (1ll << 31) - 1, "m too large: %lld", (long long)m);
  A.w = w;
  A.ldw = ldw;
  A.wq = wq;
  A.ldwq = ldwq;
  A.e = e;
  A.lde = lde;
  A.p = p;
  A.ldp = ldp;
  A.h = h;
  A.ldh = ldh;
  A.dinv = dinv;
  A.c0 = c0;
  A.nb = nb;
  A.m = m;
  A.codes = codes;
  A.code_bytes = code_bytes;
  A.code_stage_stride = code_stage_stride;
  A.code_stride = code_stride;
  // 16 rows per work-group (one per CU by its LDS) up to one round of the 256
  // CUs, 32 beyond: two waves per SIMD then share H's chunk
  const int rows = m > 16 * 256 ? kChunkMaxRows : 16;
  const size_t lds = chunk_lds(rows);
  // the limit is the same for every call, so that threads do not lower each other's
  QS_HIP(hipFuncSetAttribute((const void*)ldlq_chunk_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kChunkMaxLds));
  hipLaunchKernelGGL(ldlq_chunk_kernel, dim3((unsigned)((m + rows - 1) / rows)), dim3(16 * rows), lds,
                     as_stream(stream), A);
  QS_LAUNCHED("ldlq_chunk_kernel");
  return QS_OK;
}

extern "C" int qs_rvq_decode(const void* codes, int code_bytes, int64_t code_stage_stride, int64_t nvec,
                             int nstages, const int* kinds, const float* scales, float out_scale, float* out,
                             qs_stream_t stream) {
  QS_REQUIRE(nvec >= 0, "nvec must be >= 0");
  QS_REQUIRE(nvec == 0 || (codes && out), "null pointer");
  QS_REQUIRE(code_bytes == 2 || code_bytes == 4 || code_bytes == 8, "code_bytes must be 2, 4 or 8");
  QS_REQUIRE((reinterpret_cast<uintptr_t>(out) & 15) == 0, "out must be 16-byte aligned");
  DecodeArgs A{};
  int rc = fill_stages(A.st, nstages, kinds, scales);
  if (rc) return rc;
  A.codes = codes;
  A.code_bytes = code_bytes;
  A.stage_stride = code_stage_stride;
  A.nvec = nvec;
  A.out_scale = out_scale;
  A.out = out;
  if (nvec == 0) return QS_OK;
  hipLaunchKernelGGL(rvq_decode_kernel, dim3((unsigned)((nvec + 255) / 256)), dim3(256), 0, as_stream(stream), A);
  QS_LAUNCHED("rvq_decode_kernel");
  return QS_OK;
}

extern "C" int qs_pack_codes(const void* codes, int code_bytes, int64_t m, int64_t n, int stage_kind,
                             int layout, void* out, qs_stream_t stream) {
  QS_REQUIRE(m >= 0 && n >= 0 && n % 8 == 0, "n must be a multiple of 8");
  QS_REQUIRE(code_bytes == 2 || code_bytes == 4 || code_bytes == 8, "code_bytes must be 2, 4 or 8");
  QS_REQUIRE(stage_kind == QS_STAGE_E8P || stage_kind == QS_STAGE_E8_1BIT, "bad stage kind");
  QS_REQUIRE(layout == QS_LAYOUT_ROWMAJOR || layout == QS_LAYOUT_TILED, "bad layout");
  if (layout == QS_LAYOUT_TILED)
    QS_REQUIRE(m % 16 == 0 && n % 256 == 0, "tiled layout needs m %% 16 == 0 and n %% 256 == 0 (m=%lld n=%lld)",
               (long long)m, (long long)n);
  const int64_t total = m * (n / 8);
  if (total == 0) return QS_OK;
  QS_REQUIRE(codes && out, "null pointer");
  PackArgs A{codes, code_bytes, m, n / 8, stage_kind, layout, out};
  hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, as_stream(stream), A);
  QS_LAUNCHED("pack_kernel");
  return QS_OK;
}
