// Randomized Hadamard transform along one axis of a [outer][n][inner] fp32
// tensor: the quantize-time incoherence transforms of quipsharp/incoherence.py
// (W_hat = H_m (S_u W S_v) H_n, H_hat = H_n (S_v H S_v) H_n, their inverses,
// and transform_input/transform_output).  The Walsh-Hadamard part is bit-exact
// with quipsharp/hadamard.py:17-40.
//
//  inner == 1 : a work-group takes one or several whole rows; butterflies of up
//               to 16 elements in registers, LDS between the rounds, the first
//               round reading and the last writing memory.
//  inner  > 1 : passes of up to seven stages with a column's elements in one
//               thread's registers (no LDS), then the odd-factor pass.
#include <cmath>

#include "qs_rht_dev.h"

namespace qs {
namespace {

constexpr int kMaxRowLen = 32768;  // 128 KiB of LDS
constexpr int kMaxRowLds = padded_len(kMaxRowLen) * 4;
constexpr int kSpan = 4096;        // elements per work-group when rows are shorter
constexpr int kKronTile = 8;       // outputs per LDS read of the odd-factor stage

// Walsh-Hadamard stages h = 1, 2, ... of 2^BITS values in registers.
template <int BITS>
__device__ __forceinline__ void reg_fwht(float (&v)[1 << BITS]) {
#pragma unroll
  for (int s = 0; s < BITS; ++s) {
    const int hh = 1 << s;
#pragma unroll
    for (int j = 0; j < (1 << BITS); ++j) {
      if ((j & hh) == 0) {
        const float x = v[j], y = v[j + hh];
        v[j] = x + y;
        v[j + hh] = x - y;
      }
    }
  }
}

// s[i] = sum_c K[a0 + i][c] value(c) for i < 8 (rows past p repeat the last one),
// c ascending, K (p x p, wave-uniform addresses) in scalar registers, four
// columns of it requested together.
template <class Value>
__device__ __forceinline__ void kron_tile(const float* __restrict__ K, int p, int a0, Value value,
                                          float (&s)[kKronTile]) {
  const float* Kr[kKronTile];
#pragma unroll
  for (int i = 0; i < kKronTile; ++i) {
    Kr[i] = K + (a0 + i < p ? a0 + i : p - 1) * p;
    s[i] = 0.0f;
  }
  int c = 0;
  for (; c + 4 <= p; c += 4) {
    float k[kKronTile][4], v[4];
#pragma unroll
    for (int i = 0; i < kKronTile; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) k[i][u] = Kr[i][c + u];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = value(c + u);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < kKronTile; ++i) s[i] = __builtin_fmaf(k[i][u], v[u], s[i]);
  }
  for (; c < p; ++c) {
    const float v = value(c);
#pragma unroll
    for (int i = 0; i < kKronTile; ++i) s[i] = __builtin_fmaf(Kr[i][c], v, s[i]);
  }
}

struct RowArgs {
  const float* in;
  float* out;
  int64_t outer;
  int n, logL, p, G;
  int rows;  // rows per work-group (more than one: n is a power of two)
  const float* pre;
  const float* post;
  float scale;
  int wide;  // rows start on 16 bytes
};

// First round: 2^BITS consecutive elements per thread, from memory.  total:
// elements of this work-group (the rows are adjacent).
template <int BITS, class Put>
__device__ __forceinline__ void first_round(const RowArgs& A, const float* src, int total, Put put) {
  constexpr int R = 1 << BITS;
  for (int g = threadIdx.x; g < (total >> BITS); g += blockDim.x) {
    float v[R];
    if (BITS >= 2 && A.wide) {
#pragma unroll
      for (int j = 0; j < R / 4; ++j) {
        const float4 f = reinterpret_cast<const float4*>(src + g * R)[j];
        v[4 * j] = f.x, v[4 * j + 1] = f.y, v[4 * j + 2] = f.z, v[4 * j + 3] = f.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = src[g * R + j];
    }
    if (A.pre) {
      const int i0 = A.rows == 1 ? g * R : (g * R) & (A.n - 1);
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = v[j] * A.pre[i0 + j];
    }
    reg_fwht<BITS>(v);
    put(g, v);
  }
}

// A later round: elements 2^logh0 apart, from LDS.
template <int BITS, class Put>
__device__ __forceinline__ void later_round(const float* buf, int total, int logh0, Put put) {
  constexpr int R = 1 << BITS;
  for (int g = threadIdx.x; g < (total >> BITS); g += blockDim.x) {
    const int off = g & ((1 << logh0) - 1);
    const int base = ((g >> logh0) << (logh0 + BITS)) + off;
    float v[R];
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = buf[pad_idx(base + (j << logh0))];
    reg_fwht<BITS>(v);
    put(base, v);
  }
}

// The stages of rows of length n = p L: rounds of up to four stages, then the
// odd factor.  Bound by memory (8 bytes an element): a 4096-point row is 256
// threads of 16 elements and two exchanges through LDS, with eight such
// work-groups on a CU (six radix-4 rounds on 1024 threads, each between two
// barriers, ran at half the copy rate).  4096 x 11008 (p = 43) 393 -> 174 us.
//
// The odd-factor stage is p FMAs per element: a wave takes 64 columns b and
// eight rows a of K at a time, K in scalar registers, so that one LDS read
// serves eight FMAs (one read each of K and the value per FMA was bound by LDS).
template <int BITS>  // stages per round (the last round takes what is left)
__global__ __launch_bounds__(512) void rht_rows_kernel(RowArgs A, const float* __restrict__ K) {
  extern __shared__ float buf[];
  const int64_t first = (int64_t)(blockIdx.x / A.G) * A.rows;
  const int part = blockIdx.x % A.G;
  const int here = A.outer - first < A.rows ? (int)(A.outer - first) : A.rows;
  const int total = here * A.n;
  const float* src = A.in + first * A.n;
  float* dst = A.out + first * A.n;
  const float scale = A.scale;
  auto finish = [&](int i, float v) __attribute__((always_inline)) {  // p == 1
    v = v * scale;
    if (A.post) v = v * A.post[A.rows == 1 ? i : i & (A.n - 1)];
    dst[i] = v;
  };
  if (A.logL <= BITS && A.p == 1) {  // logL == BITS: one round, registers only
    first_round<BITS>(A, src, total, [&](int g, float (&v)[1 << BITS]) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < (1 << BITS); ++j) finish((g << BITS) + j, v[j]);
    });
    return;
  }
  const float first_scale = A.logL <= BITS ? scale : 1.0f;
  first_round<BITS>(A, src, total, [&](int g, float (&v)[1 << BITS]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < (1 << BITS); ++j) buf[pad_idx((g << BITS) + j)] = v[j] * first_scale;
  });
  __syncthreads();
  for (int done = BITS; done < A.logL;) {
    const int left = A.logL - done;
    if (left > BITS) {
      later_round<BITS>(buf, total, done, [&](int base, float (&v)[1 << BITS]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < (1 << BITS); ++j) buf[pad_idx(base + (j << done))] = v[j];
      });
    } else {  // the last round: scaled, to memory or back for the odd factor
      auto last = [&](auto bits) __attribute__((always_inline)) {
        constexpr int B = decltype(bits)::value;
        later_round<B>(buf, total, done, [&](int base, float (&v)[1 << B]) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < (1 << B); ++j) {
            const int i = base + (j << done);
            if (A.p == 1) finish(i, v[j]);
            else buf[pad_idx(i)] = v[j] * scale;
          }
        });
      };
      if (left == 1) last(std::integral_constant<int, 1>());
      else if (BITS >= 2 && left == 2) last(std::integral_constant<int, BITS >= 2 ? 2 : 1>());
      else if (BITS >= 3 && left == 3) last(std::integral_constant<int, BITS >= 3 ? 3 : 1>());
      else last(std::integral_constant<int, BITS>());
    }
    done += left > BITS ? BITS : left;
    __syncthreads();
  }
  if (A.p == 1) return;
  const int p = A.p, L = 1 << A.logL;
  const float* post = A.post;
  if (L < 64) {  // few columns: one output per thread
    kron_cols(buf, K, p, A.logL, part * (L / A.G), (part + 1) * (L / A.G), threadIdx.x, blockDim.x,
              [&](int a, int b, float v) {
                const int i = (a << A.logL) + b;
                dst[i] = post ? v * post[i] : v;
              });
    return;
  }
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const int tiles = (p + kKronTile - 1) / kKronTile, items = tiles * (L >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(part * waves + (threadIdx.x >> 6));
  for (int t = wave; t < items; t += A.G * waves) {
    const int a0 = (t % tiles) * kKronTile, b = ((t / tiles) << 6) + lane;
    float s[kKronTile];
    kron_tile(K, p, a0, [&](int c) { return buf[pad_idx((c << A.logL) + b)]; }, s);
#pragma unroll
    for (int i = 0; i < kKronTile; ++i) {
      if (a0 + i < p) {
        const int o = ((a0 + i) << A.logL) + b;
        dst[o] = post ? s[i] * post[o] : s[i];
      }
    }
  }
}

// Walsh-Hadamard stages h0, 2 h0, ..., h0 2^(BITS - 1) on the axis: a thread
// takes one column of one butterfly group (2^BITS elements, h0 apart), so every
// access of a wave is 256 consecutive bytes, all loads of a group are in flight
// at once and nothing is exchanged.  Bound by memory: 4096 x 11008, six stages:
// 124 -> 65 us (a 64 x 64 tile in LDS with a barrier per stage before).
struct ColArgs {
  const float* in;
  float* out;
  int64_t outer, n, inner;
  int L;         // length of the Walsh-Hadamard part (n = p*L)
  int h0;        // first stage of this pass
  const float* pre_axis;
  const float* pre_inner;
  const float* post_axis;
  float scale;   // applied when != 0 (last Walsh-Hadamard pass)
};

template <int BITS>
__global__ __launch_bounds__(256) void rht_cols_pass_kernel(ColArgs A) {
  constexpr int R = 1 << BITS;
  // group id -> (o, a, blk, off): elements a*L + blk*h0*R + off + h0*j
  const int64_t per_seg = A.L >> BITS, per_o = (A.n / A.L) * per_seg;
  const int64_t o = blockIdx.x / per_o, g = blockIdx.x - o * per_o;
  const int64_t a = g / per_seg, gi = g - a * per_seg;
  const int64_t blk = gi / A.h0, off = gi - blk * A.h0;
  const int64_t i0 = a * A.L + blk * (int64_t)A.h0 * R + off;
  const int64_t c = (int64_t)blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= A.inner) return;
  const int64_t step = (int64_t)A.h0 * A.inner, at = (o * A.n + i0) * A.inner + c;
  float v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = A.in[at + j * step];
  if (A.pre_axis) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = v[j] * A.pre_axis[i0 + (int64_t)A.h0 * j];
  }
  if (A.pre_inner) {
    const float s = A.pre_inner[c];
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = v[j] * s;
  }
  reg_fwht<BITS>(v);
  if (A.scale != 0.0f) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = v[j] * A.scale;
  }
  if (A.post_axis) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = v[j] * A.post_axis[i0 + (int64_t)A.h0 * j];
  }
#pragma unroll
  for (int j = 0; j < R; ++j) A.out[at + j * step] = v[j];
}

// Odd-factor pass: for each (o, b, c): out[a] = sum_a' K[a][a'] in[a'], a = 0..p-1.
// The p values of 64 columns in LDS; a wave forms eight outputs per LDS read,
// K in scalar registers.
struct KronColArgs {
  const float* in;
  float* out;
  int64_t outer, n, inner;
  int L, p;
  const float* post_axis;
};

__global__ __launch_bounds__(256) void rht_cols_kron_kernel(KronColArgs A, const float* __restrict__ K) {
  __shared__ float tile[QS_MAX_KRON][64];
  const int64_t o = blockIdx.x / A.L;
  const int64_t b = blockIdx.x - o * A.L;
  const int tc = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t c = (int64_t)blockIdx.y * 64 + tc;
  const bool cvalid = c < A.inner;
  const int p = A.p;
#pragma unroll 4
  for (int a = wave; a < p; a += 4)
    tile[a][tc] = cvalid ? A.in[(o * A.n + a * (int64_t)A.L + b) * A.inner + c] : 0.0f;
  __syncthreads();
  for (int a0 = wave * kKronTile; a0 < p; a0 += 4 * kKronTile) {
    float s[kKronTile];
    kron_tile(K, p, a0, [&](int c) { return tile[c][tc]; }, s);
#pragma unroll
    for (int i = 0; i < kKronTile; ++i) {
      if (a0 + i < p && cvalid) {
        const int64_t at = (a0 + i) * (int64_t)A.L + b;
        A.out[(o * A.n + at) * A.inner + c] = A.post_axis ? s[i] * A.post_axis[at] : s[i];
      }
    }
  }
}

template <int BITS>
void launch_cols(const ColArgs& A, int64_t groups, hipStream_t s) {
  const int threads = A.inner >= 256 ? 256 : (int)((A.inner + 63) / 64 * 64);
  hipLaunchKernelGGL(rht_cols_pass_kernel<BITS>, dim3((unsigned)groups, (unsigned)((A.inner + threads - 1) / threads)),
                     dim3(threads), 0, s, A);
}

template <int BITS>
int launch_rows(const RowArgs& A, const float* K, int64_t blocks, int threads, size_t lds, hipStream_t s) {
  if (lds > 65536)  // the longest row's: a limit of its own could be another thread's next launch's
    QS_HIP(hipFuncSetAttribute((const void*)rht_rows_kernel<BITS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               kMaxRowLds));
  hipLaunchKernelGGL(rht_rows_kernel<BITS>, dim3((unsigned)blocks), dim3(threads), lds, s, A, K);
  QS_LAUNCHED("rht_rows_kernel");
  return QS_OK;
}

}  // namespace
}  // namespace qs

using namespace qs;

extern "C" int qs_rht_f32(const float* in, float* out, int64_t outer, int64_t n, int64_t inner,
                          const float* pre_axis, const float* pre_inner, const float* post_axis, int kron_p,
                          const float* kron_mat, qs_stream_t stream) {
  QS_REQUIRE(outer >= 0 && n >= 1 && inner >= 1, "bad shape outer=%lld n=%lld inner=%lld", (long long)outer,
             (long long)n, (long long)inner);
  QS_REQUIRE(kron_p >= 1 && (kron_p & 1) && kron_p <= QS_MAX_KRON, "kron_p must be odd in [1, %d]", QS_MAX_KRON);
  QS_REQUIRE(n % kron_p == 0, "n=%lld is not divisible by kron_p=%d", (long long)n, kron_p);
  const int64_t L = n / kron_p;
  QS_REQUIRE((L & (L - 1)) == 0, "n / kron_p must be a power of two (n=%lld, p=%d)", (long long)n, kron_p);
  QS_REQUIRE(kron_p == 1 || kron_mat, "kron_mat is required when kron_p > 1");
  QS_REQUIRE(in && out, "null pointer");
  if (outer == 0) return QS_OK;
  hipStream_t s = as_stream(stream);
  const float scale = inv_sqrt_len(L);
  const int logL = log2_exact(L);
  if (inner == 1) {
    QS_REQUIRE(n <= kMaxRowLen, "row transform supports n <= %d (got %lld)", kMaxRowLen, (long long)n);
    RowArgs A{};
    A.in = in;
    A.out = out;
    A.outer = outer;
    A.n = (int)n;
    A.logL = logL;
    A.p = kron_p;
    A.pre = pre_axis;
    A.post = post_axis;
    A.scale = scale;
    // short rows without an odd factor share a work-group
    A.rows = kron_p == 1 && n < kSpan ? (int)(kSpan / n) : 1;
    A.wide = (reinterpret_cast<uintptr_t>(in) & 15) == 0 && n % 4 == 0;
    // 16 elements per thread, 512 threads at most; few rows: several
    // work-groups read a row and share its odd-factor stage (when the output
    // does not overwrite the input)
    const int64_t span = A.rows * n;
    const int threads = span <= kSpan ? 256 : 512;
    A.G = 1;
    if (kron_p > 1 && in != out && outer < 256) {
      const int64_t shares = L >= 64 ? ((kron_p + kKronTile - 1) / kKronTile * (L / 64) + threads / 64 - 1) / (threads / 64)
                                     : 1;
      // a last doubling that leaves some waves without a tile only while the rows leave CUs free
      // (1 to 16 rows of 11008: 14 -> 10 us; 33 rows of 18944: 17 -> 19)
      while (A.G < shares && A.G * 2 * outer <= (A.G * 2 <= shares ? 512 : 256) && A.G < 16) A.G *= 2;
    }
    const int64_t blocks = (outer + A.rows - 1) / A.rows * A.G;
    QS_REQUIRE(blocks < (1ll << 31), "too many rows");
    // rounds of equal depth, four stages at most
    const int rounds = logL > 0 ? (logL + 3) / 4 : 1, bits = (logL + rounds - 1) / rounds;
    const bool direct = rounds == 1 && kron_p == 1;
    const size_t lds = direct ? 0 : (size_t)padded_len((int)span) * sizeof(float);
    switch (bits) {
      case 0: return launch_rows<0>(A, kron_mat, blocks, threads, lds, s);
      case 1: return launch_rows<1>(A, kron_mat, blocks, threads, lds, s);
      case 2: return launch_rows<2>(A, kron_mat, blocks, threads, lds, s);
      case 3: return launch_rows<3>(A, kron_mat, blocks, threads, lds, s);
      default: return launch_rows<4>(A, kron_mat, blocks, threads, lds, s);
    }
  }
  // column passes of equal depth, seven stages (128 registers) at most; a length
  // without stages still runs one pass to apply the signs
  QS_REQUIRE((inner + 63) / 64 < 65536, "inner too large");
  const int passes = logL > 0 ? (logL + 6) / 7 : 1;
  const float* src = in;
  int done = 0;
  for (int pass = 0; pass < passes; ++pass) {
    const int bits = (logL - done + passes - pass - 1) / (passes - pass);
    const bool last = pass == passes - 1;
    ColArgs A{};
    A.in = src;
    A.out = out;
    A.outer = outer;
    A.n = n;
    A.inner = inner;
    A.L = (int)L;
    A.h0 = 1 << done;
    A.pre_axis = pass == 0 ? pre_axis : nullptr;
    A.pre_inner = pass == 0 ? pre_inner : nullptr;
    A.post_axis = (last && kron_p == 1) ? post_axis : nullptr;
    A.scale = last ? scale : 0.0f;
    const int64_t groups = outer * kron_p * (L >> bits);
    QS_REQUIRE(groups < (1ll << 31), "too many groups");
    switch (bits) {
      case 0: launch_cols<0>(A, groups, s); break;
      case 1: launch_cols<1>(A, groups, s); break;
      case 2: launch_cols<2>(A, groups, s); break;
      case 3: launch_cols<3>(A, groups, s); break;
      case 4: launch_cols<4>(A, groups, s); break;
      case 5: launch_cols<5>(A, groups, s); break;
      case 6: launch_cols<6>(A, groups, s); break;
      default: launch_cols<7>(A, groups, s); break;
    }
    QS_LAUNCHED("rht_cols_pass_kernel");
    src = out;
    done += bits;
  }
  if (kron_p > 1) {
    KronColArgs K{out, out, outer, n, inner, (int)L, kron_p, post_axis};
    const int64_t groups = outer * L;
    QS_REQUIRE(groups < (1ll << 31), "too many groups");
    hipLaunchKernelGGL(rht_cols_kron_kernel, dim3((unsigned)groups, (unsigned)((inner + 63) / 64)), dim3(256), 0, s, K,
                       kron_mat);
    QS_LAUNCHED("rht_cols_kron_kernel");
  }
  return QS_OK;
}
