// Wide-batch quantized-linear forward (prefill: 17 or more activation rows
// per call), the path QuantizedLinear.forward takes for a long prompt
// (quipsharp/checkpoint.py:141-146 -> quipsharp/quantize.py:116-124: the
// reference decodes the whole weight and multiplies densely).  With many
// rows the contraction is a real GEMM: wg_kernel decodes the codes inside
// its K loop (byte LUTs in LDS, exactly as the narrow kernels) and feeds
// every decoded fragment to several 16 x 16 x 32 fp16 MFMAs; the codes' +-1/4
// shifts are one extra MFMA per slice against the operand's group sums.
// Single-stage calls of more than 128 rows, and large linears from 65, take
// wp_kernel instead, which splits decoding and multiplying between the waves of
// a work-group.  The transforms around it write the fragment-major operand and
// read the partial sums: one row per wave for a long batch (qs_linear_rows.hip),
// otherwise the per-row kernels of the batched path (qs_linear_batched.hip,
// qs_linear_big.hip) or, for lengths that these do not cover, the LDS-radix
// kernels of qs_linear.hip.
#include <type_traits>

#include "qs_forward_dev.h"
#include "qs_linear_dev.h"

namespace qs {
namespace {

constexpr int kDqOffHi = 0;                // 4096 x uint32 LUT entries
constexpr int kDqOffLo = 16384;
constexpr int kDqOffLut1 = 32768;          // 256 x uint4 (E8 1-bit rows, fp16)

// ---------------------------------------------------------------------------
// Decode in the GEMM loop
// ---------------------------------------------------------------------------
// A work-group's 4 waves take 128 weight rows and up to 128 activation rows.
// Two reads bound the loop: the LDS tables (two words a code, 16 bytes more with
// a second stage: 10 and 26 clocks per 64 codes) and the operand through the
// L1 (1 KiB a fragment, 16 clocks).  With WC = 1 every wave has two 16-row code
// tiles of its own and multiplies all of the activation rows, so that a code is
// decoded once and a fragment read four times; with WC = 2, 65 to 128 rows of
// one stage (the large linears of which wp_kernel takes), the waves are 2 x 2,
// four code tiles by half the rows each, both twice.  (A wave with all the weight
// rows and activation rows of its own, as this kernel was, decodes every code
// four times.)  A wave's code tiles go from memory to its registers a slice
// ahead, and the loop has no barrier.
//
// A layer's linears and transforms, graph-replayed (that form -> now):
//   Llama-3-8B 3 bits  17 rows 178 -> 127 us, 45 202 -> 163, 128 308 -> 267, 700 1256 -> 1154
//   Qwen3-32B 2 bits   17 rows 250 -> 184 us, 45 291 -> 239, 64 325 -> 272
//   the same, 128 rows 437 -> 417 us (WC = 1: 520), 359 with wp_kernel for the
//   large ones; 3 bits 559 -> 501 (WC = 2: 522)
//
// Linears of one operand width share a launch, each with the slice groups that
// it has alone, so that the outputs do not depend on the company.
constexpr int kWgThreads = 256;
constexpr int kWgWaves = kWgThreads / 64;
constexpr int kWgRowTiles = 8;                       // 16-row code tiles of a work-group
constexpr int kWgMaxCols = 8;                        // 16-row activation tiles of a work-group
constexpr int kWgLds = kDqOffLut1 + 4096;
constexpr int64_t kWgPartialBytes = 8 << 20;         // of partial sums for a second work-group per CU
static_assert(kWgThreads >= 256, "E8 one-bit table rows: one per thread of the first 256");

// Activation tiles per work-group: the tiles dealt evenly over as few
// work-group columns as take them, rounded up to a compiled width.
inline int wg_cols(int64_t B) {
  const int64_t nbt = (B + 15) / 16, nct = (nbt + kWgMaxCols - 1) / kWgMaxCols;
  const int64_t nb = (nbt + nct - 1) / nct;
  return nb <= 2 ? 2 : nb <= 3 ? 3 : nb <= 4 ? 4 : nb <= 6 ? 6 : 8;
}
// Single-stage linears run wp_kernel (256 activation rows per work-group) beyond
// 128 rows, those of more than 2^24 weights beyond 64: wg_kernel's 2 x 2 form
// wants two work-groups per CU, which one linear of 65 to 128 rows seldom has
// (alone it was 2 to 22 % slower than the form before it).
// One linear, 128 rows, wg_kernel -> wp_kernel: 5120 x 25600 123 -> 89 us, 11008
// x 4096 56.2 -> 45.6, 4096 x 4096 34.2 -> 33.1.  The smaller ones are mostly
// members of a group, whose launch wg_kernel shares whatever their m: 4096 to
// 4096 + 1024 + 1024 42.5 us, by wp_kernel, each or together, 46.6 and more.
constexpr int64_t kWpWeights = 1 << 24;
inline bool use_wp(int64_t m, int64_t n, int64_t B, bool has2) {
  return !has2 && (B > 16 * kWgMaxCols || (B > 64 && m * n > kWpWeights));
}
inline bool use_wp(const WideMfma& F) { return use_wp(F.m, F.n, F.B, F.codes1 != nullptr); }

// One linear of a launch.  wp_kernel: linears of one shape (m, n, rows) that
// read their own operands share a launch, job j taking tiles j T1 .. (j + 1) T1
// - 1 of the grid's tile order (T1 = nrt nct SGk).
struct WpJob {
  const uint16_t* codes0;
  const _Float16* x2f;
  float* y1p;
  float s0;
  // wg_kernel
  const uint8_t* codes1;
  const _Float16* sgf;
  float s1;
  int m, RB, nrt, SGk, spg;
  int wg0, tiles;      // first work-group (a multiple of 8), tiles
};

struct WgArgs {
  int m, B, S, RB;     // RB: 16-row blocks
  int nrt, nct;        // work-group tiles along the weight rows / activation rows
  int SGk, spg;        // slice groups, slices per group
  int njobs;
  WpJob job[QS_MAX_GROUP];
};

template <bool HAS2, int NB, int WC>
__global__ __launch_bounds__(kWgThreads, 2) void wg_kernel(WgArgs A) {
  constexpr int RT = kWgRowTiles * WC / kWgWaves;  // code tiles of a wave
  // steps between an operand load and its use (one where two stages' sums take the registers)
  constexpr int kAhead = NB <= 4 ? 3 : 1, kRing = kAhead + 1;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  uint4* lut1 = reinterpret_cast<uint4*>(lds + kDqOffLut1);
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, r16 = lane & 15;

  // A job's tiles are ordered weight-row tiles fastest, then activation tiles,
  // then slice groups, and dealt to the XCDs in contiguous runs: work-group i
  // runs on XCD i % 8, so tile (i % 8) * ceil(T / 8) + i / 8 keeps each XCD's L2
  // on a few activation columns and slice groups (surplus work-groups exit at
  // once).  Each job by itself: in one run over the jobs the tiles of a large
  // linear, which has few slice groups of many slices, fell on a few XCDs (two
  // stages, 5120 columns to 8192 + 1024 + 1024 at 300 rows: 285 us in one run,
  // 220 in a launch each, 162 dealt job by job; linears of one shape equal).
  int jj = 0;
#pragma unroll
  for (int k = 1; k < QS_MAX_GROUP; ++k)
    if (k < A.njobs && (int)blockIdx.x >= A.job[k].wg0) jj = k;
  const WpJob& J = A.job[jj];
  const int local = (int)blockIdx.x - J.wg0;
  int bid = (local & 7) * ((J.tiles + 7) >> 3) + (local >> 3);
  if (bid >= J.tiles) return;
  const int rt = bid % J.nrt;
  bid /= J.nrt;
  const int ct = bid % A.nct;
  const int g = bid / A.nct;
  const int s_begin = g * J.spg;
  const int s_end = s_begin + J.spg < A.S ? s_begin + J.spg : A.S;
  const int s_last = s_end > s_begin ? s_end - 1 : (A.S - 1);  // an empty group reads, never uses, slice S - 1

  // this wave's code tiles; row blocks past the end read the last one (decoded, never stored)
  const int rb0 = rt * kWgRowTiles + w / WC * RT;
  uint4 cw[RT], nw[RT];
  uint2 cw1[RT], nw1[RT];
  auto load_codes = [&](int s) __attribute__((always_inline)) {
    s = s < s_last ? s : s_last;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int rb = rb0 + i < J.RB ? rb0 + i : J.RB - 1;
      const size_t tile = (size_t)rb * A.S + s;
      nw[i] = ld_nt_u4(reinterpret_cast<const char*>(J.codes0) + tile * 1024 + 16 * lane);
      if (HAS2) nw1[i] = *reinterpret_cast<const uint2*>(J.codes1 + tile * 512 + 8 * lane);
    }
  };

  // activation tiles (clamped to the last one: computed, never stored)
  const int nbt = (A.B + 15) >> 4;
  const _Float16* xb[NB];
  const _Float16* sb[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    int c = NB * (WC * ct + w % WC) + t;
    c = c < nbt ? c : nbt - 1;
    xb[t] = J.x2f + (size_t)c * A.S * 8 * 512 + 8 * lane;  // + (s * 8 + step) * 512 halves
    sb[t] = J.sgf + (size_t)c * A.S * 512 + 8 * lane;      // + s * 512 halves
  }
  half8 bring[kRing][NB];
  auto load_b = [&](int s, int step, half8 (&dst)[NB]) __attribute__((always_inline)) {
    s = s < s_last ? s : s_last;
#pragma unroll
    for (int t = 0; t < NB; ++t) dst[t] = *reinterpret_cast<const half8*>(xb[t] + ((size_t)s * 8 + step) * 512);
  };

  load_codes(s_begin);
#pragma unroll
  for (int k = 0; k < kAhead; ++k) load_b(s_begin, k, bring[k]);
  {
    LutCopy<kWgThreads> lc;
    load_luts(tid, lc);
    uint4 t1 = make_uint4(0, 0, 0, 0);
    if (HAS2) t1 = *reinterpret_cast<const uint4*>(kE81h.w[tid]);
    store_luts(lds, tid, lc);
    if (HAS2) lut1[tid] = t1;
  }
  __syncthreads();  // LUTs complete

  floatx4 acc[RT][NB];
  floatx4 acc2[RT][NB];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
      acc2[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

  for (int s = s_begin; s < s_end; ++s) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      cw[i] = nw[i];
      if (HAS2) cw1[i] = nw1[i];
    }
    load_codes(s + 1);
    half8 sgs[NB];  // group sums / 4 of this slice, used after its 8 steps
#pragma unroll
    for (int t = 0; t < NB; ++t) sgs[t] = *reinterpret_cast<const half8*>(sb[t] + (size_t)s * 512);

    auto word = [&](int i, int c) -> uint32_t {
      return c < 2 ? cw[i].x : c < 4 ? cw[i].y : c < 6 ? cw[i].z : cw[i].w;
    };
    // LUT words of step c + 1 are read while the MFMAs of step c run, and the
    // fp16 A fragments of step c + 1 are built between them, so neither the
    // LDS latency nor the decode VALU work stalls the matrix cores.
    uint32_t hv[RT], lv[RT];
    half8 l1[2][RT];
    auto read_luts = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        code_lut_words(word(i, c), c & 1, kDqOffHi, kDqOffLo, hv[i], lv[i]);
        if (HAS2) {
          const uint32_t idx = ((c < 4 ? cw1[i].x : cw1[i].y) >> (8 * (c & 3))) & 0xFFu;
          l1[c & 1][i] = __builtin_bit_cast(half8, lut1[idx]);
        }
      }
    };
    // E8P value +-(k + 1/2); the code's +-1/4 shift is added per slice below
    half8 a[2][RT];
    read_luts(0);
#pragma unroll
    for (int i = 0; i < RT; ++i) a[0][i] = code_operand(hv[i], lv[i]);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      // B fragments of step c + kAhead (into the ring slot step c - 1 freed)
      load_b(c + kAhead < 8 ? s : s + 1, (c + kAhead) & 7, bring[(c + kAhead) % kRing]);
      if (c < 7) read_luts(c + 1);
      const half8(&bf)[NB] = bring[c % kRing];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
#pragma unroll
        for (int t = 0; t < NB; ++t)
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c & 1][i], bf[t], acc[i][t], 0, 0, 0);
        if (HAS2) {
#pragma unroll
          for (int t = 0; t < NB; ++t)
            acc2[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(l1[c & 1][i], bf[t], acc2[i][t], 0, 0, 0);
        }
        if (c < 7) a[(c + 1) & 1][i] = code_operand(hv[i], lv[i]);
      }
    }
    // shifts: +-1 per code (its shift bit) times the group sums / 4 -- one
    // MFMA per tile pair for the slice's 8 steps
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const uint32_t wd[4] = {cw[i].x, cw[i].y, cw[i].z, cw[i].w};
      uint32_t sh[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) sh[k] = 0xBC00BC00u ^ ((wd[k] & 0x10001u) * 0x8000u);
      const half8 so = __builtin_bit_cast(half8, make_uint4(sh[0], sh[1], sh[2], sh[3]));
#pragma unroll
      for (int t = 0; t < NB; ++t)
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(so, sgs[t], acc[i][t], 0, 0, 0);
    }
  }

  // lane (q, r16) holds weight rows 4 q .. 4 q + 3 of tile i for activation
  // row r16 of tile t: four consecutive outputs
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int b = (NB * (WC * ct + w % WC) + t) * 16 + r16;
    if (b >= A.B) continue;
    float* yrow = J.y1p + ((size_t)g * A.B + b) * J.m;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int rb = rb0 + i;
      if (rb >= J.RB) continue;
      floatx4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = HAS2 ? J.s0 * acc[i][t][j] + J.s1 * acc2[i][t][j] : J.s0 * acc[i][t][j];
      *reinterpret_cast<floatx4*>(yrow + rb * 16 + 4 * q) = v;
    }
  }
}

template <bool HAS2, int NB, int WC>
int launch_wg(const WgArgs& A, unsigned grid, hipStream_t stream) {
  static int done = 0;
  if (!done) {
    hipFuncAttributes fa{};
    QS_HIP(hipFuncGetAttributes(&fa, (const void*)wg_kernel<HAS2, NB, WC>));
    QS_REQUIRE(fa.sharedSizeBytes == 0, "wg_kernel: static LDS would move the tables off address 0");
    done = 1;
  }
  hipLaunchKernelGGL((wg_kernel<HAS2, NB, WC>), dim3(grid), dim3(kWgThreads), kWgLds, stream, A);
  QS_LAUNCHED("wg_kernel");
  return QS_OK;
}
template <bool HAS2>
int launch_wg(const WgArgs& A, int cols, unsigned grid, hipStream_t stream) {
  switch (cols) {
    case 2: return launch_wg<HAS2, 2, 1>(A, grid, stream);
    case 3: return launch_wg<HAS2, 3, 1>(A, grid, stream);
    case 4: return launch_wg<HAS2, 4, 1>(A, grid, stream);
    case 6: return launch_wg<HAS2, HAS2 ? 6 : 3, HAS2 ? 1 : 2>(A, grid, stream);
    default: return launch_wg<HAS2, HAS2 ? 8 : 4, HAS2 ? 1 : 2>(A, grid, stream);
  }
}

// ---------------------------------------------------------------------------
// Producer / consumer variant for single-stage batches (use_wp)
// ---------------------------------------------------------------------------
// The wave that feeds the matrix cores should issue nothing but MFMAs and
// their operand loads: VALU work issued by that wave is not hidden behind its
// MFMAs.  So a work-group of 8 waves splits the roles, one of each per SIMD:
// decode waves 4..7 turn the codes of 32 weight rows each into fp16 A
// fragments (E8P value plus the code's +-1/4 shift, exact in fp16) in the
// 32x32x16 MFMA layout, one half slice (128 columns) at a time into a double
// buffer in LDS; MFMA waves 0..3 each multiply all 128 weight rows by 64
// activation rows with v_mfma_f32_32x32x16_f16 (4 x 2 accumulator tiles),
// reading the A fragments from LDS and the B fragments from the
// fragment-major operand through a register ring.  One barrier per half
// slice hands the buffers over.  The tile order, slice groups and partial
// sums are wg_kernel's (with 256 activation rows per work-group).
//
// A fragment (R, k) of a half slice (R: 32-row weight tile, k: 16-column
// step) is 64 lanes x 8 fp16: lane l holds row 32 R + l % 32, columns
// 16 k + 8 (l / 32) .. + 7, i.e. one code.  Code (tile i, lane (q, r16),
// step c = 4 h + cc) of the packed layout holds row 16 i + r16, columns
// 32 c + 8 q: fragment (i / 2, 2 cc + q / 2), lane 16 (i % 2) + r16 + 32 (q % 2).
constexpr int kWpThreads = 512;
constexpr int kWpMfmaWaves = 4;
constexpr int kWpOffA = 32768;                  // after the byte LUTs
constexpr int kWpABuf = 32 * 1024;              // 4 x 8 fragments of 1 KiB
constexpr int kWpLds = kWpOffA + 2 * kWpABuf;
constexpr int kWpRing = 8;                      // B fragment steps in flight per MFMA wave (one half slice)
static_assert(kWpLds <= 160 * 1024, "LDS budget");
static_assert(kWpMfmaWaves * 32 * 528 <= kWpLds, "output staging fits");
typedef float floatx16 __attribute__((ext_vector_type(16)));

__global__ __launch_bounds__(kWpThreads) void wp_kernel(WgArgs A) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // tile order as wg_kernel (XCD-contiguous runs), job after job
  const int T1 = A.nrt * A.nct * A.SGk;
  const int T = A.njobs * T1;
  const int per = (T + 7) >> 3;
  int bid = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (bid >= T) return;
  int jj = 0;
#pragma unroll
  for (int k = 1; k < QS_MAX_GROUP; ++k)
    if (k < A.njobs && bid >= k * T1) jj = k;
  const WpJob& J = A.job[jj];
  bid -= jj * T1;
  const int rt = bid % A.nrt;
  bid /= A.nrt;
  const int ct = bid % A.nct;
  const int g = bid / A.nct;
  const int s_begin = g * A.spg;
  const int s_end = s_begin + A.spg < A.S ? s_begin + A.spg : A.S;
  const int s_last = s_end > s_begin ? s_end - 1 : (A.S - 1);

  // every wave issues its first global loads (code words, B fragments), then
  // copies its share of the LUTs into LDS
  auto build_luts = [&]() {
    LutCopy<kWpThreads> lc;
    load_luts(tid, lc);
    store_luts(lds, tid, lc);
    __syncthreads();  // LUTs complete
  };

  const int nsl = s_end > s_begin ? s_end - s_begin : 0;  // slices of this work-group
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  if (w >= kWpMfmaWaves) {
    // ---------------- decode waves ----------------
    const int d = w - kWpMfmaWaves;  // weight rows 32 d .. 32 d + 31: code tiles 2 d, 2 d + 1
    const int q = lane >> 4, r16 = lane & 15;
    // code words are read once per work-group (nontemporal loads)
    auto words = [&](int ii, int s) -> uint4 {
      int rb = rt * 8 + 2 * d + ii;
      rb = rb < A.RB ? rb : A.RB - 1;  // past the end: the last row block (decoded, never stored)
      s = s < s_last ? s : s_last;
      return ld_nt_u4(reinterpret_cast<const char*>(J.codes0) + ((size_t)rb * A.S + s) * 1024 + 16 * lane);
    };
    // half h of the slice whose code words are c0 / c1 into buffer h
    auto decode_half = [&](auto hc, const uint4& c0, const uint4& c1) {
      constexpr int h = decltype(hc)::value;
      char* buf = lds + kWpOffA + h * kWpABuf;
#pragma unroll
      for (int ii = 0; ii < 2; ++ii) {
        const uint4& cw = ii ? c1 : c0;
        // the two code words of steps 4 h .. 4 h + 3
        const uint32_t wd[2] = {h ? cw.z : cw.x, h ? cw.w : cw.y};
        uint32_t hv[4], lv[4];
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) code_lut_words(wd[cc >> 1], cc & 1, kDqOffHi, kDqOffLo, hv[cc], lv[cc]);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
          const uint32_t sh = (wd[cc >> 1] >> (16 * (cc & 1))) & 1u;  // shift bit: +1/4 set, -1/4 clear
          half8 v = code_operand(hv[cc], lv[cc]);
          v = v + (sh ? (_Float16)0.25f : (_Float16)-0.25f);
          const int kk = 2 * cc + (q >> 1);
          const int l = 16 * ii + r16 + 32 * (q & 1);
          *reinterpret_cast<half8*>(buf + ((d * 8 + kk) * 64 + l) * 16) = v;
        }
      }
    };
    uint4 c0 = words(0, s_begin), c1 = words(1, s_begin);
    build_luts();
    if (nsl > 0) decode_half(H0{}, c0, c1);
    __syncthreads();
    for (int sl = 0; sl < nsl; ++sl) {
      const uint4 n0 = words(0, s_begin + sl + 1), n1 = words(1, s_begin + sl + 1);  // next slice, in flight
      decode_half(H1{}, c0, c1);  // while the MFMA waves take half 0
      __syncthreads();
      c0 = n0;
      c1 = n1;
      if (sl + 1 < nsl) decode_half(H0{}, c0, c1);  // while they take half 1
      __syncthreads();
    }
    return;
  }

  // ---------------- MFMA waves ----------------
  const int nbt = (A.B + 15) >> 4;  // 16-row fragments of the operand
  const int row0 = (kWpMfmaWaves * ct + w) * 64;  // this wave's activation rows row0 .. row0 + 63
  // B fragment (t, slice s, half h, step k): lane l reads activation row row0 + 32 t + l % 32,
  // columns 128 h + 16 k + 8 (l / 32) of the slice; fragment-major operand: 16-row fragment
  // c16, 32-column step st of slice s at ((c16 S + s) 8 + st) 512 halves, lane' = q' 16 + r16'
  // at 8 lane' halves, q' = 2 (k % 2) + l / 32
  const _Float16* xrow[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int r = row0 + 32 * t + (lane & 31);
    int c16 = r >> 4;
    c16 = c16 < nbt ? c16 : nbt - 1;  // rows past the batch: computed, never stored
    xrow[t] = J.x2f + (size_t)c16 * A.S * 8 * 512 + 8 * ((lane >> 5) * 16 + (r & 15));
  }
  // slices past the work-group's last are clamped to it: those loads are in
  // bounds and never used, so every load is unconditional
  auto load_b = [&](int s, int h, int k, half8 (&dst)[2]) {
    s = s < s_last ? s : s_last;
    const size_t off = ((size_t)s * 8 + 4 * h + (k >> 1)) * 512 + 8 * 16 * 2 * (k & 1);
#pragma unroll
    for (int t = 0; t < 2; ++t) dst[t] = *reinterpret_cast<const half8*>(xrow[t] + off);
  };
  auto a_frag = [&](int h, int R, int k) {
    return *reinterpret_cast<const half8*>(lds + kWpOffA + h * kWpABuf + ((R * 8 + k) * 64 + lane) * 16);
  };
  floatx16 acc[4][2];
#pragma unroll
  for (int R = 0; R < 4; ++R)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[R][t] = floatx16{};
  // ring entry k holds step k of the half slice being multiplied; step k of
  // the next half slice (slice sn, half hn) replaces it once its MFMAs are
  // issued, one half slice of MFMAs ahead of its use.  The scheduling
  // barriers keep that order (and the ring in the same registers across the
  // loop): each step reads the next step's A fragments from LDS, issues its
  // 8 MFMAs, then its 2 ring loads.
  half8 ring[kWpRing][2];
  auto mfma_half = [&](auto hc, int sn, int hn) {
    constexpr int h = decltype(hc)::value;
    half8 a[2][4];
#pragma unroll
    for (int R = 0; R < 4; ++R) a[0][R] = a_frag(h, R, 0);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (k < 7) {
#pragma unroll
        for (int R = 0; R < 4; ++R) a[(k + 1) & 1][R] = a_frag(h, R, k + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int R = 0; R < 4; ++R)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[R][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[k & 1][R], ring[k][t], acc[R][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_b(sn, hn, k, ring[k]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const bool wave_on = row0 < A.B;
  if (wave_on) {
#pragma unroll
    for (int k = 0; k < kWpRing; ++k) {
      load_b(s_begin, 0, k, ring[k]);  // in the order the loop issues them
      __builtin_amdgcn_sched_barrier(0);
    }
    build_luts();
    __syncthreads();  // the first half slice's fragments are in buffer 0
    for (int sl = 0; sl < nsl; ++sl) {
      const int s = s_begin + sl;
      mfma_half(H0{}, s, 1);
      __syncthreads();  // buffer 0 free; half 1 complete
      mfma_half(H1{}, s + 1, 0);
      __syncthreads();  // buffer 1 free; the next slice's half 0 complete
    }
  } else {
    // no activation rows: only the barriers that hand the buffers over
    build_luts();
    __syncthreads();
    for (int sl = 0; sl < nsl; ++sl) {
      __syncthreads();
      __syncthreads();
    }
    return;
  }
  // lane l, accumulator v of tile (R, t): weight row 32 R + 8 (v / 4) + 4 (l / 32) + v % 4,
  // activation row row0 + 32 t + l % 32; four consecutive weight rows per float4.
  // The tiles go out through LDS (each MFMA wave its own 32 x 528-byte area
  // in the LUT and fragment space, free after the last barrier), so that each
  // store instruction writes two activation rows' 512 contiguous bytes
  // instead of 32 rows' 32 bytes (2 % of the 512-row step).
  char* stg = lds + w * (32 * 528);
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int R = 0; R < 4; ++R)
#pragma unroll
      for (int vg = 0; vg < 4; ++vg) {
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = J.s0 * acc[R][t][4 * vg + e];
        *reinterpret_cast<floatx4*>(stg + (lane & 31) * 528 + (32 * R + 8 * vg + 4 * (lane >> 5)) * 4) = v;
      }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
    const int row = rt * 128 + 4 * (lane & 31);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int r = 2 * k + (lane >> 5);
      const int b = row0 + 32 * t + r;
      const floatx4 v = *reinterpret_cast<const floatx4*>(stg + r * 528 + (lane & 31) * 16);
      if (b < A.B && row < A.m) *reinterpret_cast<floatx4*>(J.y1p + ((size_t)g * A.B + b) * A.m + row) = v;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
  }
}

int launch_wp(const WgArgs& A, unsigned grid, hipStream_t stream) {
  static int done = 0;
  if (!done) {
    hipFuncAttributes fa{};
    QS_HIP(hipFuncGetAttributes(&fa, (const void*)wp_kernel));
    QS_REQUIRE(fa.sharedSizeBytes == 0, "wp_kernel must not use static LDS");
    QS_HIP(hipFuncSetAttribute((const void*)wp_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kWpLds));
    done = 1;
  }
  hipLaunchKernelGGL(wp_kernel, dim3(grid), dim3(kWpThreads), kWpLds, stream, A);
  QS_LAUNCHED("wp_kernel");
  return QS_OK;
}

}  // namespace

// Work-group tiles of one linear (128 weight rows by the work-group's activation rows).
static int64_t wide_tiles(int64_t m, int64_t n, int64_t B, bool has2) {
  const int64_t cols = use_wp(m, n, B, has2) ? 256 : 16 * wg_cols(B);
  return ((m / 16 + kWgRowTiles - 1) / kWgRowTiles) * ((B + cols - 1) / cols);
}
static int groups_within(int64_t tiles, int64_t n, int64_t limit) {
  const int64_t S = n / 256;
  int64_t g = 1;
  while (g < kWideMaxGroups && g < S && tiles * (g + 1) <= limit) ++g;
  return (int)g;
}

int wide_splits(int64_t m, int64_t n, int64_t B, int ncu, bool has2) {
  const int64_t tiles = wide_tiles(m, n, B, has2);
  int g = groups_within(tiles, n, ncu);
  // up to 128 rows a second work-group per CU, while the partial sums stay few;
  // with one stage only where no CU then has more slices to go through (8192 x
  // 5120, 32 rows: five slices each in 4 groups 25.6 us, three and two groups per
  // CU in 8 29.9; 18944 x 3584: fourteen in one group, five in 3 36.9)
  if (B <= 16 * kWgMaxCols && !use_wp(m, n, B, has2)) {
    const int64_t S = n / 256;
    int64_t g2 = groups_within(tiles, n, 2 * ncu);
    const int64_t most = kWgPartialBytes / (B * m * 4);
    if (g2 > most) g2 = most;
    if (g2 > g && (has2 || (tiles * g2 + ncu - 1) / ncu * ((S + g2 - 1) / g2) <= (S + g - 1) / g)) g = (int)g2;
  }
  return g;
}

size_t wide_partial_bytes(int64_t m, int64_t n, int64_t B, int ncu) {
  const int64_t row = m * 4, nrt = wide_tiles(m, n, 1, false), first = B < 16 * kWgMaxCols ? B : 16 * kWgMaxCols;
  // up to 128 rows: one column of tiles, whatever the rows
  size_t most = (size_t)(groups_within(nrt, n, ncu) * first * row), two = (size_t)(groups_within(nrt, n, 2 * ncu) * first * row);
  if (two > (size_t)kWgPartialBytes) two = (size_t)kWgPartialBytes;
  if (two > most) most = two;
  // beyond: the most rows of each count of groups (a second stage never has more groups than one stage)
  for (int64_t g = 1; g <= kWideMaxGroups && g <= n / 256 && B > first; ++g) {
    const int64_t rows = g == 1 ? B : ncu / (g * nrt) * 256;
    const size_t b = (size_t)(g * (rows < B ? rows : B) * row);
    if (rows > first && b > most) most = b;
  }
  return most;
}

int wide_group_splits(int64_t m, int64_t n, int64_t B, int count, int ncu) {
  if (count < 2 || B <= 16 * kWgMaxCols) return 0;
  const int64_t tiles = wide_tiles(m, n, B, false) * count;
  return tiles > ncu ? 0 : groups_within(tiles, n, ncu);
}

namespace {
int wide_args(const WideMfma* G, int count, WgArgs& A, int64_t& wgs) {
  const bool has2 = G[0].codes1 != nullptr;
  const int cols = use_wp(G[0]) ? 256 : 16 * wg_cols(G[0].B);
  A.m = (int)G[0].m;
  A.B = G[0].B;
  A.S = (int)(G[0].n / 256);
  A.RB = (int)(G[0].m / 16);
  A.nrt = (A.RB + kWgRowTiles - 1) / kWgRowTiles;
  A.nct = (G[0].B + cols - 1) / cols;
  A.SGk = G[0].SGk;
  A.spg = (A.S + A.SGk - 1) / A.SGk;
  A.njobs = count;
  wgs = 0;
  for (int j = 0; j < count; ++j) {
    const WideMfma& F = G[j];
    QS_REQUIRE(F.m % 16 == 0 && F.n % 256 == 0 && F.B >= 1, "wide GEMM: m %% 16, n %% 256");
    QS_REQUIRE(F.SGk >= 1 && F.SGk <= kWideMaxGroups, "wide GEMM: 1..%d slice groups", kWideMaxGroups);
    QS_REQUIRE(F.m * F.n / 4 < ((int64_t)1 << 40), "wide GEMM: codes too large");
    QS_REQUIRE(F.n == G[0].n && F.B == A.B && (F.codes1 != nullptr) == has2 && use_wp(F) == use_wp(G[0]),
               "wide GEMM: linears of one operand width and kernel");
    const int RB = (int)(F.m / 16), nrt = (RB + kWgRowTiles - 1) / kWgRowTiles;
    const int64_t tiles = (int64_t)nrt * A.nct * F.SGk;
    A.job[j] = WpJob{static_cast<const uint16_t*>(F.codes0), F.x2f, F.y1p, F.s0, static_cast<const uint8_t*>(F.codes1),
                     F.sgf, F.s1, (int)F.m, RB, nrt, F.SGk, (A.S + F.SGk - 1) / F.SGk, (int)wgs, (int)tiles};
    wgs += (tiles + 7) / 8 * 8;
    QS_REQUIRE(wgs < ((int64_t)1 << 30), "wide GEMM: grid too large");
  }
  return QS_OK;
}
}  // namespace

int launch_linear_wide(const WideMfma* G, int count, hipStream_t stream) {
  QS_REQUIRE(count >= 1 && count <= QS_MAX_GROUP, "wide GEMM: 1..%d linears", QS_MAX_GROUP);
  WgArgs A{};
  int64_t wgs = 0;
  const int rc = wide_args(G, count, A, wgs);
  if (rc) return rc;
  const bool has2 = G[0].codes1 != nullptr;
  if (use_wp(G[0])) {
    for (int j = 1; j < count; ++j)
      QS_REQUIRE(G[j].m == G[0].m && G[j].SGk == G[0].SGk, "wide GEMM: wp_kernel takes linears of one shape");
    // one run of tiles over the jobs, which are alike
    const int64_t tiles = (int64_t)count * A.job[0].tiles;
    return launch_wp(A, (unsigned)((tiles + 7) / 8 * 8), stream);
  }
  const unsigned grid = (unsigned)wgs;
  return has2 ? launch_wg<true>(A, wg_cols(A.B), grid, stream) : launch_wg<false>(A, wg_cols(A.B), grid, stream);
}

bool wide_shares_launch(const WideMfma& a, const WideMfma& b) {
  if (use_wp(a) || use_wp(b)) return use_wp(a) && use_wp(b) && a.m == b.m && a.B <= 16 * kWgMaxCols;
  return true;
}

}  // namespace qs
