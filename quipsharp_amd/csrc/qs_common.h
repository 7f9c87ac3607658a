// Shared definitions for the gfx950 QuIP# kernels: status plumbing, the fp16
// form of the codebook tables (qs_tables.h), and small device helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "../../include/quipsharp_hip.h"
#include "qs_tables.h"

namespace qs {

// ----------------------------------------------------------------------------
// status
// ----------------------------------------------------------------------------
void set_error(const char* fmt, ...);
int hip_status(hipError_t e, const char* what);

#define QS_REQUIRE(cond, ...)                                 \
  do {                                                        \
    if (!(cond)) {                                            \
      ::qs::set_error(__VA_ARGS__);                           \
      return QS_ERR_INVALID;                                  \
    }                                                         \
  } while (0)

#define QS_SUPPORTED(cond, ...)                               \
  do {                                                        \
    if (!(cond)) {                                            \
      ::qs::set_error(__VA_ARGS__);                           \
      return QS_ERR_UNSUPPORTED;                              \
    }                                                         \
  } while (0)

#define QS_HIP(expr)                                          \
  do {                                                        \
    hipError_t e_ = (expr);                                   \
    if (e_ != hipSuccess) return ::qs::hip_status(e_, #expr); \
  } while (0)

#define QS_LAUNCHED(name)                                     \
  do {                                                        \
    hipError_t e_ = hipGetLastError();                        \
    if (e_ != hipSuccess) return ::qs::hip_status(e_, name);  \
  } while (0)

inline hipStream_t as_stream(qs_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// fp16 bit pattern of a float that fp16 represents exactly (zero or normal).
constexpr uint16_t f16_bits_exact(float f) {
  const uint16_t sign = f < 0.0f ? 0x8000 : 0;
  float a = f < 0.0f ? -f : f;
  if (a == 0.0f) return sign;
  int e = 0;
  while (a >= 2.0f) a *= 0.5f, ++e;
  while (a < 1.0f) a *= 2.0f, --e;
  return (uint16_t)(sign | ((e + 15) << 10) | (int)((a - 1.0f) * 1024.0f));
}

// A Table8 as fp16 pairs: w[r][i] holds elements 2i (low half) and 2i + 1.
struct Table8h {
  uint32_t w[256][4];
};

constexpr Table8h pack_table_f16(const Table8& t) {
  Table8h h{};
  for (int r = 0; r < 256; ++r)
    for (int i = 0; i < 4; ++i)
      h.w[r][i] = (uint32_t)f16_bits_exact(t.v[r][2 * i]) | ((uint32_t)f16_bits_exact(t.v[r][2 * i + 1]) << 16);
  return h;
}

// ----------------------------------------------------------------------------
// device helpers
// ----------------------------------------------------------------------------
__device__ __forceinline__ float load_as_float(const void* p, int dtype, int64_t i) {
  if (dtype == QS_DTYPE_F32) return static_cast<const float*>(p)[i];
  if (dtype == QS_DTYPE_F16) return (float)static_cast<const _Float16*>(p)[i];
  uint32_t b = (uint32_t) static_cast<const uint16_t*>(p)[i] << 16;  // bf16
  return __uint_as_float(b);
}

// Round-to-nearest-even fp32 -> bf16, NaN kept quiet: (u + 0x7FFF + lsb) >> 16
// of the bits u, and (u >> 16) | 0x40 for a NaN.  gfx950's conversion
// instruction (v_cvt_pk_bf16_f32) gives exactly these bits for every one of
// the 2^32 fp32 inputs (checked exhaustively on the device), in one
// instruction for two values instead of six or seven integer operations per
// value.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint16_t f32_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
// Two values: lo in bits 0-15, hi in bits 16-31.
__device__ __forceinline__ uint32_t f32x2_to_bf16x2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){lo, hi}, bf16x2_t));
}

__device__ __forceinline__ void store_from_float(void* p, int dtype, int64_t i, float v) {
  if (dtype == QS_DTYPE_F32) static_cast<float*>(p)[i] = v;
  else if (dtype == QS_DTYPE_F16) static_cast<_Float16*>(p)[i] = (_Float16)v;
  else static_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
}

inline int dtype_bytes(int dtype) { return dtype == QS_DTYPE_F32 ? 4 : 2; }

}  // namespace qs
