// kv800_common.h -- constants, bit-exact scalar helpers and host-side error plumbing shared by the gfx950 kernels
// of the 800h path. Layout constants follow kv800.py:32-34; the fp8 / bf16 helpers follow the semantics the
// reference gets from torch (fp8 e4m3fn encode: round to nearest even, |x| > 464 -> 0x7F NaN; bf16: round to nearest
// even) and its kernels (fp8 decode without NaN handling, kv800_sycl.sycl:41-45).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kv800 {

constexpr int BLK = 256;      // tokens per quantized sub-block
constexpr int LAG = 128;      // newest tokens that always stay exact
constexpr int NSINK = 4;
constexpr int SUB = 51200;    // bytes per sub-block
constexpr int KC_O = 0, VB_O = 32768, VLO_O = 49152, VSC_O = 49664, KLO_O = 50176, KSC_O = 50688;

// ---------------------------------------------------------------- device scalar helpers
__device__ __forceinline__ float bf2f(uint32_t b16) { return __uint_as_float(b16 << 16); }
__device__ __forceinline__ float bf2f_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ float bf2f_lo(uint32_t w) { return __uint_as_float(w << 16); }

// float -> bf16 bits, round to nearest even (finite values)
__device__ __forceinline__ uint32_t f2bf(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bfround(float f) { return __uint_as_float(f2bf(f) << 16); }

// fp8 e4m3fn byte -> float, exact; no NaN handling (the scales the quantizer writes are finite for finite input): the
// hardware conversion, with the two NaN bytes read as the +-480 that their bits spell
__device__ __forceinline__ float f8d(uint32_t b) {
  const float r = __builtin_amdgcn_cvt_f32_fp8((int)b, 0);
  return r == r ? r : __uint_as_float(0x43F00000u | ((b & 0x80u) << 24));
}

// float -> fp8 e4m3fn byte with torch's .to(float8_e4m3fn) semantics (round to nearest even on the e4m3 grid,
// results past 448 and inf / NaN -> 0x7F with the sign bit). The hardware conversion does that for every float but NaN
// (compared over all 2^32 against the bit arithmetic), whose sign it drops.
__device__ __forceinline__ uint32_t f8e(float f) {
  const uint32_t r = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f, f, 0, false) & 0xFFu;
  return f == f ? r : ((__float_as_uint(f) >> 24) & 0x80u) | 0x7Fu;
}

__device__ __forceinline__ float clamp_min_1e8(float a) { return a < 1e-8f ? 1e-8f : a; }

// v_min_f32 / v_max_f32 / v_max3_f32 as the bare instructions. fminf and fmaxf first quiet signalling NaNs of operands
// whose origin the compiler cannot see (cross-lane moves, selects, inline assembly); arithmetic never produces a
// signalling NaN, so for arithmetic results and copies of them the quieting is dead work. The operands must be written
// by ordinary VALU or memory instructions, not straight by an MFMA (no hazard wait states are inserted for inline
// assembly reading an MFMA result).
__device__ __forceinline__ float vmin(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

}  // namespace kv800

// ---------------------------------------------------------------- host error plumbing
namespace kv800 {
void set_error(const char* fmt, ...);
int check_launch(const char* what);
}  // namespace kv800

#define KV800_REQUIRE(cond, ...)                 \
  do {                                           \
    if (!(cond)) {                               \
      ::kv800::set_error(__VA_ARGS__);           \
      return KV800_EINVAL;                       \
    }                                            \
  } while (0)
