// kv800_quant.hip -- 800h quantize / paged flush / dequantize kernels for gfx950 and their C-ABI entry points.
//
// Reference semantics: kv800.py:56-76 (quantize_blocks), kv800.py:79-92 (dequantize_blocks), the flush plan of
// vllm_attn.py:297-317 and the PagedStore flush loop kv800.py:433-440. Output bytes are bit-identical to the
// reference quantizer on CPU torch:
//   * K: per (head, channel) min / max over the 256 tokens; lo8 = fp8(lo), sc8 = fp8(max((hi - lo) / 3, 1e-8));
//     code = clamp(rne((x - f32(lo8)) / max(f32(sc8), 1e-8)), 0, 3) with IEEE division;
//   * V: y = f32(v) @ H per (token, head) as the sequential fma chain over k = 0..127 that torch-CPU's sgemm
//     evaluates for this shape, then per (token, 2-head group) lo8 / sc8 and 1-bit codes the same way.
// Workgroups of 8 waves quantize one 256-token sub-block: its K per head, its V per token range; the input is
// gathered straight from the exact pages (paged flush) or from dense (M, 256, 4, 128) tensors, and the 51,200-byte
// result is written through the quant block table, so a flush is one launch with no host loop and no intermediate
// copies.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "kv800_common.h"
#include "../../include/kv800_hip.h"

namespace kv800 {

static thread_local char g_err[512];

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
}

int check_launch(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: %s", what, hipGetErrorString(e));
    return KV800_EHIP;
  }
  return KV800_OK;
}

namespace {

constexpr int QTHREADS = 512;    // 8 waves per sub-block, 32 tokens each
constexpr int QWPS = 4;          // waves per SIMD the throughput kernels are built for (two workgroups per CU)
constexpr int QW = QTHREADS / 64;

// ---------------------------------------------------------------- token-row sources
struct DenseSrc {   // (M, 256, 4, 128) contiguous K and V
  const uint16_t* k;
  const uint16_t* v;
  int64_t m;
  __device__ void prepare(int64_t*) {}
  __device__ const uint16_t* krow(int t, int h) const { return k + ((m * BLK + t) * 4 + h) * 128; }
  __device__ const uint16_t* vrow(int t, int h) const { return v + ((m * BLK + t) * 4 + h) * 128; }
};

struct PagedSrc {   // exact pages: K of (position p, head h) at eoff[r, p / ebs] + h e_hs + (p % ebs) e_ts; V at + e_v
  const uint16_t* ep;
  const int64_t* et;   // this row's page table
  int64_t ebs, e_hs, e_ts, e_v, p0;
  const int64_t* rowoff = nullptr;   // LDS: element offset of token t's head-0 K row, t < 256
  // Element offset of token t's head-0 K row. The division is a 32-bit one (20 instructions against 150) unless the
  // positions or the page size need more (a scalar branch).
  __device__ __forceinline__ int64_t row(int t) const {
    const int64_t p = p0 + t;
    if (((p0 + BLK) | ebs) >> 32) return et[p / ebs] + (p % ebs) * e_ts;
    const uint32_t pg = (uint32_t)p / (uint32_t)ebs;
    return et[pg] + (int64_t)((uint32_t)p - pg * (uint32_t)ebs) * e_ts;
  }
  // K pass: one page-table lookup per token for the whole workgroup (every thread must call it). A V lane reads one
  // row per group of tokens and looks it up itself, without the barrier.
  __device__ void prepare(int64_t* tab) {
    for (int t = threadIdx.x; t < BLK; t += blockDim.x) tab[t] = row(t);
    __syncthreads();
    rowoff = tab;
  }
  __device__ const uint16_t* krow(int t, int h) const { return ep + rowoff[t] + h * e_hs; }
  __device__ const uint16_t* vrow(int t, int h) const { return ep + row(t) + h * e_hs + e_v; }
};

// K code clamp(rne(fl(d / den)), 0, 3) without the division. fl(q) > 1/2 <=> d > den / 2 (a float above den / 2 is
// at least an ulp of den / 2 above it); fl(q) >= 3/2 <=> q >= 3/2 - 2^-24 and fl(q) > 5/2 <=> q > 5/2 + 2^-23 (the
// midpoints round to the even 3/2 and 5/2). Those two are decided on r = fl(d - t den) (one fma): near the threshold
// d - t den is a small multiple of 2^-24 times den's power of two, hence exact, and a second fma adds the margin
// den 2^-24 (den 2^-23) with the sign of the exact sum; far from it |r| dwarfs the margin. den >= 1e-8 is normal; a
// NaN d or den gives code 0, as the clamp of a NaN quotient does.
__device__ __forceinline__ uint32_t kcode(float d, float den) {
  const bool c1 = d > den * 0.5f;
  const bool c2 = __builtin_fmaf(den, 0x1p-24f, __builtin_fmaf(-den, 1.5f, d)) >= 0.f;
  const bool c3 = __builtin_fmaf(-den, 0x1p-23f, __builtin_fmaf(-den, 2.5f, d)) > 0.f;
  return (uint32_t)c1 + (uint32_t)c2 + (uint32_t)c3;
}

// x of the lane `n` places further round its 16-lane row (DPP row_ror)
__device__ __forceinline__ uint32_t row_ror(uint32_t x, int n) {
  return n == 4 ? (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x124, 0xF, 0xF, false)
                : (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x128, 0xF, 0xF, false);
}

// bf16 pairs as ordered 16-bit keys: the bits of a non-negative value as they are, a negative one's magnitude bits
// flipped, so that signed 16-bit compares order the values (-0 below +0) and one packed instruction takes two of them.
// The map is its own inverse. NaN keys lie outside [KEY_NINF, KEY_INF].
typedef short s2 __attribute__((ext_vector_type(2)));
constexpr int KEY_INF = 0x7F80, KEY_NINF = -32641;
__device__ __forceinline__ uint32_t as_u(s2 x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ s2 as_s2(uint32_t x) { return __builtin_bit_cast(s2, x); }
__device__ __forceinline__ s2 bf_keys(uint32_t w) {
  const s2 x = as_s2(w);
  return as_s2(w ^ (as_u(x >> (short)15) & 0x7FFF7FFFu));
}
__device__ __forceinline__ float key_float(int k) {   // the value of one key
  return bf2f((uint32_t)(uint16_t)(k ^ ((k >> 15) & 0x7FFF)));
}
// min / max over the lanes l, l ^ 16, l ^ 32, l ^ 48
template <bool MAX>
__device__ __forceinline__ s2 reduce4rows(s2 x) {
  auto r = __builtin_amdgcn_permlane16_swap(as_u(x), as_u(x), false, false);
  x = MAX ? __builtin_elementwise_max(as_s2(r[0]), as_s2(r[1])) : __builtin_elementwise_min(as_s2(r[0]), as_s2(r[1]));
  r = __builtin_amdgcn_permlane32_swap(as_u(x), as_u(x), false, false);
  return MAX ? __builtin_elementwise_max(as_s2(r[0]), as_s2(r[1])) : __builtin_elementwise_min(as_s2(r[0]), as_s2(r[1]));
}

// K codes and scales of one head hh of one sub-block, its 256 token rows read once: lane (g, c) of wave w holds the
// 8 channels 8 c .. 8 c + 7 of the tokens 32 i + 4 w + g (i = 0..7) as key pairs in registers through both passes (min /
// max, then codes). Min / max across the 4 token rows of a wave by permlane swaps, across the 8 waves through LDS.
// d = fl(x - lo) never decreases with x and the code never with d, so a channel's code is the number of its three
// thresholds T_c (the smallest bf16 value of code >= c) that x reaches: thread 128 c + channel computes T_c and settles
// it with kcode itself. An element then costs 2 VALU instructions for min / max and 4 for its code, against 24 with the
// arithmetic per element, and they matter because the V workgroups' fp32 MFMA and VALU share the part's FMA units.
// A workgroup that holds a NaN takes the arithmetic per element (min / max skip NaN, its code is 0).
struct QuantLds {
  s2 red_min[QW][64], red_max[QW][64];   // per wave, channel pairs
  short thr[3][128];                     // T_c - 1
  float lo[128], den[128];
};
template <typename Src>
__device__ void quantize_k(const Src& src, uint8_t* __restrict__ out, char* lds, int hh) {
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 4, c16 = lane & 15, c0 = 8 * c16;
  QuantLds& S = *reinterpret_cast<QuantLds*>(lds);
  constexpr int NT = BLK / 32;   // tokens per lane
  s2 kx[NT][4];
  {
    uint4 raw[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) raw[i] = *reinterpret_cast<const uint4*>(src.krow(32 * i + 4 * w + g, hh) + c0);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      kx[i][0] = bf_keys(raw[i].x); kx[i][1] = bf_keys(raw[i].y);
      kx[i][2] = bf_keys(raw[i].z); kx[i][3] = bf_keys(raw[i].w);
    }
  }
  bool nan = false;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    s2 mn = kx[0][d], mx = kx[0][d];
#pragma unroll
    for (int i = 1; i < NT; ++i) {
      mn = __builtin_elementwise_min(mn, kx[i][d]);
      mx = __builtin_elementwise_max(mx, kx[i][d]);
    }
    mn = reduce4rows<false>(mn);
    mx = reduce4rows<true>(mx);
    nan |= mn.x < KEY_NINF || mn.y < KEY_NINF || mx.x > KEY_INF || mx.y > KEY_INF;
    if (g == 0) { S.red_min[w][4 * c16 + d] = mn; S.red_max[w][4 * c16 + d] = mx; }
  }
  nan = __syncthreads_or(nan);   // uniform over the workgroup
  if (nan) {                     // min / max of the values that are no NaN (none: +inf, -inf), as fminf / fmaxf give
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      s2 mn = {(short)KEY_INF, (short)KEY_INF}, mx = {(short)KEY_NINF, (short)KEY_NINF};
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const s2 k = kx[i][d];
        if (k.x >= KEY_NINF && k.x <= KEY_INF) { mn.x = min(mn.x, k.x); mx.x = max(mx.x, k.x); }
        if (k.y >= KEY_NINF && k.y <= KEY_INF) { mn.y = min(mn.y, k.y); mx.y = max(mx.y, k.y); }
      }
      mn = reduce4rows<false>(mn);
      mx = reduce4rows<true>(mx);
      if (g == 0) { S.red_min[w][4 * c16 + d] = mn; S.red_max[w][4 * c16 + d] = mx; }
    }
    __syncthreads();
  }
  {
    const int col = tid & 127, c = tid >> 7;
    int kmn = reinterpret_cast<const short*>(S.red_min[0])[col], kmx = reinterpret_cast<const short*>(S.red_max[0])[col];
#pragma unroll
    for (int ww = 1; ww < QW; ++ww) {
      kmn = min(kmn, (int)reinterpret_cast<const short*>(S.red_min[ww])[col]);
      kmx = max(kmx, (int)reinterpret_cast<const short*>(S.red_max[ww])[col]);
    }
    const float lo = key_float(kmn), hi = key_float(kmx);
    const uint32_t lo8 = f8e(lo);
    const uint32_t sc8 = f8e(clamp_min_1e8(__fdiv_rn(__fsub_rn(hi, lo), 3.0f)));
    const float lof = f8d(lo8), den = clamp_min_1e8(f8d(sc8));
    if (c == 0) {   // uniform over the wave
      out[KLO_O + hh * 128 + col] = (uint8_t)lo8;
      out[KSC_O + hh * 128 + col] = (uint8_t)sc8;
      S.lo[col] = lof;
      S.den[col] = den;
    } else {
      auto reaches = [&](int k) { return kcode(__fsub_rn(key_float(k), lof), den) >= (uint32_t)c; };
      // D: the smallest d of code >= c (an ulp or two about (c - 1/2) den, which is exact); then x with x - lo at the
      // rounding midpoint below D, exact or to an fp32 rounding of x itself
      const uint32_t base = __float_as_uint(((float)c - 0.5f) * den);
      uint32_t db = base - 1;
#pragma unroll
      for (int k = -1; k < 2; ++k) db += kcode(__uint_as_float(base + k), den) < (uint32_t)c;
      const float D = __uint_as_float(db);
      const float x0 = __fsub_rn(__fadd_rn(lof, D), 0.5f * __fsub_rn(D, __uint_as_float(db - 1)));
      const int k0 = as_s2(as_u(bf_keys(f2bf(x0)))).x;
      int a = k0 - 1, b = k0 + 1;   // T_c in (a, b], or anywhere when either end says otherwise
      if (reaches(a)) a = KEY_NINF - 1;
      if (!reaches(b)) b = KEY_INF + 1;
      while (b - a > 1) {
        const int mid = (a + b) >> 1;
        if (reaches(mid)) b = mid; else a = mid;
      }
      S.thr[c - 1][col] = (short)(b - 1);
    }
  }
  __syncthreads();
  const int p = c16 >> 2, q = c16 & 3;   // plane of these 8 channels, byte quarter 8q .. 8q + 7
  auto store = [&](int i, uint32_t d0, uint32_t d1) {
    // the 4 planes of these bytes sit in the lanes 4, 8, 12 apart within the 16-lane row
    d0 |= row_ror(d0, 4); d1 |= row_ror(d1, 4);
    d0 |= row_ror(d0, 8); d1 |= row_ror(d1, 8);
    if (p == 0) {
      const int t = 32 * i + 4 * w + g;
      *reinterpret_cast<uint2*>(out + KC_O + (t * 4 + hh) * 32 + 8 * q) = make_uint2(d0, d1);
    }
  };
  if (nan) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      uint32_t dw[2] = {0, 0};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = (e & 1) ? kx[i][e >> 1].y : kx[i][e >> 1].x;
        dw[e >> 2] |= kcode(__fsub_rn(key_float(k), S.lo[c0 + e]), S.den[c0 + e]) << (2 * p + 8 * (e & 3));
      }
      store(i, dw[0], dw[1]);
    }
    return;
  }
  s2 th[3][4];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const uint4 t = *reinterpret_cast<const uint4*>(&S.thr[c][c0]);
    th[c][0] = as_s2(t.x); th[c][1] = as_s2(t.y); th[c][2] = as_s2(t.z); th[c][3] = as_s2(t.w);
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    __builtin_amdgcn_sched_barrier(0);   // one token row at a time
    // sign bits: u_c = x >= T_c; the code's high bit is u_2, its low bit u_3 where u_2, else u_1
    uint32_t dw[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      uint32_t lb[2], hb[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const s2 x = kx[i][2 * d + k];
        const uint32_t u1 = as_u(__builtin_elementwise_sub_sat(th[0][2 * d + k], x));
        const uint32_t u2 = as_u(__builtin_elementwise_sub_sat(th[1][2 * d + k], x));
        const uint32_t u3 = as_u(__builtin_elementwise_sub_sat(th[2][2 * d + k], x));
        lb[k] = (u2 & u3) | (~u2 & u1);
        hb[k] = u2;
      }
      // the 4 channels' sign bytes side by side, then code bits 7 and 6 of each byte down to the plane's two bits
      const uint32_t lw = __builtin_amdgcn_perm(lb[1], lb[0], 0x07050301u);
      const uint32_t hw = __builtin_amdgcn_perm(hb[1], hb[0], 0x07050301u);
      dw[d] = (((hw & 0x80808080u) | ((lw >> 1) & 0x7F7F7F7Fu)) & 0xC0C0C0C0u) >> (6 - 2 * p);
    }
    store(i, dw[0], dw[1]);
  }
}

// ---------------------------------------------------------------- V path
// One lane owns 8 dims of one head row: lane = 16 hh + jj computes head hh's dims jj + 16 i (i = 0..7), which are
// exactly the 8 bits of the row's code byte jj. For k = 16 m + kl (m, i < 8, kl < 16),
// H[k][jj + 16 i] = H[kl][jj] (-1)^popcount(m & i), so the lane keeps the 16 values H[kl][jj] and every other sign is
// a compile-time negation.
__device__ __forceinline__ void hadamard_low(float (&hl)[16], int jj) {
  const float c = __uint_as_float(0x3DB504F3u);   // fp32(1 / sqrt(128))
#pragma unroll
  for (int kl = 0; kl < 16; ++kl) hl[kl] = (__builtin_popcount(kl & jj) & 1) ? -c : c;
}

__device__ __forceinline__ constexpr bool hneg(int m, int i) { return __builtin_popcount(m & i) & 1; }

// y[i] = sum_k x[k] H[k][jj + 16 i], each output by torch-CPU's sequential fma chain over k = 0..127. Outputs whose
// signs agree on a prefix of k share its partial sums: one chain for k < 16, two for k < 32 (by i & 1), four for
// k < 64 (by i & 3), eight after (688 fmas for the 8 outputs instead of 1024). x (the lane's staged row) is read one
// float4 at a time, two reads ahead of their use.
__device__ __forceinline__ void hadamard_row8(const float* x, const float (&hl)[16], float (&y)[8]) {
  float4 buf[3];
  buf[0] = *reinterpret_cast<const float4*>(x);
  buf[1] = *reinterpret_cast<const float4*>(x + 4);
  float ch[8];
  ch[0] = 0.f;
#pragma unroll
  for (int g = 0; g < 32; ++g) {   // k = 4 g .. 4 g + 3
    if (g + 2 < 32) buf[(g + 2) % 3] = *reinterpret_cast<const float4*>(x + 4 * (g + 2));
    const float4 v = buf[g % 3];
    const float xv[4] = {v.x, v.y, v.z, v.w};
    const int m = g >> 2;   // k >> 4
    if (g == 4) ch[1] = ch[0];
    if (g == 8) { ch[2] = ch[0]; ch[3] = ch[1]; }
    if (g == 16) { ch[4] = ch[0]; ch[5] = ch[1]; ch[6] = ch[2]; ch[7] = ch[3]; }
    const int nch = m == 0 ? 1 : m == 1 ? 2 : m < 4 ? 4 : 8;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float h = hl[(4 * g + e) & 15];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i < nch) ch[i] = __builtin_fmaf(xv[e], hneg(m, i) ? -h : h, ch[i]);
    }
    // the group's fmas stay before this point and the next group's reads after it: two reads ahead, no further (the
    // live chains only; the last group's results stay plain fma results)
    if (nch == 1) asm volatile("" : "+v"(ch[0])::"memory");
    else if (nch == 2) asm volatile("" : "+v"(ch[0]), "+v"(ch[1])::"memory");
    else if (nch == 4) asm volatile("" : "+v"(ch[0]), "+v"(ch[1]), "+v"(ch[2]), "+v"(ch[3])::"memory");
    else if (g < 31)
      asm volatile("" : "+v"(ch[0]), "+v"(ch[1]), "+v"(ch[2]), "+v"(ch[3]), "+v"(ch[4]), "+v"(ch[5]), "+v"(ch[6]),
                   "+v"(ch[7])::"memory");
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = ch[i];
}

// min(x, x of a DPP partner lane); s_nop 1 gives the two wait states a DPP read of a just-written VGPR needs
#define KV800_MIN_DPP(x, ctrl)                                                                                \
  ({                                                                                                          \
    float r_;                                                                                                 \
    asm("s_nop 1\n\tv_min_f32_dpp %0, %1, %1 " ctrl " row_mask:0xf bank_mask:0xf" : "=v"(r_) : "v"(x));     \
    r_;                                                                                                       \
  })

// min over each 16-lane row, the result in every lane of the row (quad swaps, then half-row and row mirrors)
__device__ __forceinline__ float row_min16(float x) {
  x = KV800_MIN_DPP(x, "quad_perm:[1,0,3,2]");
  x = KV800_MIN_DPP(x, "quad_perm:[2,3,0,1]");
  x = KV800_MIN_DPP(x, "row_half_mirror");
  x = KV800_MIN_DPP(x, "row_mirror");
  return x;
}

// Scales of one token's V rows from the 8 chain outputs y each lane holds (lane 16 hh + jj: row hh): per 2-head group g
// (lanes 32 g .. 32 g + 31, 256 outputs) the min and max through a 16-row swap -- afterwards rows 0 / 1 hold group
// 0's min / -max partials (lanes l, l + 16 combined), rows 2 / 3 group 1's -- and DPP row reductions; lanes q = 0..3
// then encode lo (q even) or max(hi - lo, 1e-8) (q odd) of group q >> 1 in one pass. b8 is that byte (lanes 0..3);
// lof, scf are the lane's group's decoded lo and scale, den = max(scf, 1e-8) the quantizer's divisor.
struct VScales { uint32_t b8; float lof, scf, den; };
__device__ __forceinline__ VScales v_scales(const float (&y)[8], int lane) {
  const int q = lane & 3, g = lane >> 5;
  const float mn = fminf(fminf(fminf(y[0], y[1]), fminf(y[2], y[3])), fminf(fminf(y[4], y[5]), fminf(y[6], y[7])));
  const float mx = fmaxf(fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])), fmaxf(fmaxf(y[4], y[5]), fmaxf(y[6], y[7])));
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(mn), __float_as_uint(-mx), false, false);
  const float red = row_min16(vmin(__uint_as_float(sw[0]), __uint_as_float(sw[1])));
  const float lo0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(red), 0));
  const float hi0 = -__int_as_float(__builtin_amdgcn_readlane(__float_as_int(red), 16));
  const float lo1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(red), 32));
  const float hi1 = -__int_as_float(__builtin_amdgcn_readlane(__float_as_int(red), 48));
  const float glo = (q & 2) ? lo1 : lo0, ghi = (q & 2) ? hi1 : hi0;
  const uint32_t b8 = f8e((q & 1) ? clamp_min_1e8(__fsub_rn(ghi, glo)) : glo);
  const float dec = f8d(b8);
  const float lof0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dec), 0));
  const float scf0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dec), 1));
  const float lof1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dec), 2));
  const float scf1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dec), 3));
  const float scf = g ? scf1 : scf0;
  return VScales{b8, g ? lof1 : lof0, scf, clamp_min_1e8(scf)};
}

// ---------------------------------------------------------------- V path on the fp32 matrix cores
// y = x H for 16 head rows at once (4 tokens x 4 heads; row m = 4 token + head), every output still the sequential fma
// chain over k = 0..127: v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after another, k
// ascending, each as one IEEE fma (denormals, infinities and NaN included; measured against the scalar chain bit for
// bit), so 32 steps of four k make the chain. Prefixes are shared as in hadamard_row8: tile i holds dims j + 16 i
// (column j), one tile for k < 16, two for k < 32, four for k < 64, eight after: 172 MFMA for 16 rows' 2,048 outputs.
// Why: the part issues 75 T fp32 fma/s through MFMA and sustained 35 T through these vector chains.
//   A operand: lane (g, m) = (lane / 16, lane % 16) holds x[m][4 s + g] in x[s];
//   B operand: H[4 s + g][j] for s < 4 (the other k differ by hneg's sign), and its negation;
//   result:    lane (g, j), y[i][r] = output j + 16 i of row 4 g + r: the lane's eight tiles at one r are the eight
//              bits of code byte j of head r of token g.
typedef float f4 __attribute__((ext_vector_type(4)));
struct HadB { f4 p, n; };   // element s & 3
__device__ __forceinline__ HadB had_operand(int lane) {
  const float c = __uint_as_float(0x3DB504F3u);   // fp32(1 / sqrt(128))
  auto h = [&](int s) { return (__popc((4 * s + (lane >> 4)) & (lane & 15)) & 1) ? -c : c; };
  const f4 p = {h(0), h(1), h(2), h(3)};
  return HadB{p, -p};
}
// conv(in[q], x) delivers x[m][4 s + g], s = 8 q .. 8 q + 7, as the chain reaches them
template <typename T, typename Conv>
__device__ __forceinline__ void hadamard_rows16(const T (&in)[4], Conv conv, const HadB& b, f4 (&y)[8]) {
  y[0] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float x[8];
    conv(in[q], x);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int s = 8 * q + u, m = s >> 2, nch = m == 0 ? 1 : m == 1 ? 2 : m < 4 ? 4 : 8;
      if (s == 4 || s == 8 || s == 16) {
#pragma unroll
        for (int i = 0; i < nch / 2; ++i) y[nch / 2 + i] = y[i];
      }
#pragma unroll
      for (int i = 0; i < nch; ++i)
        y[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], hneg(m, i) ? b.n[s & 3] : b.p[s & 3], y[i], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);   // one piece's x at a time
  }
}

// 4 x 4 transpose between four registers and the lanes l, l ^ 16, l ^ 32, l ^ 48: lane group g's register e becomes
// register g of lane group e. All 64 lanes must be active.
__device__ __forceinline__ void transpose_rows4(float& a0, float& a1, float& a2, float& a3) {
  auto sw32 = [](float& u, float& v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(u), __float_as_uint(v), false, false);
    u = __uint_as_float(r[0]); v = __uint_as_float(r[1]);
  };
  auto sw16 = [](float& u, float& v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(v), false, false);
    u = __uint_as_float(r[0]); v = __uint_as_float(r[1]);
  };
  sw32(a0, a2); sw32(a1, a3);
  sw16(a0, a1); sw16(a2, a3);
}

// x of lane's dpp partner inside its quad (CTRL: a quad_perm control word)
template <int CTRL>
__device__ __forceinline__ uint32_t quad(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ float quadf(float x) { return __uint_as_float(quad<CTRL>(__float_as_uint(x))); }
constexpr int QUAD0 = 0x00, QUAD1 = 0x55, QUAD2 = 0xAA, QUAD3 = 0xFF, QUAD_X1 = 0xB1, QUAD_X2 = 0x4E;

// Scales of four tokens' V rows from y (lane (g, j): token g): per 2-head pair (r = 0, 1 and r = 2, 3) the min and max
// of its 256 outputs, in-lane, then over the token's 16 lanes by DPP row reductions; lane j encodes byte q = j & 3 of
// its token: lo (q even) or max(hi - lo, 1e-8) (q odd) of pair q >> 1. lof / scf: both pairs' decoded lo and scale.
struct VScales4 { uint32_t b8; float lof[2], scf[2]; };
__device__ __forceinline__ VScales4 v_scales4(const f4 (&y)[8], int lane) {
  const int q = lane & 3;
  float lo[2], hi[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    float mn = fminf(y[0][2 * p], y[0][2 * p + 1]), mx = fmaxf(y[0][2 * p], y[0][2 * p + 1]);
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      mn = fminf(fminf(mn, y[i][2 * p]), y[i][2 * p + 1]);
      mx = fmaxf(fmaxf(mx, y[i][2 * p]), y[i][2 * p + 1]);
    }
    lo[p] = row_min16(mn);
    hi[p] = -row_min16(-mx);
  }
  const float glo = (q & 2) ? lo[1] : lo[0], ghi = (q & 2) ? hi[1] : hi[0];
  VScales4 s;
  s.b8 = f8e((q & 1) ? clamp_min_1e8(__fsub_rn(ghi, glo)) : glo);
  const float dec = f8d(s.b8);
  s.lof[0] = quadf<QUAD0>(dec); s.scf[0] = quadf<QUAD1>(dec);
  s.lof[1] = quadf<QUAD2>(dec); s.scf[1] = quadf<QUAD3>(dec);
  return s;
}

// Code bytes of four tokens' V rows, packed: byte r of the result is byte j of head r of token g. bit = rne(fl(d / den))
// >= 1 with d = fl(y - lo) is evaluated without the division as d > den / 2: a float d above den / 2 exceeds it by at
// least an ulp of den / 2, so d / den > 1/2 + 2^-25 and the quotient rounds above 1/2; at d = den / 2 it is 1/2, which
// rounds to 0 (den >= 1e-8 is normal; a NaN den or d gives 0 both ways).
__device__ __forceinline__ uint32_t v_bits4(const f4 (&y)[8], const VScales4& s) {
  uint32_t w = 0;
#pragma unroll
  for (int r = 3; r >= 0; --r) {
    const float lo = s.lof[r >> 1], half = clamp_min_1e8(s.scf[r >> 1]) * 0.5f;
#pragma unroll
    for (int i = 7; i >= 0; --i) {   // w = 2 w + bit, the compare's mask as the carry
      const float d = __fsub_rn(y[i][r], lo);
      asm("v_cmp_gt_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(w) : "v"(d), "v"(half) : "vcc");
    }
  }
  return w;
}
// 4 x 4 byte transpose within each quad of lanes: byte r of lane e becomes byte e of lane r, so that lane j = 4 a + e
// holds bytes 4 a .. 4 a + 3 of head e.
__device__ __forceinline__ uint32_t quad_bytes(uint32_t w, int lane) {
  const uint32_t x = quad<QUAD_X1>(w);
  const uint32_t v = __builtin_amdgcn_perm(w, x, (lane & 1) ? 0x07030501u : 0x02060004u);
  const uint32_t z = quad<QUAD_X2>(v);
  return __builtin_amdgcn_perm(v, z, (lane & 2) ? 0x07060302u : 0x01000504u);
}

// The quantizer needs the chain's value only where rounding decides a byte. Its fast form takes y' = c D, D = sum of
// the +-x by v_mfma_f32_16x16x32_bf16 (x and +-1 are exact in bf16; 36 MFMA at twice the rate per instruction and off
// the VALU, which the fp32 MFMA occupies), with a bound on |y' - y|: the chain rounds 128 times, each time by at most
// 2^-24 of a partial sum that is at most c l1, l1 = sum |x| of the row, and D is within 9 2^-24 l1 of the exact sum (the
// largest deviation measured on cancelling, wide-range and denormal rows; 32 is allowed), so |D - y / c| <= 160 2^-24 l1.
// With E = 192 2^-24 l1 (and 1e-30 for flushed denormals) a group of four tokens is done if for every scale byte both
// ends of the value's interval encode alike and every D keeps E plus the threshold's own rounding from its bit's
// threshold; otherwise (one group in six for normal values; infinities and NaN always) the exact chain runs. All
// bytes are those of the chain. Per group of four tokens: 7.1 K cycles of a SIMD for the exact chain alone, about 2.5 K
// for this form with its share of exact ones.
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
struct SignB { u4v even, odd; };   // B operand k = 32 q + 8 g + e, column j + 16 i: set i & 1, negated by parity(q & i >> 1)
__device__ __forceinline__ SignB sign_operand(int lane) {
  const int g = lane >> 4, j = lane & 15;
  auto pair = [&](int d) {
    return 0x3F803F80u | ((uint32_t)(__popc((8 * g + 2 * d) & j) & 1) << 15) |
           ((uint32_t)(__popc((8 * g + 2 * d + 1) & j) & 1) << 31);
  };
  SignB b;
  b.even = u4v{pair(0), pair(1), pair(2), pair(3)};
  b.odd = b.even ^ ((g & 2) ? 0x80008000u : 0u);
  return b;
}
__device__ __forceinline__ f4 mfma_bf(u4v a, u4v b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}
constexpr float VE_L1 = 192.f * 0x1p-24f, VE_ABS = 1e-30f, HC = 0x1.6a09e6p-4f, HC_INV = 0x1.6a09e6p+3f;

// The fast form on one group's raw rows: in[q] = dims 32 q + 8 g .. + 7 of row m in lane (g, m). True where every byte
// is settled (the same in all lanes); b8 is then lane j's scale byte, w the packed code bytes as v_bits4 gives them.
__device__ __forceinline__ bool quick_v4(const uint4 (&in)[4], const SignB& sb, int lane, uint32_t& b8, uint32_t& w) {
  f4 D[8], N = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 8; ++i) D[i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const u4v a = {in[q].x, in[q].y, in[q].z, in[q].w};
    const u4v one = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
    const u4v na = a ^ 0x80008000u;
    N = mfma_bf(a & 0x7FFF7FFFu, one, N);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      D[i] = mfma_bf((__builtin_popcount(q & (i >> 1)) & 1) ? na : a, (i & 1) ? sb.odd : sb.even, D[i]);
  }
  const int q = lane & 3;
  float lo[2], hi[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    float mn = fminf(D[0][2 * p], D[0][2 * p + 1]), mx = fmaxf(D[0][2 * p], D[0][2 * p + 1]);
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      mn = fminf(fminf(mn, D[i][2 * p]), D[i][2 * p + 1]);
      mx = fmaxf(fmaxf(mx, D[i][2 * p]), D[i][2 * p + 1]);
    }
    lo[p] = row_min16(mn);
    hi[p] = -row_min16(-mx);
  }
  float E[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) E[r] = N[r] * VE_L1 + VE_ABS;
  const float e2 = (q & 2) ? fmaxf(E[2], E[3]) : fmaxf(E[0], E[1]);
  const float glo = (q & 2) ? lo[1] : lo[0], ghi = (q & 2) ? hi[1] : hi[0];
  const float mid = ((q & 1) ? ghi - glo : glo) * HC, rad = e2 * ((q & 1) ? 2.f * HC : HC);
  float va = mid - rad, vb = mid + rad;
  if (q & 1) { va = clamp_min_1e8(va); vb = clamp_min_1e8(vb); }
  // the hardware conversion gives f8e's byte for every finite float (checked over all of them)
  const uint32_t ends = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(va, vb, 0, false);
  b8 = ends & 0xFFu;
  bool ok = b8 == ((ends >> 8) & 0xFFu);
  const float dec = f8d(b8);
  const float lof[2] = {quadf<QUAD0>(dec), quadf<QUAD2>(dec)}, scf[2] = {quadf<QUAD1>(dec), quadf<QUAD3>(dec)};
  float T[2], slack[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {   // bit: D > T, T = (lo + den / 2) / c
    const float half = clamp_min_1e8(scf[p]) * 0.5f;
    T[p] = (lof[p] + half) * HC_INV;
    slack[p] = (fabsf(lof[p]) + half) * (HC_INV * 0x1p-20f);
  }
  w = 0;
#pragma unroll
  for (int r = 3; r >= 0; --r) {
    float least = INFINITY;
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      const float t = D[i][r] - T[r >> 1];
      least = fminf(least, fabsf(t));
      asm("v_cmp_lt_f32 vcc, 0, %1\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(w) : "v"(t) : "vcc");
    }
    ok = ok && least > E[r] + slack[r >> 1];   // false for NaN and infinite l1
  }
  return __all(ok);
}

// V bits and scales of tokens [t0, t0 + 4 VG QW) of one sub-block: wave w takes VG groups of four consecutive tokens.
// Lane (g, m) loads dims 8 g + 32 q .. + 7 of row m (four 16-byte pieces, every group's requested up front), the bf16 MFMA's A operand as
// they are; for the exact chain the pieces' elements change places with the other lane groups' so
// that the lane holds x[m][4 s + g].
constexpr int VSPLIT = 4, VTOK = BLK / VSPLIT, VTPW = VTOK / QW;
constexpr int VROW = 132;   // floats per staged row: the 4 rows of a token start on different LDS banks

// Elements 4 u + e (u < 2, e < 4) of the 16-byte bf16 pieces 8 g' + 32 q in the lane groups g' -> lane group g's
// x[2 g' + u] = element 4 u + g of group g', i.e. k = 4 (8 q + 2 g' + u) + g
__device__ __forceinline__ void unpack_piece(const uint4& in, float (&x)[8]) {
  float f[8] = {bf2f_lo(in.x), bf2f_hi(in.x), bf2f_lo(in.y), bf2f_hi(in.y),
                bf2f_lo(in.z), bf2f_hi(in.z), bf2f_lo(in.w), bf2f_hi(in.w)};
  transpose_rows4(f[0], f[1], f[2], f[3]);
  transpose_rows4(f[4], f[5], f[6], f[7]);
#pragma unroll
  for (int gg = 0; gg < 4; ++gg) { x[2 * gg] = f[gg]; x[2 * gg + 1] = f[4 + gg]; }
}

template <int VG, typename Src>
__device__ void quantize_v(const Src& src, uint8_t* __restrict__ out, int t0) {
  const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
  const int tw = t0 + 4 * VG * (threadIdx.x >> 6);   // this wave's first token
  uint4 raw[VG][4];
#pragma unroll
  for (int v = 0; v < VG; ++v) {
    const uint16_t* row = src.vrow(tw + 4 * v + (m >> 2), m & 3) + 8 * g;
#pragma unroll
    for (int q = 0; q < 4; ++q) raw[v][q] = *reinterpret_cast<const uint4*>(row + 32 * q);
  }
  const SignB sb = sign_operand(lane);
#pragma unroll
  for (int v = 0; v < VG; ++v) {
    const uint4 (&in)[4] = raw[v];
    uint32_t b8, w;
    if (!quick_v4(in, sb, lane, b8, w)) {   // uniform over the wave
      f4 y[8];
      hadamard_rows16(in, unpack_piece, had_operand(lane), y);
      const VScales4 sc = v_scales4(y, lane);
      b8 = sc.b8;
      w = v_bits4(y, sc);
    }
    const int t = tw + 4 * v + g;
    if (m < 4) out[((m & 1) ? VSC_O : VLO_O) + t * 2 + (m >> 1)] = (uint8_t)b8;
    *reinterpret_cast<uint32_t*>(out + VB_O + t * 64 + (m & 3) * 16 + (m & ~3)) = quad_bytes(w, lane);
  }
}

// A quantize grid holds, per sub-block, VSPLIT V workgroups (V is independent per token) and 4 K workgroups (one per
// head: all 256 tokens per channel, each row read once). All V workgroups come first: they are the long ones, and the K
// workgroups fill in behind them (448 sub-blocks: 91 us, 98-118 us interleaved, 100 us with K first). V alone takes
// 65 us, K alone 40 us, both mostly the latency of one-shot workgroups at two per CU; 448 sub-blocks of paged rows took
// 147 us with a scalar fma chain per V lane and the code arithmetic per K element, and take 90 us now (2.9 TB/s).
// 32-bit throughout (the host bounds the grid): scalar compares and selects.
struct Part { int unit; bool kpass; int part; };
__device__ __forceinline__ Part part_of(int units, int vsplit) {
  const int i = (int)blockIdx.x;
  const int nv = vsplit * units;
  const bool k = i >= nv;
  const int o = k ? i - nv : i, n = k ? 4 : vsplit;
  return Part{o / n, k, o % n};
}

// kpass: part = the head of the per-head K pass; else the V token range
template <typename Src>
__device__ __forceinline__ void quantize_part(Src& src, uint8_t* __restrict__ out, char* lds, int64_t* rowtab, bool kpass,
                                              int part) {
  if (kpass) {
    src.prepare(rowtab);
    quantize_k(src, out, lds, part);
  }
  else quantize_v<VTPW / 4>(src, out, part * VTOK);
}

__global__ void __launch_bounds__(QTHREADS, QWPS) quantize_dense_kernel(const uint16_t* __restrict__ k,
                                                                   const uint16_t* __restrict__ v,
                                                                   uint8_t* __restrict__ out, int64_t M) {
  __shared__ __align__(16) char lds[sizeof(QuantLds)];
  const Part p = part_of((int)M, VSPLIT);
  DenseSrc src{k, v, p.unit};
  quantize_part(src, out + (int64_t)p.unit * SUB, lds, nullptr, p.kpass, p.part);
}

__global__ void __launch_bounds__(QTHREADS, QWPS) flush_kernel(const uint16_t* __restrict__ ep, const int64_t* __restrict__ eoff,
                                                         int64_t es, int64_t ebs, int64_t e_hs, int64_t e_ts, int64_t e_v,
                                                         uint8_t* __restrict__ qpool, const int64_t* __restrict__ qbt,
                                                         int64_t qs, int64_t bsq, int64_t qs0,
                                                         const int32_t* __restrict__ nq_prev,
                                                         const int32_t* __restrict__ nq_new, int64_t R, int max_new) {
  __shared__ __align__(16) char lds[sizeof(QuantLds)];
  __shared__ int64_t rowtab[BLK];
  const Part p = part_of((int)R * max_new, VSPLIT);
  const int r = p.unit / max_new;
  const int j = nq_prev[r] + p.unit % max_new;
  if (j >= nq_new[r]) return;   // uniform over the workgroup
  const int64_t tok0 = (int64_t)j * BLK;
  uint8_t* dst = qpool + qbt[(int64_t)r * qs + tok0 / bsq] * qs0 + ((tok0 % bsq) / BLK) * SUB;
  PagedSrc src{ep, eoff + (int64_t)r * es, ebs, e_hs, e_ts, e_v, tok0};
  quantize_part(src, dst, lds, rowtab, p.kpass, p.part);
}

// ---------------------------------------------------------------- latency-oriented flush (decode steps)
// A decode step flushes one or two sub-blocks per layer, so the flush costs one sub-block's latency, not throughput.
// Same code as the throughput flush, with finer work: one group of four tokens per V wave (8 V workgroups per sub-block
// instead of 4 of 64 tokens).
constexpr int LSPLIT = BLK / (4 * QW);   // V workgroups per sub-block in the latency flush

__global__ void __launch_bounds__(QTHREADS) flush_lat_kernel(const uint16_t* __restrict__ ep,
                                                             const int64_t* __restrict__ eoff, int64_t es, int64_t ebs,
                                                             int64_t e_hs, int64_t e_ts, int64_t e_v,
                                                             uint8_t* __restrict__ qpool, const int64_t* __restrict__ qbt,
                                                             int64_t qs, int64_t bsq, int64_t qs0,
                                                             const int32_t* __restrict__ nq_prev,
                                                             const int32_t* __restrict__ nq_new, int64_t R, int max_new) {
  __shared__ __align__(16) char lds[sizeof(QuantLds)];
  __shared__ int64_t rowtab[BLK];
  const Part p = part_of((int)R * max_new, LSPLIT);
  const int r = p.unit / max_new;
  const int j = nq_prev[r] + p.unit % max_new;
  if (j >= nq_new[r]) return;   // uniform over the workgroup
  const int64_t tok0 = (int64_t)j * BLK;
  uint8_t* dst = qpool + qbt[(int64_t)r * qs + tok0 / bsq] * qs0 + ((tok0 % bsq) / BLK) * SUB;
  PagedSrc src{ep, eoff + (int64_t)r * es, ebs, e_hs, e_ts, e_v, tok0};
  if (p.kpass) {
    src.prepare(rowtab);
    quantize_k(src, dst, lds, p.part);
  } else quantize_v<1>(src, dst, p.part * 4 * QW);
}

// ---------------------------------------------------------------- dequantize (kv800.py:79-92)
__global__ void __launch_bounds__(256) dequant_kernel(const uint8_t* __restrict__ sb, uint16_t* __restrict__ kout,
                                                      float* __restrict__ vout) {
  __shared__ __align__(16) float xbuf[4][4 * VROW];   // per wave: one token's 4 V rows
  const int64_t m = blockIdx.x;
  const uint8_t* s = sb + m * SUB;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  // K: bf16(code * ksc + klo) (product and sum rounded separately, as the reference's torch ops)
  for (int i = tid; i < BLK * 512 / 8; i += 256) {
    const int t = i / 64, hc0 = (i % 64) * 8, hh = hc0 >> 7, d0 = hc0 & 127;
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      uint32_t pr = 0;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int d = d0 + e + u;
        const uint32_t code = (s[KC_O + (t * 4 + hh) * 32 + (d & 31)] >> (2 * (d >> 5))) & 3u;
        const float kv = __fadd_rn(__fmul_rn((float)code, f8d(s[KSC_O + hh * 128 + d])), f8d(s[KLO_O + hh * 128 + d]));
        pr |= f2bf(kv) << (16 * u);
      }
      o[e >> 1] = pr;
    }
    *reinterpret_cast<uint4*>(kout + (m * BLK + t) * 512 + hc0) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  // V: (bit * vsc + vlo) @ H, wave w = tokens 64w .. 64w + 63, per token its 4 head rows staged in the wave's LDS
  // rows; lane 16 hh + jj builds dims 8 jj .. 8 jj + 7 of row hh and gets dims jj + 16 i back from the chain
  float hl[16];
  const int hh = lane >> 4, jj = lane & 15;
  hadamard_low(hl, jj);
  float* xrow = &xbuf[w][hh * VROW];
  for (int tt = 0; tt < 64; ++tt) {
    const int t = 64 * w + tt;
    {
      const float vsc = f8d(s[VSC_O + t * 2 + (hh >> 1)]), vlo = f8d(s[VLO_O + t * 2 + (hh >> 1)]);
      const uint8_t* vb = s + VB_O + (t * 4 + hh) * 16;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = 8 * jj + e;
        const float bit = (float)((vb[d & 15] >> (d >> 4)) & 1u);
        xrow[d] = __fadd_rn(__fmul_rn(bit, vsc), vlo);
      }
    }
    __builtin_amdgcn_wave_barrier();   // a wave's LDS instructions run in order: this token's rows, then its reads
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    float y[8];
    hadamard_row8(xrow, hl, y);
    float* vo = vout + ((m * BLK + t) * 4 + hh) * 128 + jj;
#pragma unroll
    for (int i = 0; i < 8; ++i) vo[16 * i] = y[i];
  }
}


// ---------------------------------------------------------------- training fake quantization (train.py:82-100)
// fake_quant_k: x (G, 256, C) fp32 -> c * sc8 + lo8 per (group, channel), the K path of the quantizer on fp32 input
// (the product and the sum rounded separately, as torch's elementwise ops). One thread per channel, 256 channels per
// workgroup: the 256 tokens are read twice (min / max, then codes; the second pass hits L2), coalesced along C.
__global__ void __launch_bounds__(256) fake_quant_k_kernel(const float* __restrict__ x, int64_t C,
                                                           float* __restrict__ out) {
  const int64_t g = blockIdx.y, c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  const float* xg = x + g * BLK * C + c;
  float lo = INFINITY, hi = -INFINITY;
#pragma unroll 8
  for (int t = 0; t < BLK; ++t) {
    const float v = xg[(int64_t)t * C];
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
  }
  const float lof = f8d(f8e(lo));
  const float scf = f8d(f8e(clamp_min_1e8(__fdiv_rn(__fsub_rn(hi, lo), 3.0f))));
  const float den = clamp_min_1e8(scf);
  float* og = out + g * BLK * C + c;
#pragma unroll 8
  for (int t = 0; t < BLK; ++t) {
    float code = __builtin_rintf(__fdiv_rn(__fsub_rn(xg[(int64_t)t * C], lof), den));
    code = fminf(fmaxf(code, 0.f), 3.f);
    og[(int64_t)t * C] = __fadd_rn(__fmul_rn(code, scf), lof);
  }
}

// fake_quant_v: v (N, 4, 128) fp32 -> per token y = v H (the quantizer's sequential fma chain), one bit per dim with
// fp8 lo / scale per pair of heads, then (bit * sc8 + lo8) H with the dequantizer's chain: the V value of a
// quantize -> dequantize round trip. One wave per token at a time, the token's rows staged in LDS; lane 16 hh + jj
// holds dims jj + 16 i of row hh in both chains (the quantizer's scales and bit test as in quantize_v).
constexpr int FQV_TPW = 8;   // tokens per wave
__global__ void __launch_bounds__(256) fake_quant_v_kernel(const float* __restrict__ v, int64_t N,
                                                           float* __restrict__ out) {
  __shared__ __align__(16) float xb[4][4 * VROW];   // per wave: the token's 4 rows (v, then the dequantized values)
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int hh = lane >> 4, jj = lane & 15;
  float hl[16];
  hadamard_low(hl, jj);
  float* xrow = &xb[w][hh * VROW];
  const int64_t t0 = ((int64_t)blockIdx.x * 4 + w) * FQV_TPW;
#pragma unroll 1
  for (int tt = 0; tt < FQV_TPW; ++tt) {
    const int64_t t = t0 + tt;
    if (t >= N) break;   // uniform over the wave
    const float4* src = reinterpret_cast<const float4*>(v + (t * 4 + hh) * 128 + 8 * jj);
    const float4 a = src[0], b = src[1];
    *reinterpret_cast<float4*>(xrow + 8 * jj) = a;
    *reinterpret_cast<float4*>(xrow + 8 * jj + 4) = b;
    __builtin_amdgcn_wave_barrier();   // a wave's LDS instructions run in order
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    float y[8];
    hadamard_row8(xrow, hl, y);
    const VScales sc = v_scales(y, lane);
    const float half = sc.den * 0.5f;
    float z[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      z[i] = __fadd_rn(__fmul_rn((__fsub_rn(y[i], sc.lof) > half) ? 1.f : 0.f, sc.scf), sc.lof);
    __builtin_amdgcn_wave_barrier();   // every lane has read the v rows
#pragma unroll
    for (int i = 0; i < 8; ++i) xrow[jj + 16 * i] = z[i];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    hadamard_row8(xrow, hl, y);
#pragma unroll
    for (int i = 0; i < 8; ++i) out[(t * 4 + hh) * 128 + jj + 16 * i] = y[i];
    __builtin_amdgcn_wave_barrier();   // the next token's rows overwrite the staged rows
  }
}


// ---------------------------------------------------------------- prefill history (vllm_attn.py:160-163, 351-380)
// Row r's positions [0, N[r]) as contiguous bf16 K (rotated when cos_t != null) and V at output rows out_off[r] + p:
// positions below 256 NQ[r] come from sub-block p / 256 (K = bf16(code ksc + klo), V = (bit vsc + vlo) H by the
// dequantizer's fp32 chain, then bf16: dequantize_blocks, kv800.py:79-92), the others from the exact pages. RoPE is the
// reference's fp32 kf c + rotate_half(kf) s over the 128-wide tables (cos32 | 1 | cos32 | 1), (sin32 | 0 | sin32 | 0),
// each product and the sum rounded once, then bf16. Unreadable rows (offsets outside their pool, positions past the
// rope table) are written as zeros. One workgroup per (hpos-position tile, row): hpos = 64, a quarter of a sub-block,
// so that the V chain (one wave per token at a time) runs at eight waves per SIMD on a long prefill, or 16 or 4 when
// 64 gives fewer than 1,024 workgroups (a single row). hpos divides 256, so a tile never straddles a sub-block; the
// outputs do not depend on it.
__device__ __forceinline__ void rope8(float (&a)[8], float (&b)[8], const uint16_t* cs, const uint16_t* sn, bool rope) {
  // a = dims d0 .. d0 + 7, b = dims d0 + 64 .. d0 + 71; rope: d0 < 32 (cs / sn the tables' entries d0 ..), else the
  // unrotated dims, for which the table holds cos 1, sin 0
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float c = rope ? bf2f(cs[e]) : 1.0f, s = rope ? bf2f(sn[e]) : 0.0f;
    const float x = a[e], y = b[e];
    a[e] = __fadd_rn(__fmul_rn(x, c), __fmul_rn(-y, s));
    b[e] = __fadd_rn(__fmul_rn(y, c), __fmul_rn(x, s));
  }
}
__device__ __forceinline__ uint4 pack_bf16x8(const float (&x)[8]) {
  return make_uint4(f2bf(x[0]) | (f2bf(x[1]) << 16), f2bf(x[2]) | (f2bf(x[3]) << 16), f2bf(x[4]) | (f2bf(x[5]) << 16),
                    f2bf(x[6]) | (f2bf(x[7]) << 16));
}

// positions per history workgroup: a quarter of a sub-block, cut by 4 (down to 4 positions, one token per wave)
// while the rows give fewer than four workgroups per CU (a single long row: the V chain then runs at four waves per
// SIMD instead of one)
constexpr int HPOS = 64, HPOS_MIN = 4, HPOS_MIN_GROUPS = 1024;
__global__ void __launch_bounds__(256) history_kernel(kv800_paged_t P, const uint16_t* __restrict__ cos_t,
                                                      const uint16_t* __restrict__ sin_t, int64_t rope_rows,
                                                      int64_t qpool_bytes, int64_t epool_elems,
                                                      const int64_t* __restrict__ out_off, uint16_t* __restrict__ kout,
                                                      uint16_t* __restrict__ vout, int hpos) {
  __shared__ __align__(16) float xbuf[4][4 * VROW];   // per wave: one token's 4 dequantized V rows
  __shared__ float klo_s[512], ksc_s[512];
  const int r = blockIdx.y, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int n = P.N[r], p0 = blockIdx.x * hpos;
  if (p0 >= n) return;   // uniform over the workgroup
  const int cnt = min(hpos, n - p0);
  const int sb = p0 / BLK, to = p0 - sb * BLK;   // the positions' sub-block and the first one's token in it
  const int64_t ob = out_off[r] + p0;
  const bool rot = cos_t != nullptr;
  const int nq = min((int64_t)max(P.NQ[r], 0), P.boff_stride);
  const uint4 zero4 = make_uint4(0, 0, 0, 0);
  if (sb < nq) {
    const int64_t base = P.boff[(int64_t)r * P.boff_stride + sb];
    const bool ok = base >= 0 && base + SUB <= qpool_bytes;   // uniform
    const uint8_t* s = P.qpool + (ok ? base : 0);
    if (ok)
      for (int i = tid; i < 512; i += 256) { klo_s[i] = f8d(s[KLO_O + i]); ksc_s[i] = f8d(s[KSC_O + i]); }
    __syncthreads();
    // K: unit u = (token t, head h, d0 = 8 (u % 8)): dims d0 .. d0 + 7 and d0 + 64 .. d0 + 71
    for (int u = tid; u < cnt * 32; u += 256) {
      const int t = u >> 5, h = (u >> 3) & 3, d0 = 8 * (u & 7);
      uint16_t* ko = kout + (ob + t) * 512 + h * 128 + d0;
      const int pos = p0 + t;
      if (!ok || (rot && pos >= rope_rows)) {
        *reinterpret_cast<uint4*>(ko) = zero4;
        *reinterpret_cast<uint4*>(ko + 64) = zero4;
        continue;
      }
      const uint2 by = *reinterpret_cast<const uint2*>(s + KC_O + ((to + t) * 4 + h) * 32 + (d0 & 31));
      const uint32_t bw[2] = {by.x, by.y};
      const int sa = 2 * (d0 >> 5), sb = sa + 4;   // code fields of dims d0 + e and d0 + 64 + e
      float a[8], b[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t byte = (bw[e >> 2] >> (8 * (e & 3))) & 0xFFu;
        const int ia = h * 128 + d0 + e, ib = ia + 64;
        a[e] = bf2f(f2bf(__fadd_rn(__fmul_rn((float)((byte >> sa) & 3u), ksc_s[ia]), klo_s[ia])));
        b[e] = bf2f(f2bf(__fadd_rn(__fmul_rn((float)((byte >> sb) & 3u), ksc_s[ib]), klo_s[ib])));
      }
      if (rot) rope8(a, b, cos_t + (int64_t)pos * 32 + d0, sin_t + (int64_t)pos * 32 + d0, d0 < 32);
      *reinterpret_cast<uint4*>(ko) = pack_bf16x8(a);
      *reinterpret_cast<uint4*>(ko + 64) = pack_bf16x8(b);
    }
    // V: wave w takes tokens w, w + 4, ...; lane 16 hh + jj builds dims 8 jj .. 8 jj + 7 of bit vsc + vlo for row hh,
    // then gets dims jj + 16 i of that row from the chain
    float hl[16];
    const int hh = lane >> 4, jj = lane & 15;
    hadamard_low(hl, jj);
    float* xrow = &xbuf[w][hh * VROW];
    for (int t = w; t < cnt; t += 4) {
      uint16_t* vo = vout + (ob + t) * 512;
      if (!ok) {
        for (int i = lane; i < 512; i += 64) vo[i] = 0;
        continue;
      }
      {
        const float vsc = f8d(s[VSC_O + (to + t) * 2 + (hh >> 1)]), vlo = f8d(s[VLO_O + (to + t) * 2 + (hh >> 1)]);
        const uint8_t* vb = s + VB_O + ((to + t) * 4 + hh) * 16;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int d = 8 * jj + e;
          const float bit = (float)((vb[d & 15] >> (d >> 4)) & 1u);
          xrow[d] = __fadd_rn(__fmul_rn(bit, vsc), vlo);
        }
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      float y[8];
      hadamard_row8(xrow, hl, y);
#pragma unroll
      for (int i = 0; i < 8; ++i) vo[hh * 128 + jj + 16 * i] = (uint16_t)f2bf(y[i]);
    }
    return;
  }
  // exact positions: unit u = (token t, head h, d0), K rotated, V copied
  const int64_t* et = P.eoff + (int64_t)r * P.eoff_stride;
  for (int u = tid; u < cnt * 32; u += 256) {
    const int t = u >> 5, h = (u >> 3) & 3, d0 = 8 * (u & 7);
    const int pos = p0 + t;
    uint16_t* ko = kout + (ob + t) * 512 + h * 128 + d0;
    uint16_t* vo = vout + (ob + t) * 512 + h * 128 + d0;
    const int64_t pg = pos / P.ebs;
    const int64_t eb = pg < P.eoff_stride ? et[pg] : -1;
    const int64_t kr = eb + h * P.e_hs + (pos - pg * P.ebs) * P.e_ts, vr = kr + P.e_v;
    if (eb < 0 || kr < 0 || vr < 0 || kr + 128 > epool_elems || vr + 128 > epool_elems || (rot && pos >= rope_rows)) {
      *reinterpret_cast<uint4*>(ko) = zero4; *reinterpret_cast<uint4*>(ko + 64) = zero4;
      *reinterpret_cast<uint4*>(vo) = zero4; *reinterpret_cast<uint4*>(vo + 64) = zero4;
      continue;
    }
    const uint4 k0 = *reinterpret_cast<const uint4*>(P.epool + kr + d0);
    const uint4 k1 = *reinterpret_cast<const uint4*>(P.epool + kr + d0 + 64);
    *reinterpret_cast<uint4*>(vo) = *reinterpret_cast<const uint4*>(P.epool + vr + d0);
    *reinterpret_cast<uint4*>(vo + 64) = *reinterpret_cast<const uint4*>(P.epool + vr + d0 + 64);
    if (!rot) {
      *reinterpret_cast<uint4*>(ko) = k0;
      *reinterpret_cast<uint4*>(ko + 64) = k1;
      continue;
    }
    const uint32_t wa[4] = {k0.x, k0.y, k0.z, k0.w}, wb[4] = {k1.x, k1.y, k1.z, k1.w};
    float a[8], b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a[e] = (e & 1) ? bf2f_hi(wa[e >> 1]) : bf2f_lo(wa[e >> 1]);
      b[e] = (e & 1) ? bf2f_hi(wb[e >> 1]) : bf2f_lo(wb[e >> 1]);
    }
    rope8(a, b, cos_t + (int64_t)pos * 32 + d0, sin_t + (int64_t)pos * 32 + d0, d0 < 32);
    *reinterpret_cast<uint4*>(ko) = pack_bf16x8(a);
    *reinterpret_cast<uint4*>(ko + 64) = pack_bf16x8(b);
  }
}

}  // namespace
}  // namespace kv800

using namespace kv800;

extern "C" {

int kv800_hip_version(void) { return 100; }

const char* kv800_hip_last_error(void) { return g_err; }

int kv800_hip_quantize_blocks(const uint16_t* k, const uint16_t* v, int64_t M, uint8_t* out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(M >= 0, "quantize_blocks: M = %lld < 0", (long long)M);
  if (M == 0) return KV800_OK;
  KV800_REQUIRE(k && v && out, "quantize_blocks: null pointer");
  KV800_REQUIRE(M * (4 + VSPLIT) <= 0x7FFFFFFF, "quantize_blocks: M = %lld too large", (long long)M);
  KV800_REQUIRE(((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0 && ((uintptr_t)out % 8) == 0,
                "quantize_blocks: k / v must be 16-byte aligned and out 8-byte aligned");
  hipLaunchKernelGGL(quantize_dense_kernel, dim3((unsigned)(M * (4 + VSPLIT))), dim3(QTHREADS), 0, (hipStream_t)stream, k,
                     v, out, M);
  return check_launch("quantize_blocks");
}

int kv800_hip_flush(const uint16_t* epool, const int64_t* eoff, int64_t eoff_stride, int64_t ebs, int64_t e_hs,
                    int64_t e_ts, int64_t e_v, uint8_t* qpool, const int64_t* qbt, int64_t qbt_stride, int64_t bsq,
                    int64_t qs0, const int32_t* nq_prev, const int32_t* nq_new, int64_t R, int64_t max_new,
                    void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(R >= 0 && max_new >= 0, "flush: R and max_new must be >= 0");
  if (R == 0 || max_new == 0) return KV800_OK;
  KV800_REQUIRE(epool && eoff && qpool && qbt && nq_prev && nq_new, "flush: null pointer");
  KV800_REQUIRE(ebs > 0 && bsq > 0 && bsq % BLK == 0, "flush: ebs must be > 0 and bsq a positive multiple of 256");
  KV800_REQUIRE(e_hs % 8 == 0 && e_ts % 8 == 0 && e_v % 8 == 0 && ((uintptr_t)epool % 16) == 0,
                "flush: exact-pool strides must be multiples of 8 elements and the pool 16-byte aligned");
  KV800_REQUIRE(R * max_new * (4 + VSPLIT) <= 0x7FFFFFFF, "flush: grid too large");
  hipLaunchKernelGGL(flush_kernel, dim3((unsigned)(R * max_new * (4 + VSPLIT))), dim3(QTHREADS), 0, (hipStream_t)stream,
                     epool, eoff, eoff_stride, ebs, e_hs, e_ts, e_v, qpool, qbt, qbt_stride, bsq, qs0, nq_prev, nq_new, R,
                     (int)max_new);
  return check_launch("flush");
}

int kv800_hip_flush_latency(const uint16_t* epool, const int64_t* eoff, int64_t eoff_stride, int64_t ebs, int64_t e_hs,
                            int64_t e_ts, int64_t e_v, uint8_t* qpool, const int64_t* qbt, int64_t qbt_stride,
                            int64_t bsq, int64_t qs0, const int32_t* nq_prev, const int32_t* nq_new, int64_t R,
                            int64_t max_new, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(R >= 0 && max_new >= 0, "flush_latency: R and max_new must be >= 0");
  if (R == 0 || max_new == 0) return KV800_OK;
  KV800_REQUIRE(epool && eoff && qpool && qbt && nq_prev && nq_new, "flush_latency: null pointer");
  KV800_REQUIRE(ebs > 0 && bsq > 0 && bsq % BLK == 0, "flush_latency: ebs must be > 0 and bsq a positive multiple of 256");
  KV800_REQUIRE(e_hs % 8 == 0 && e_ts % 8 == 0 && e_v % 8 == 0 && ((uintptr_t)epool % 16) == 0,
                "flush_latency: exact-pool strides must be multiples of 8 elements and the pool 16-byte aligned");
  KV800_REQUIRE(R * max_new * (4 + LSPLIT) <= 0x7FFFFFFF, "flush_latency: grid too large");
  hipLaunchKernelGGL(flush_lat_kernel, dim3((unsigned)(R * max_new * (4 + LSPLIT))), dim3(QTHREADS), 0,
                     (hipStream_t)stream, epool, eoff, eoff_stride, ebs, e_hs, e_ts, e_v, qpool, qbt, qbt_stride, bsq,
                     qs0, nq_prev, nq_new, R, (int)max_new);
  return check_launch("flush_latency");
}

int kv800_hip_dequantize_blocks(const uint8_t* sb, int64_t M, uint16_t* k_out, float* v_out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(M >= 0, "dequantize_blocks: M = %lld < 0", (long long)M);
  if (M == 0) return KV800_OK;
  KV800_REQUIRE(sb && k_out && v_out, "dequantize_blocks: null pointer");
  KV800_REQUIRE(M <= 0x7FFFFFFF, "dequantize_blocks: M too large");
  KV800_REQUIRE(((uintptr_t)k_out % 16) == 0, "dequantize_blocks: k_out must be 16-byte aligned");
  hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)M), dim3(256), 0, (hipStream_t)stream, sb, k_out, v_out);
  return check_launch("dequantize_blocks");
}

int kv800_hip_fake_quant_k(const float* x, int64_t G, int64_t C, float* out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(G >= 0 && C >= 0, "fake_quant_k: G and C must be >= 0");
  if (G == 0 || C == 0) return KV800_OK;
  KV800_REQUIRE(x && out, "fake_quant_k: null pointer");
  KV800_REQUIRE(G <= 65535 && (C + 255) / 256 <= 0x7FFFFFFF, "fake_quant_k: at most 65535 groups per call");
  hipLaunchKernelGGL(fake_quant_k_kernel, dim3((unsigned)((C + 255) / 256), (unsigned)G), dim3(256), 0,
                     (hipStream_t)stream, x, C, out);
  return check_launch("fake_quant_k");
}

int kv800_hip_fake_quant_v(const float* v, int64_t N, float* out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(N >= 0, "fake_quant_v: N < 0");
  if (N == 0) return KV800_OK;
  KV800_REQUIRE(v && out, "fake_quant_v: null pointer");
  KV800_REQUIRE(((uintptr_t)v % 16) == 0, "fake_quant_v: v must be 16-byte aligned");
  const int64_t nb = (N + 4 * FQV_TPW - 1) / (4 * FQV_TPW);
  KV800_REQUIRE(nb <= 0x7FFFFFFF, "fake_quant_v: N too large");
  hipLaunchKernelGGL(fake_quant_v_kernel, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, v, N, out);
  return check_launch("fake_quant_v");
}

int kv800_hip_history(const kv800_paged_t* P, int64_t R, int64_t max_n, const uint16_t* cos_t, const uint16_t* sin_t,
                       int64_t rope_rows, int64_t qpool_bytes, int64_t epool_elems, const int64_t* out_off,
                       uint16_t* k_out, uint16_t* v_out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(P && R >= 0 && max_n >= 0, "history: bad arguments");
  if (R == 0 || max_n == 0) return KV800_OK;
  KV800_REQUIRE(P->N && P->NQ && P->epool && P->eoff && out_off && k_out && v_out, "history: null pointer");
  KV800_REQUIRE(!cos_t == !sin_t, "history: cos_t and sin_t go together");
  KV800_REQUIRE(P->ebs > 0 && P->e_hs % 8 == 0 && P->e_ts % 8 == 0 && P->e_v % 8 == 0 && ((uintptr_t)P->epool % 16) == 0,
                "history: exact strides must be multiples of 8 elements and the pool 16-byte aligned");
  KV800_REQUIRE(P->boff_stride == 0 || (P->qpool && P->boff), "history: quantized rows need qpool and boff");
  KV800_REQUIRE(((uintptr_t)k_out % 16) == 0 && ((uintptr_t)v_out % 16) == 0, "history: outputs must be 16-byte aligned");
  KV800_REQUIRE(R <= 65535, "history: at most 65535 rows per call");
  int hpos = HPOS;
  while (hpos > HPOS_MIN && (max_n + hpos - 1) / hpos * R < HPOS_MIN_GROUPS) hpos /= 4;
  const int64_t tiles = (max_n + hpos - 1) / hpos;
  KV800_REQUIRE(tiles <= 0x7FFFFFFF, "history: max_n too large");
  hipLaunchKernelGGL(history_kernel, dim3((unsigned)tiles, (unsigned)R), dim3(256), 0, (hipStream_t)stream, *P, cos_t,
                     sin_t, rope_rows, qpool_bytes, epool_elems, out_off, k_out, v_out, hpos);
  return check_launch("history");
}

}  // extern "C"
