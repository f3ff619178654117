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

#include <algorithm>

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

constexpr int QTHREADS = 512;    // a K workgroup: one head of a sub-block; a V workgroup: a token range of it
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
// For k = 16 m + kl (m, i < 8, kl < 16), H[k][j + 16 i] = H[kl][j] (-1)^popcount(m & i): a column j keeps the 16 values
// H[kl][j] and every other sign is a compile-time negation; dims j + 16 i (i = 0..7) are the 8 bits of code byte j.
__device__ __forceinline__ constexpr bool hneg(int m, int i) { return __builtin_popcount(m & i) & 1; }

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

// ---------------------------------------------------------------- V path on the fp32 matrix cores
// y = x H for 16 head rows at once (4 tokens x 4 heads; row m = 4 token + head), every output still the sequential fma
// chain over k = 0..127: v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after another, k
// ascending, each as one IEEE fma (denormals, infinities and NaN included; measured against the scalar chain bit for
// bit), so 32 steps of four k make the chain. Outputs whose signs agree on a prefix of k share its partial sums: tile i
// holds dims j + 16 i (column j), one tile for k < 16, two for k < 32, four for k < 64, eight after: 172 MFMA for 16
// rows' 2,048 outputs. Why: the part issues 75 T fp32 fma/s through MFMA and sustained 35 T in vector chains.
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
// Step S of the chain: every tile that exists for its k (templates, so that no tile is indexed at run time)
template <int S>
__device__ __forceinline__ void had_step(float x, const HadB& b, f4 (&y)[8]) {
  constexpr int m = S >> 2, nch = m == 0 ? 1 : m == 1 ? 2 : m < 4 ? 4 : 8;
  if constexpr (S == 4 || S == 8 || S == 16) {
#pragma unroll
    for (int i = 0; i < nch / 2; ++i) y[nch / 2 + i] = y[i];
  }
#pragma unroll
  for (int i = 0; i < nch; ++i)
    y[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, hneg(m, i) ? b.n[S & 3] : b.p[S & 3], y[i], 0, 0, 0);
}
template <int Q, typename Get>
__device__ __forceinline__ void had_piece(const Get& get, const HadB& b, f4 (&y)[8]) {
  float x[8];
  get(Q, x);
  had_step<8 * Q>(x[0], b, y);
  had_step<8 * Q + 1>(x[1], b, y);
  had_step<8 * Q + 2>(x[2], b, y);
  had_step<8 * Q + 3>(x[3], b, y);
  had_step<8 * Q + 4>(x[4], b, y);
  had_step<8 * Q + 5>(x[5], b, y);
  had_step<8 * Q + 6>(x[6], b, y);
  had_step<8 * Q + 7>(x[7], b, y);
  __builtin_amdgcn_sched_barrier(0);   // one piece's x at a time
}
// get(q, x) delivers x[m][4 s + g], s = 8 q .. 8 q + 7, as the chain reaches them
template <typename Get>
__device__ __forceinline__ void hadamard_rows16(const Get& get, const HadB& b, f4 (&y)[8]) {
  y[0] = f4{0.f, 0.f, 0.f, 0.f};
  had_piece<0>(get, b, y);
  had_piece<1>(get, b, y);
  had_piece<2>(get, b, y);
  had_piece<3>(get, b, y);
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
// 2^-24 of a partial sum that is at most c l1, l1 = sum |x| of the row. D's deviations from the exact sum are those of 16
// roundings, one for each eight products added to the accumulator: at most 16 2^-24 l1. Measured over 32 K rows a kind: 15.9
// with one large value and 127 of 2^-20 to 2^-30 of it, 4 with two large values that cancel, 5 over wide ranges, 0.5 for
// normal values; 32 is allowed, so |D - y / c| <= 160 2^-24 l1 (measured: 123, nearly all of it the chain's).
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
// Lane (g, m) loads dims 8 g + 32 q .. + 7 of row m (four 16-byte pieces, every group's requested up front), the bf16
// MFMA's A operand as they are; for the exact chain the pieces' elements change places with the other lane groups' so
// that the lane holds x[m][4 s + g].
constexpr int VSPLIT = 4, VTOK = BLK / VSPLIT, VTPW = VTOK / QW;

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
      hadamard_rows16([&](int q, float (&x)[8]) { unpack_piece(in[q], x); }, had_operand(lane), y);
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
// workgroups fill in behind them (448 sub-blocks: 90 us, 98-118 us interleaved, 100 us with K first, before the chain's
// tiles were indexed at compile time). V alone takes about 60 us, K alone 40 us, both mostly the latency of one-shot
// workgroups at two per CU: by the counters VALU and MFMA issue takes 56 % of the SIMD cycles (bf16 MFMA busy 21 %) at 2.7
// waves per SIMD, which wait in 73 % of theirs. 448 sub-blocks of paged rows took 147 us with a scalar fma chain per V
// lane and the code arithmetic per K element, and take 84 us now (3.1 TB/s).
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
// Loads of sub-block bytes wherever the caller's sub-blocks start (the hardware takes any alignment)
struct __attribute__((packed, aligned(1))) Bytes16 { uint32_t x, y, z, w; };
struct __attribute__((packed, aligned(1))) Bytes8 { uint32_t x, y; };
__device__ __forceinline__ uint4 load16(const uint8_t* p) {
  const Bytes16 b = *reinterpret_cast<const Bytes16*>(p);
  return make_uint4(b.x, b.y, b.z, b.w);
}
__device__ __forceinline__ uint2 load8(const uint8_t* p) {
  const Bytes8 b = *reinterpret_cast<const Bytes8*>(p);
  return make_uint2(b.x, b.y);
}

// V rows back from their bits: y = (bit vsc + vlo) H for four tokens x 4 heads by the exact chain. Lane (g, m) holds row
// m's 16 code bytes and its two values; step s = 4 i + a takes bit i of byte 4 a + g.
__device__ __forceinline__ void dequant_rows16(const uint4& vb, float vsc, float vlo, const HadB& hb, int g, f4 (&y)[8]) {
  const uint32_t lo = __float_as_uint(__fadd_rn(__fmul_rn(0.f, vsc), vlo)), hi = __float_as_uint(__fadd_rn(vsc, vlo));
  const uint32_t b0 = (vb.x >> (8 * g)) & 0xFFu, b1 = (vb.y >> (8 * g)) & 0xFFu;
  const uint32_t b2 = (vb.z >> (8 * g)) & 0xFFu, b3 = (vb.w >> (8 * g)) & 0xFFu;
  auto pick = [&](uint32_t b, int i) {
    const uint32_t mask = (uint32_t)((int32_t)(b << (31 - i)) >> 31);
    return __uint_as_float((mask & hi) | (~mask & lo));
  };
  hadamard_rows16(
      [&](int q, float (&x)[8]) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii) {
          x[4 * ii] = pick(b0, 2 * q + ii);
          x[4 * ii + 1] = pick(b1, 2 * q + ii);
          x[4 * ii + 2] = pick(b2, 2 * q + ii);
          x[4 * ii + 3] = pick(b3, 2 * q + ii);
        }
      },
      hb, y);
}

// Two rounded dequantized keys, packed: bf16(code sc + lo) of byte E of the codes c (the product is exact in fp32, so
// the fused multiply-add rounds where torch's add does); v_cvt_pk_bf16_f32 rounds as f2bf for finite values.
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bfpk(float a, float b) {
  const bf2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float ubyte(uint32_t c, int e) { return (float)((c >> (8 * e)) & 0xFFu); }   // one conversion

// One workgroup per quarter of a sub-block and side (its K, its V), so that 448 sub-blocks fill the part and the V
// chains' workgroups run beside the K workgroups' stores. K: a lane keeps its 8 channels' scales in registers and a
// wave writes whole 1 KB token rows. 448 sub-blocks: 205 us as one workgroup per sub-block with per-element scale
// reads and vector chains, 122 us now (3.1 TB/s). The chains are 5.05 G FMA, 67 us of fp32 MFMA at 75 T FMA/s (MFMA busy 64 %
// of the SIMD cycles, VALU 22 %), the 378 MB 73 us at the rate of a large copy: the V workgroups' scalar dword stores and
// the K workgroups behind them overlap the chains only in part.
constexpr int DPARTS = 4, DTOK = BLK / DPARTS;
__global__ void __launch_bounds__(256) dequant_kernel(const uint8_t* __restrict__ sb, int M, uint16_t* __restrict__ kout,
                                                      float* __restrict__ vout) {
  const int i = (int)blockIdx.x, nv = DPARTS * M;
  const bool kside = i >= nv;                       // V workgroups, the longer ones, first
  const int o = kside ? i - nv : i;
  const int64_t mb = o / DPARTS;
  const uint8_t* s = sb + mb * SUB;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, t0 = (o % DPARTS) * DTOK;
  if (kside) {
    const int h = lane >> 4, p = (lane >> 2) & 3, q = lane & 3, hc0 = 8 * lane;   // dims 32 p + 8 q .. + 7 of head h
    float sc[8], lo[8];
    {
      const uint2 a = load8(s + KSC_O + hc0), b = load8(s + KLO_O + hc0);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sc[e] = f8d(((e < 4 ? a.x : a.y) >> (8 * (e & 3))) & 0xFFu);
        lo[e] = f8d(((e < 4 ? b.x : b.y) >> (8 * (e & 3))) & 0xFFu);
      }
    }
    const uint8_t* kc = s + KC_O + ((t0 + w) * 4 + h) * 32 + 8 * q;
    uint16_t* ko = kout + (mb * BLK + t0 + w) * 512 + hc0;
#pragma unroll 4
    for (int t = 0; t < DTOK; t += 4) {
      const uint2 by = load8(kc + t * 128);
      const uint32_t c0 = (by.x >> (2 * p)) & 0x03030303u, c1 = (by.y >> (2 * p)) & 0x03030303u;
      uint4 r;
      r.x = bfpk(__builtin_fmaf(ubyte(c0, 0), sc[0], lo[0]), __builtin_fmaf(ubyte(c0, 1), sc[1], lo[1]));
      r.y = bfpk(__builtin_fmaf(ubyte(c0, 2), sc[2], lo[2]), __builtin_fmaf(ubyte(c0, 3), sc[3], lo[3]));
      r.z = bfpk(__builtin_fmaf(ubyte(c1, 0), sc[4], lo[4]), __builtin_fmaf(ubyte(c1, 1), sc[5], lo[5]));
      r.w = bfpk(__builtin_fmaf(ubyte(c1, 2), sc[6], lo[6]), __builtin_fmaf(ubyte(c1, 3), sc[7], lo[7]));
      *reinterpret_cast<uint4*>(ko + (int64_t)t * 512) = r;
    }
    return;
  }
  const int g = lane >> 4, m = lane & 15;
  const HadB hb = had_operand(lane);
#pragma unroll 1
  for (int t = t0 + 4 * w; t < t0 + DTOK; t += 16) {
    const int tm = t + (m >> 2);
    const uint4 vb = load16(s + VB_O + tm * 64 + (m & 3) * 16);
    f4 y[8];
    dequant_rows16(vb, f8d(s[VSC_O + tm * 2 + ((m >> 1) & 1)]), f8d(s[VLO_O + tm * 2 + ((m >> 1) & 1)]), hb, g, y);
    float* vo = vout + (mb * BLK + t + g) * 512 + m;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i8 = 0; i8 < 8; ++i8) vo[r * 128 + 16 * i8] = y[i8][r];
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

// The same for C a multiple of 4 and 16-byte aligned tensors: a workgroup takes 64 channels of one group and keeps its
// 256 x 64 values in registers through both passes (a lane: 4 channels of the tokens 16 i + 4 w + g), so x is read once,
// in 16-byte pieces; codes by kcode instead of an IEEE division. 32,768 tokens x 512 channels: 38 -> 20 us (of
// 134 MB); tensors that are not aligned so, or other C, take the kernel above.
__global__ void __launch_bounds__(256) fake_quant_k4_kernel(const float* __restrict__ x, int64_t C, float* __restrict__ out) {
  __shared__ f4 red[2][4][16];
  __shared__ f4 col[2][16];   // lo and scale of the 64 channels
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int64_t c = (int64_t)blockIdx.x * 64 + 4 * c16;
  const int64_t at = ((int64_t)blockIdx.y * BLK + 4 * w + g) * C + c;
  const bool in = c < C;
  f4 v[16];
  if (in) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = *reinterpret_cast<const f4*>(x + at + 16 * i * C);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = f4{0.f, 0.f, 0.f, 0.f};
  }
  f4 mn, mx;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) { lo = fminf(lo, v[i][e]); hi = fmaxf(hi, v[i][e]); }
    auto swap16 = [](float t) { return __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false); };
    auto swap32 = [](float t) { return __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false); };
    auto a = swap16(lo); lo = fminf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    a = swap32(lo); mn[e] = fminf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    auto b = swap16(hi); hi = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
    b = swap32(hi); mx[e] = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
  }
  if (g == 0) { red[0][w][c16] = mn; red[1][w][c16] = mx; }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int t = threadIdx.x;
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      lo = fminf(lo, reinterpret_cast<const float*>(red[0][ww])[t]);
      hi = fmaxf(hi, reinterpret_cast<const float*>(red[1][ww])[t]);
    }
    reinterpret_cast<float*>(col[0])[t] = f8d(f8e(lo));
    reinterpret_cast<float*>(col[1])[t] = f8d(f8e(clamp_min_1e8(__fdiv_rn(__fsub_rn(hi, lo), 3.0f))));
  }
  __syncthreads();
  if (!in) return;
  const f4 lo = col[0][c16], sc = col[1][c16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    f4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)   // code sc is exact, so the fma rounds where the sum does
      o[e] = __builtin_fmaf((float)kcode(__fsub_rn(v[i][e], lo[e]), clamp_min_1e8(sc[e])), sc[e], lo[e]);
    *reinterpret_cast<f4*>(out + at + 16 * i * C) = o;
  }
}

// fake_quant_v: v (N, 4, 128) fp32 -> per token y = v H (the quantizer's sequential fma chain), one bit per dim with
// fp8 lo / scale per pair of heads, then (bit * sc8 + lo8) H with the dequantizer's chain: the V value of a
// quantize -> dequantize round trip. A wave takes four tokens at a time through both chains on fp32 MFMA; lane (g, m)
// loads the float4s 4 (4 u + g) of row m, whose elements change places with the other lane groups'. Between the chains
// the code bytes and the scales go from the result's lanes to the next operand's through the wave's 320 bytes of LDS.
// 32,768 tokens: 67 us with vector chains, 54-57 us now; bound: 2.9 G FMA, 38 us of fp32 MFMA at 75 T FMA/s (busy 76 % of the
// SIMD cycles), beside the scales and bits on the VALU.
constexpr int FQV_GROUPS = 2;   // groups of four tokens per wave
struct FqvLds { uint32_t vb[16][4]; float sc[4][4]; };   // row's code bytes; token's (lo, scale) per pair of heads
__global__ void __launch_bounds__(256) fake_quant_v_kernel(const float* __restrict__ v, int64_t N,
                                                           float* __restrict__ out) {
  __shared__ FqvLds xb[4];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
  FqvLds& L = xb[w];
  const HadB hb = had_operand(lane);
#pragma unroll 1
  for (int gr = 0; gr < FQV_GROUPS; ++gr) {
    const int64_t t = (((int64_t)blockIdx.x * 4 + w) * FQV_GROUPS + gr) * 4;
    if (t >= N) break;   // uniform over the wave
    const int64_t tm = min(t + (m >> 2), N - 1);   // rows past the end repeat the last token's and are not stored
    const float4* src = reinterpret_cast<const float4*>(v + (tm * 4 + (m & 3)) * 128) + g;
    float4 in[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) in[u] = src[4 * u];
    f4 y[8];
    hadamard_rows16(
        [&](int q, float (&x)[8]) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float4 f = in[2 * q + u];
            transpose_rows4(f.x, f.y, f.z, f.w);
            x[4 * u] = f.x; x[4 * u + 1] = f.y; x[4 * u + 2] = f.z; x[4 * u + 3] = f.w;
          }
        },
        hb, y);
    const VScales4 sc = v_scales4(y, lane);
    L.vb[4 * g + (m & 3)][m >> 2] = quad_bytes(v_bits4(y, sc), lane);
    if (m == 0) *reinterpret_cast<float4*>(L.sc[g]) = make_float4(sc.lof[0], sc.scf[0], sc.lof[1], sc.scf[1]);
    __builtin_amdgcn_wave_barrier();   // a wave's LDS instructions run in order
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const uint4 vb = *reinterpret_cast<const uint4*>(L.vb[m]);
    const float2 ls = *reinterpret_cast<const float2*>(&L.sc[m >> 2][m & 2]);
    __builtin_amdgcn_wave_barrier();   // and the next group's writes follow these reads
    dequant_rows16(vb, ls.y, ls.x, hb, g, y);
    if (t + g < N) {
      float* vo = out + (t + g) * 512 + m;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 8; ++i) vo[r * 128 + 16 * i] = y[i][r];
    }
  }
}


// ---------------------------------------------------------------- prefill history (vllm_attn.py:160-163, 351-380)
// Row r's positions [0, N[r]) as contiguous bf16 K (rotated when cos_t != null) and V at output rows out_off[r] + p:
// positions below 256 NQ[r] come from sub-block p / 256 (K = bf16(code ksc + klo), V = (bit vsc + vlo) H by the
// dequantizer's fp32 chain, then bf16: dequantize_blocks, kv800.py:79-92), the others from the exact pages. RoPE is the
// reference's fp32 kf c + rotate_half(kf) s over the 128-wide tables (cos32 | 1 | cos32 | 1), (sin32 | 0 | sin32 | 0),
// each product and the sum rounded once, then bf16. Unreadable rows (offsets outside their pool, positions past the
// rope table) are written as zeros. One workgroup per (hpos-position tile, row): hpos = 32 (two MFMA groups of four
// tokens per wave), or 16 when 32 gives fewer than 1,024 workgroups (a single row). hpos divides 256, so a tile never
// straddles a sub-block; the outputs do not depend on it. 8 rows of 16K positions: 212 us with vector chains and
// software rounding, 134 us now (64 or 16 positions: 137 / 144 us); one row 48 -> 24 us. Bound: 5.8 G FMA, 77 us of fp32 MFMA
// at 75 T FMA/s (busy 57 % of the SIMD cycles), beside 293 MB of stores.
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

// positions per history workgroup
constexpr int HPOS = 32, HPOS_MIN = 16, HPOS_MIN_GROUPS = 1024;
// The new rows of a prefill chunk, appended to each row's history by the workgroups after its `tiles` history tiles
// (the copy and rotation of rope_rows_kernel; one launch where the history, the rotation and two index copies took four).
struct NewRows {
  const uint16_t* k;      // (T, 4, 128) new rows, row r's at [qsl[r], qsl[r + 1])
  const uint16_t* v;
  const int64_t* prev;    // history lengths (instead of P.N); null: history only
  const int64_t* qsl;
  int tiles;              // history tiles of the grid
};
constexpr int NEW_ROWS = 32;   // new rows per workgroup

// One unit of a plain K / V row: dims d0 .. d0 + 7 and d0 + 64 .. of one head from kr / vr (any alignment) to ko / vo,
// the keys rotated at position pos when cos_t is given (clamped into the tables)
__device__ __forceinline__ void copy_unit(const uint16_t* kr, const uint16_t* vr, uint16_t* ko, uint16_t* vo, int d0,
                                          int64_t pos, const uint16_t* cos_t, const uint16_t* sin_t, int64_t rope_rows) {
  const uint4 k0 = load16(reinterpret_cast<const uint8_t*>(kr + d0)), k1 = load16(reinterpret_cast<const uint8_t*>(kr + d0 + 64));
  *reinterpret_cast<uint4*>(vo + d0) = load16(reinterpret_cast<const uint8_t*>(vr + d0));
  *reinterpret_cast<uint4*>(vo + d0 + 64) = load16(reinterpret_cast<const uint8_t*>(vr + d0 + 64));
  if (!cos_t) {
    *reinterpret_cast<uint4*>(ko + d0) = k0;
    *reinterpret_cast<uint4*>(ko + d0 + 64) = k1;
    return;
  }
  const uint32_t wa[4] = {k0.x, k0.y, k0.z, k0.w}, wb[4] = {k1.x, k1.y, k1.z, k1.w};
  float a[8], b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    a[e] = (e & 1) ? bf2f_hi(wa[e >> 1]) : bf2f_lo(wa[e >> 1]);
    b[e] = (e & 1) ? bf2f_hi(wb[e >> 1]) : bf2f_lo(wb[e >> 1]);
  }
  pos = min(max(pos, (int64_t)0), rope_rows - 1);
  rope8(a, b, cos_t + pos * 32 + d0, sin_t + pos * 32 + d0, d0 < 32);
  *reinterpret_cast<uint4*>(ko + d0) = pack_bf16x8(a);
  *reinterpret_cast<uint4*>(ko + d0 + 64) = pack_bf16x8(b);
}

__global__ void __launch_bounds__(256) history_kernel(kv800_paged_t P, const uint16_t* __restrict__ cos_t,
                                                      const uint16_t* __restrict__ sin_t, int64_t rope_rows,
                                                      int64_t qpool_bytes, int64_t epool_elems,
                                                      const int64_t* __restrict__ out_off, uint16_t* __restrict__ kout,
                                                      uint16_t* __restrict__ vout, int hpos, NewRows X) {
  __shared__ float klo_s[512], ksc_s[512];
  const int r = blockIdx.y, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int n = X.prev ? (int)X.prev[r] : P.N[r];
  if (X.prev && (int)blockIdx.x >= X.tiles) {
    const int64_t q0 = X.qsl[r], i0 = (int64_t)((int)blockIdx.x - X.tiles) * NEW_ROWS;
    const int cnt = (int)min((int64_t)NEW_ROWS, X.qsl[r + 1] - q0 - i0);
    for (int u = tid; u < cnt * 32; u += 256) {
      const int h = (u >> 3) & 3, d0 = 8 * (u & 7);
      const int64_t i = i0 + (u >> 5), src = (q0 + i) * 512 + h * 128, dst = (out_off[r] + n + i) * 512 + h * 128;
      copy_unit(X.k + src, X.v + src, kout + dst, vout + dst, d0, n + i, cos_t, sin_t, rope_rows);
    }
    return;
  }
  const int p0 = blockIdx.x * hpos;
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
    bool neg = false;   // a negative scale (the quantizer writes none) can give a key -0
    if (ok)
      for (int i = tid; i < 512; i += 256) {
        klo_s[i] = f8d(s[KLO_O + i]);
        ksc_s[i] = f8d(s[KSC_O + i]);
        neg |= s[KSC_O + i] > 0x7F;
      }
    neg = __syncthreads_or(neg);
    // K: unit = (token t, head h, q): the code bytes 8 q .. 8 q + 7 of (t, h) give dims 32 k + 8 q .. + 7, k = 0..3, of
    // which k = 0 and 2 are rotated
    for (int u = tid; u < cnt * 16; u += 256) {
      const int t = u >> 4, h = (u >> 2) & 3, q = u & 3;
      uint16_t* ko = kout + (ob + t) * 512 + h * 128 + 8 * q;
      const int pos = p0 + t;
      if (!ok || (rot && pos >= rope_rows)) {
#pragma unroll
        for (int k = 0; k < 4; ++k) *reinterpret_cast<uint4*>(ko + 32 * k) = zero4;
        continue;
      }
      const uint2 by = load8(s + KC_O + ((to + t) * 4 + h) * 32 + 8 * q);
      uint32_t o[4][4];   // dims 32 k + 8 q .. + 7, packed pairs
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float* sc = ksc_s + h * 128 + 32 * k + 8 * q;
        const float* lo = klo_s + h * 128 + 32 * k + 8 * q;
        const uint32_t c0 = (by.x >> (2 * k)) & 0x03030303u, c1 = (by.y >> (2 * k)) & 0x03030303u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t c = e < 2 ? c0 : c1;
          const int b = 2 * (e & 1);
          o[k][e] = bfpk(__builtin_fmaf(ubyte(c, b), sc[2 * e], lo[2 * e]),
                         __builtin_fmaf(ubyte(c, b + 1), sc[2 * e + 1], lo[2 * e + 1]));
        }
      }
      if (rot) {
        const uint4 cv = *reinterpret_cast<const uint4*>(cos_t + (int64_t)pos * 32 + 8 * q);
        const uint4 sv = *reinterpret_cast<const uint4*>(sin_t + (int64_t)pos * 32 + 8 * q);
        const uint32_t cw[4] = {cv.x, cv.y, cv.z, cv.w}, sw[4] = {sv.x, sv.y, sv.z, sv.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x0 = bf2f_lo(o[0][e]), x1 = bf2f_hi(o[0][e]), y0 = bf2f_lo(o[2][e]), y1 = bf2f_hi(o[2][e]);
          const float c0 = bf2f_lo(cw[e]), c1 = bf2f_hi(cw[e]), s0 = bf2f_lo(sw[e]), s1 = bf2f_hi(sw[e]);
          o[0][e] = bfpk(__fadd_rn(__fmul_rn(x0, c0), __fmul_rn(-y0, s0)), __fadd_rn(__fmul_rn(x1, c1), __fmul_rn(-y1, s1)));
          o[2][e] = bfpk(__fadd_rn(__fmul_rn(y0, c0), __fmul_rn(x0, s0)), __fadd_rn(__fmul_rn(y1, c1), __fmul_rn(x1, s1)));
          if (neg) {   // the other dims' rotation by cos 1, sin 0 changes nothing but the sign of such a zero
            const float a0 = bf2f_lo(o[1][e]), a1 = bf2f_hi(o[1][e]), b0 = bf2f_lo(o[3][e]), b1 = bf2f_hi(o[3][e]);
            o[1][e] = bfpk(__fadd_rn(a0, __fmul_rn(-b0, 0.f)), __fadd_rn(a1, __fmul_rn(-b1, 0.f)));
            o[3][e] = bfpk(__fadd_rn(b0, __fmul_rn(a0, 0.f)), __fadd_rn(b1, __fmul_rn(a1, 0.f)));
          }
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) *reinterpret_cast<uint4*>(ko + 32 * k) = make_uint4(o[k][0], o[k][1], o[k][2], o[k][3]);
    }
    // V: wave w takes four tokens at a time through the dequantizer's chain; the quads' 4 x 4 exchange of packed pairs
    // leaves each lane four consecutive dims per store
    const int g = lane >> 4, m = lane & 15, e = m & 3;
    const HadB hb = had_operand(lane);
    for (int t = 4 * w; t < cnt; t += 16) {
      const int tm = to + min(t + (m >> 2), cnt - 1);   // rows past the end repeat the last one and are not stored
      uint4 vb = zero4;
      float vsc = 0.f, vlo = 0.f;
      if (ok) {
        vb = load16(s + VB_O + tm * 64 + (m & 3) * 16);
        vsc = f8d(s[VSC_O + tm * 2 + ((m >> 1) & 1)]);
        vlo = f8d(s[VLO_O + tm * 2 + ((m >> 1) & 1)]);
      }
      f4 y[8];
      dequant_rows16(vb, vsc, vlo, hb, g, y);   // zeros where the sub-block is not readable
      uint16_t* vo = vout + (ob + t + g) * 512 + (m & ~3);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        uint32_t v[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t x = bfpk(y[2 * p][r], y[2 * p + 1][r]);
          v[p] = __builtin_amdgcn_perm(x, quad<QUAD_X1>(x), (e & 1) ? 0x07060302u : 0x01000504u);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {   // plane 4 p + e, dims m & ~3 .. + 3
          const uint32_t own = (e & 2) ? v[2 * p + 1] : v[2 * p];
          const uint32_t got = quad<QUAD_X2>((e & 2) ? v[2 * p] : v[2 * p + 1]);
          if (t + g < cnt)
            *reinterpret_cast<uint2*>(vo + r * 128 + 16 * (4 * p + e)) =
                (e & 2) ? make_uint2(got, own) : make_uint2(own, got);
        }
      }
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

// ---------------------------------------------------------------- prefill keys of a window layer
// Row r's attended rows in order, (its sinks, its kept exact rows [lo, prev), its new rows), as contiguous K (rotated at
// their positions when cos_t is given) and V at output rows ksl[r] + i, with their positions in kp: one launch for what
// the host assembled with some 40 gathers, concatenations and index uploads. lo = max(0, prev - (win - 1)), sinks
// 0 .. min(nsink, lo) - 1. Rows outside the pools are zeros. A workgroup copies WIN_ROWS rows, 32 units a row.
// 8 rows of 2,048 new tokens over a full window: the whole call 555 -> 134 us.
constexpr int WIN_ROWS = 32;
constexpr int64_t MAX_GRID_Y = 65535;
__global__ void __launch_bounds__(256) window_keys_kernel(kv800_paged_t P, const uint16_t* __restrict__ cos_t,
                                                          const uint16_t* __restrict__ sin_t, int64_t rope_rows,
                                                          int64_t epool_elems, int64_t sink_elems, int nsink,
                                                          const int64_t* __restrict__ prev, const int64_t* __restrict__ ksl,
                                                          const int64_t* __restrict__ qsl,
                                                          const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                                          uint16_t* __restrict__ kout, uint16_t* __restrict__ vout,
                                                          int32_t* __restrict__ kp) {
  const int r = blockIdx.y;
  const int64_t n = prev[r], lo = max(n - (P.win - 1), (int64_t)0), ns = min((int64_t)nsink, lo);
  const int64_t rows = ksl[r + 1] - ksl[r], i0 = (int64_t)blockIdx.x * WIN_ROWS;
  const int cnt = (int)min((int64_t)WIN_ROWS, rows - i0);
  for (int u = threadIdx.x; u < cnt * 32; u += 256) {
    const int h = (u >> 3) & 3, d0 = 8 * (u & 7);
    const int64_t i = i0 + (u >> 5), dst = (ksl[r] + i) * 512 + h * 128;
    const int64_t pos = i < ns ? i : lo + (i - ns);
    const uint16_t *kr = nullptr, *vr = nullptr;
    if (i < ns) {
      const int64_t a = P.skoff[r] + (i * 4 + h) * 128, b = P.svoff[r] + (i * 4 + h) * 128;
      if (a >= 0 && b >= 0 && a + 128 <= sink_elems && b + 128 <= sink_elems) { kr = P.sk + a; vr = P.sv + b; }
    } else if (pos < n) {
      const int64_t pg = pos / P.ebs, base = pg < P.eoff_stride ? P.eoff[r * P.eoff_stride + pg] : -1;
      const int64_t a = base + h * P.e_hs + (pos - pg * P.ebs) * P.e_ts, b = a + P.e_v;
      if (base >= 0 && a >= 0 && b >= 0 && a + 128 <= epool_elems && b + 128 <= epool_elems) {
        kr = P.epool + a;
        vr = P.epool + b;
      }
    } else {
      kr = k + (qsl[r] + (pos - n)) * 512 + h * 128;
      vr = v + (qsl[r] + (pos - n)) * 512 + h * 128;
    }
    if ((u & 31) == 0) kp[ksl[r] + i] = (int32_t)pos;
    if (kr) {
      copy_unit(kr, vr, kout + dst, vout + dst, d0, pos, cos_t, sin_t, rope_rows);
    } else {
      const uint4 zero4 = make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(kout + dst + d0) = zero4; *reinterpret_cast<uint4*>(kout + dst + d0 + 64) = zero4;
      *reinterpret_cast<uint4*>(vout + dst + d0) = zero4; *reinterpret_cast<uint4*>(vout + dst + d0 + 64) = zero4;
    }
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
  KV800_REQUIRE(M <= 0x7FFFFFFF / (2 * DPARTS), "dequantize_blocks: M too large");
  KV800_REQUIRE(((uintptr_t)k_out % 16) == 0, "dequantize_blocks: k_out must be 16-byte aligned");
  hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)(M * 2 * DPARTS)), dim3(256), 0, (hipStream_t)stream, sb, (int)M, k_out,
                     v_out);
  return check_launch("dequantize_blocks");
}

int kv800_hip_fake_quant_k(const float* x, int64_t G, int64_t C, float* out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(G >= 0 && C >= 0, "fake_quant_k: G and C must be >= 0");
  if (G == 0 || C == 0) return KV800_OK;
  KV800_REQUIRE(x && out, "fake_quant_k: null pointer");
  KV800_REQUIRE(G <= 65535 && (C + 255) / 256 <= 0x7FFFFFFF, "fake_quant_k: at most 65535 groups per call");
  if (C % 4 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)out % 16) == 0)
    hipLaunchKernelGGL(fake_quant_k4_kernel, dim3((unsigned)((C + 63) / 64), (unsigned)G), dim3(256), 0,
                       (hipStream_t)stream, x, C, out);
  else
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
  const int64_t nb = (N + 16 * FQV_GROUPS - 1) / (16 * FQV_GROUPS);
  KV800_REQUIRE(nb <= 0x7FFFFFFF, "fake_quant_v: N too large");
  hipLaunchKernelGGL(fake_quant_v_kernel, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, v, N, out);
  return check_launch("fake_quant_v");
}

// The history launch, with the chunk's new rows when X.k is given (max_new their largest count per row).
static int launch_history(const kv800_paged_t* P, int64_t R, int64_t max_n, const uint16_t* cos_t, const uint16_t* sin_t,
                          int64_t rope_rows, int64_t qpool_bytes, int64_t epool_elems, const int64_t* out_off,
                          uint16_t* k_out, uint16_t* v_out, NewRows X, int64_t max_new, void* stream) {
  KV800_REQUIRE(!cos_t == !sin_t, "history: cos_t and sin_t go together");
  KV800_REQUIRE(P->ebs > 0 && P->e_hs % 8 == 0 && P->e_ts % 8 == 0 && P->e_v % 8 == 0 && ((uintptr_t)P->epool % 16) == 0,
                "history: exact strides must be multiples of 8 elements and the pool 16-byte aligned");
  KV800_REQUIRE(P->boff_stride == 0 || (P->qpool && P->boff), "history: quantized rows need qpool and boff");
  KV800_REQUIRE(((uintptr_t)k_out % 16) == 0 && ((uintptr_t)v_out % 16) == 0, "history: outputs must be 16-byte aligned");
  KV800_REQUIRE(R <= 65535, "history: at most 65535 rows per call");
  int hpos = HPOS;
  while (hpos > HPOS_MIN && (max_n + hpos - 1) / hpos * R < HPOS_MIN_GROUPS) hpos /= 2;
  const int64_t tiles = (max_n + hpos - 1) / hpos, grid = tiles + (max_new + NEW_ROWS - 1) / NEW_ROWS;
  KV800_REQUIRE(grid <= 0x7FFFFFFF, "history: max_n too large");
  X.tiles = (int)tiles;
  hipLaunchKernelGGL(history_kernel, dim3((unsigned)grid, (unsigned)R), dim3(256), 0, (hipStream_t)stream, *P, cos_t,
                     sin_t, rope_rows, qpool_bytes, epool_elems, out_off, k_out, v_out, hpos, X);
  return check_launch("history");
}

int kv800_hip_history(const kv800_paged_t* P, int64_t R, int64_t max_n, const uint16_t* cos_t, const uint16_t* sin_t,
                       int64_t rope_rows, int64_t qpool_bytes, int64_t epool_elems, const int64_t* out_off,
                       uint16_t* k_out, uint16_t* v_out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(P && R >= 0 && max_n >= 0, "history: bad arguments");
  if (R == 0 || max_n == 0) return KV800_OK;
  KV800_REQUIRE(P->N && P->NQ && P->epool && P->eoff && out_off && k_out && v_out, "history: null pointer");
  return launch_history(P, R, max_n, cos_t, sin_t, rope_rows, qpool_bytes, epool_elems, out_off, k_out, v_out, NewRows{},
                        0, stream);
}

int kv800_hip_prefill_keys(const kv800_paged_t* P, int64_t R, int64_t max_prev, int64_t max_new, const uint16_t* cos_t,
                           const uint16_t* sin_t, int64_t rope_rows, int64_t qpool_bytes, int64_t epool_elems,
                           const int64_t* prev, const int64_t* qsl, const int64_t* ksl, const uint16_t* k,
                           const uint16_t* v, uint16_t* k_out, uint16_t* v_out, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(P && R >= 0 && max_prev >= 0 && max_new >= 0, "prefill_keys: bad arguments");
  if (R == 0 || max_prev + max_new == 0) return KV800_OK;
  KV800_REQUIRE(P->NQ && P->epool && P->eoff && prev && qsl && ksl && (!max_new || (k && v)) && k_out && v_out,
                "prefill_keys: null pointer");
  KV800_REQUIRE(!cos_t || rope_rows > 0, "prefill_keys: empty RoPE tables");
  return launch_history(P, R, max_prev, cos_t, sin_t, rope_rows, qpool_bytes, epool_elems, ksl, k_out, v_out,
                        NewRows{k, v, prev, qsl, 0}, max_new, stream);
}

int kv800_hip_window_keys(const kv800_paged_t* P, int64_t R, int64_t max_rows, const uint16_t* cos_t,
                          const uint16_t* sin_t, int64_t rope_rows, int64_t epool_elems, int64_t sink_elems,
                          int64_t nsink, const int64_t* prev, const int64_t* qsl, const int64_t* ksl, const uint16_t* k,
                          const uint16_t* v, uint16_t* k_out, uint16_t* v_out, int32_t* kp, void* stream) {
  g_err[0] = 0;
  KV800_REQUIRE(P && R >= 0 && max_rows >= 0 && nsink >= 0, "window_keys: bad arguments");
  if (R == 0 || max_rows == 0) return KV800_OK;
  KV800_REQUIRE(P->epool && P->eoff && prev && qsl && ksl && k_out && v_out && kp, "window_keys: null pointer");
  KV800_REQUIRE(!nsink || (P->sk && P->sv && P->skoff && P->svoff), "window_keys: sinks need sk, sv, skoff and svoff");
  KV800_REQUIRE(!cos_t == !sin_t && (!cos_t || rope_rows > 0), "window_keys: cos_t and sin_t go together, with rows");
  KV800_REQUIRE(P->ebs > 0 && P->win > 0, "window_keys: ebs and win must be > 0");
  KV800_REQUIRE(((uintptr_t)k_out % 16) == 0 && ((uintptr_t)v_out % 16) == 0,
                "window_keys: outputs must be 16-byte aligned");
  KV800_REQUIRE(max_rows < (1ll << 31), "window_keys: rows of 2^31 keys and more");
  for (int64_t r0 = 0; r0 < R; r0 += MAX_GRID_Y) {   // one launch, but for more rows than a grid's y holds
    kv800_paged_t rows = *P;
    rows.eoff += r0 * P->eoff_stride;
    if (nsink) { rows.skoff += r0; rows.svoff += r0; }
    hipLaunchKernelGGL(window_keys_kernel,
                       dim3((unsigned)((max_rows + WIN_ROWS - 1) / WIN_ROWS), (unsigned)std::min(R - r0, MAX_GRID_Y)),
                       dim3(256), 0, (hipStream_t)stream, rows, cos_t, sin_t, rope_rows, epool_elems, sink_elems,
                       (int)nsink, prev + r0, ksl + r0, qsl + r0, k, v, k_out, v_out, kp);
    const int rc = check_launch("window_keys");
    if (rc != KV800_OK) return rc;
  }
  return KV800_OK;
}

}  // extern "C"
