// kv800_prefill.hip -- prefill / extend attention of the 800h layers on gfx950 (the attention of vllm_attn.py:168-211
// and 351-402 for rows that bring more than one new token).
//
//   rope_rows_kernel  keys (S, 4, 128) bf16 rotated at their positions with the (P, 32) bf16 tables of the 32 rotating
//                     frequencies, as vllm_attn.py:160-163 does over its 128-wide tables (cos32 | 1 | cos32 | 1,
//                     sin32 | 0 | sin32 | 0): every element is k * c + rot(k) * s in fp32 (both products exact), then
//                     rounded to bf16 -- the same value, bit for bit, dims without a frequency included.
//   prefill_kernel    flash attention of R ragged rows. Row i has queries q[qsl[i], qsl[i+1]) (T, 16 heads, 128) at the
//                     consecutive positions qpos0[i], qpos0[i] + 1, ... and keys / values K, V[ksl[i], ksl[i+1])
//                     (S, 4 KV heads, 128) at the ascending positions kp (kp = null: key j of a row at position
//                     j, as quantized layers assemble them); query head h reads KV head h / 4. A key is
//                     kept when kp <= query position and, with window > 0, kp > query position - window or kp < nsink
//                     (the quantized, window + sinks and sliding masks of vllm_attn.py:168-184). fp32 scores and
//                     online softmax, bf16 probabilities for the P.V product, fp32 accumulation, bf16 out.
//
// prefill_kernel, one workgroup = 32 consecutive queries of one row and one KV head g; wave w computes query head
// 4 g + w for its 32 queries, so the 4 waves share each 64-key tile staged in LDS. Per wave and tile, with
// v_mfma_f32_32x32x16_bf16 (lane l: D column l % 32, D rows 8 c + 4 (l / 32) + 0..3; A row l % 32 and B column l % 32
// over k = 8 (l / 32) + 0..7):
//   S^T = K . Q^T   (keys x queries): A = K rows from LDS, B = the wave's queries held in registers;
//   O^T += V^T . P^T (dims x queries): A = V^T read from the V rows by ds_read_b64_tr_b16, B = the lane's own
//                    probabilities.
// Both results keep one query per lane column (l % 32), so the softmax statistics of a query live in two lanes and are
// combined with one cross-lane step, and the O rescale (when a query's running max grows, over one long list of keys only
// when it grows by more than PLAZY; 16 queries at a time) needs no data movement. P^T's B operand is the lane's 8
// probabilities of keys 4 G + i and 8 + 4 G + i (G = l / 32) of each 16-key step, the key order in which the transposed
// reads deliver V^T. The tiles are double-buffered in LDS and
// loaded straight into it (buffer loads with the lds modifier, through a buffer resource whose reads past the row's keys
// return zeros; the next tile's loads are in flight while the current one is multiplied, one barrier per tile), and a
// tile whose keys are all in range, precede the workgroup's first query and lie in its last query's window (or are sinks)
// is not masked.
// Bound: matrix and VALU issue, which overlap only in part, at the clock the part holds under them (1.9 GHz here). 32 x 32
// MFMA instead of twice as many 16 x 16 ones, with half the cross-lane steps, and the phase priorities: 8 ragged rows of up
// to 2048 queries over up to 16K keys (2.2 TFLOP), whole call, 2,424 -> 2,370 -> 2,240 us on one box, 2,120-2,200 us on
// others (this kernel 1.03-1.07 PFLOP/s; a library product of 8192^3 reaches 1.14 on the same card). MFMA busy 58 % of the
// SIMD cycles, waves wait in 61 % of theirs at 1.85 per SIMD; the LDS counts two conflict cycles per MFMA, which the 16 x 16
// reads did not have, and waves wait for it in 4 %.
// Key tiles outside [first key a query of the workgroup can see, last key not in its future] are skipped: for window
// layers only the sink keys and the keys of the window are read, as one list (template flag WIN: its addresses cost the
// windowless kernel 4 %). A window workgroup has 5 tiles, so its start counts as much: the row and the three key bounds
// are found by 64-way searches side by side, behind the query loads. 8 rows x 2048 queries, window 256 + 4 sinks, whole
// call: 131 us with a sink tile, masks on every tile and one search after the other, 117 us now (34 GFLOP, 134 MB of Q and
// output: latency of the tiles' loads, two workgroups per CU).
// The grid is one workgroup per (KV head, 32-query tile), numbered so that each XCD runs whole (KV head, row) runs of
// tiles: the 64 workgroups of a 2048-query chunk walk the same key tiles together through one L2.
#include "kv800_common.h"
#include "../../include/kv800_hip.h"

namespace kv800 {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef short b8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4 lds_s4;

typedef __bf16 mb8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f16v mfma_bf(u4v a, u4v b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mb8, a), __builtin_bit_cast(mb8, b), c, 0, 0, 0);
}

// ---------------------------------------------------------------- RoPE of key rows
// one thread per (row, head, d < 64): the pair (d, d + 64)
__global__ void __launch_bounds__(256)
rope_rows_kernel(const uint16_t* __restrict__ k, const int64_t* __restrict__ pos, int64_t S,
                 const uint16_t* __restrict__ cos_t, const uint16_t* __restrict__ sin_t, int64_t P,
                 uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= S * 256) return;
  const int64_t row = i >> 8;
  const int hd = (int)(i & 255), h = hd >> 6, d = hd & 63;
  int64_t p = pos[row];
  p = p < 0 ? 0 : (p >= P ? P - 1 : p);            // positions past the table are a caller error; stay in bounds
  const float c = d < 32 ? bf2f(cos_t[p * 32 + d]) : 1.0f;
  const float s = d < 32 ? bf2f(sin_t[p * 32 + d]) : 0.0f;
  const int64_t base = (row * 4 + h) * 128;
  const float lo = bf2f(k[base + d]), hi = bf2f(k[base + d + 64]);
  out[base + d] = (uint16_t)f2bf(lo * c + (-hi) * s);
  out[base + d + 64] = (uint16_t)f2bf(hi * c + lo * s);
}

// two floats -> packed bf16, round to nearest even (one v_cvt_pk_bf16_f32; equal to f2bf for finite values)
__device__ __forceinline__ uint32_t bfpk(float a, float b) {
  const bf2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}

// ---------------------------------------------------------------- flash attention of ragged rows
// A workgroup of 4 waves takes PQ = 32 consecutive queries of one row (one interface tile) and one KV head g; wave w
// computes query head 4 g + w for its 32 queries. Every workgroup of the grid has work (a
// grid whose idle workgroups sat at every other index put all the work on half the XCDs under round-robin dispatch),
// and the workgroups of one (KV head, row) run on one XCD, in order, so the row's key tiles are read once into that
// XCD's L2 for its 64 query tiles. Keys come in tiles of 64, loaded into LDS as K and V rows by LDS-direct loads (no
// register staging) and double-buffered: the next tile's loads are in flight while the current one is multiplied, one
// barrier per tile. A tile that every query of the workgroup sees whole needs no mask: in a chunk over a long history,
// nearly every tile.
constexpr int PQ = 32;      // queries per workgroup = per interface tile (tile_off counts these)
constexpr int PPART = 132;  // floats per key-split partial of (query, head): 128 dims of o, m, l, 2 of padding
constexpr int PMAXSPLIT = 256;
constexpr int PK = 64;      // keys per LDS tile

// a tile as staged by LDS-direct loads: K and V rows of 256 bytes, unpadded, their 16-byte pieces permuted within
// each row so that the operand reads spread over the banks: piece p of key row j at piece p ^ (j & 15) (K: 32 rows
// read at one piece per instruction) and p ^ 2 (j & 7) (V: 32-byte pairs of pieces, 4 rows per 16 lanes)
struct alignas(16) PTile {
  uint16_t k[PK * 128];
  uint16_t v[PK * 128];
  int32_t kp[PK];
};
__device__ __forceinline__ int kswz(int j, int p) { return p ^ (j & 15); }
__device__ __forceinline__ int vswz(int j, int p) { return p ^ (2 * (j & 7)); }
// Log2 units a query's running max may lag its scores (p <= 2^8 in bf16) where it sees the keys as one long list. A window
// workgroup or a key split sees a few tiles, and there the max is kept exact (no lag): the largest key's probability is then
// 1, without a bf16 rounding, while a max of the first tile that later keys just exceed puts these where the rounding is
// coarsest. Error against 64 bits with the lag / without: window 256 + 4 sinks 2.24e-3 / 1.85e-3, split rows 2.06-2.21e-3 /
// 1.71-1.77e-3 (1.66e-3 is the rounding of the output alone); time 113.7 / 116.4 us (8 x 2048 queries, window), 26.0 / 26.7
// us (64 queries x 16K keys, 32 splits). Over 16K keys unsplit, 2.204e-3, no lag would rescale in most tiles.
constexpr float PLAZY = 8.f;
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int RSRC_WORD3 = 0x00020000;   // raw (untyped, unswizzled) buffer access on gfx9-family parts

// r[k] = first index in [0, n) with a[index] > x[k] (a ascending), n if none: NX 64-way searches by the whole wave, side
// by side (lane l probes lo + l step; the count of probes <= x, from a ballot, narrows [lo, hi) 64-fold), so n = 4K
// entries take two dependent loads for all of them. All 64 lanes must be active; the results are the same in every lane.
template <int NX, typename A>
__device__ __forceinline__ void upper(const A* a, int n, const int64_t (&x)[NX], int (&r)[NX]) {
  int lo[NX], hi[NX];
#pragma unroll
  for (int k = 0; k < NX; ++k) { lo[k] = 0; hi[k] = n; }   // the answer lies in [lo, hi]
  const int lane = threadIdx.x & 63;
  for (bool more = n > 0; more;) {
    more = false;
    int64_t v[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const int idx = lo[k] + lane * ((hi[k] - lo[k] + 63) / 64);
      v[k] = a[idx < hi[k] ? idx : 0];
    }
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const int step = (hi[k] - lo[k] + 63) / 64;
      const int c = __popcll(__ballot(lo[k] + lane * step < hi[k] && v[k] <= x[k]));   // probes 0 .. c - 1 are <= x
      const int next = c == 0 ? lo[k] : lo[k] + c * step;                // the first probe > x, or past hi
      if (c > 0) lo[k] += (c - 1) * step + 1;                            // behind the last probe <= x
      hi[k] = step <= 1 ? lo[k] : (next < hi[k] ? next : hi[k]);
      more = more || hi[k] > lo[k];
    }
  }
#pragma unroll
  for (int k = 0; k < NX; ++k) r[k] = lo[k];
}

// x's values of lanes l and l ^ 32 without an LDS round trip: v_permlane32_swap on two copies of x leaves both halves in
// every lane. All 64 lanes must be active.
__device__ __forceinline__ float max2halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum2halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <bool WIN>   // window > 0
__global__ void __launch_bounds__(256, 2)
prefill_kernel(const uint16_t* __restrict__ q, const int64_t* __restrict__ qsl, const int64_t* __restrict__ qpos0,
               const uint16_t* __restrict__ K, const uint16_t* __restrict__ V, const int32_t* __restrict__ kp,
               const int64_t* __restrict__ ksl, const int64_t* __restrict__ tile_off, int64_t R, int64_t window,
               int64_t nsink, float scale_log2, uint16_t* __restrict__ out, int splits, float* __restrict__ part) {
  __shared__ PTile tA, tB;   // two buffers as two objects: a read of one is not held for the other's loads
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  // workgroup b runs on XCD b % 8 (round-robin dispatch): XCD x takes the contiguous run L = [x per + min(x, rem),
  // ...) of the (g, t, split) order (split fastest, then t), so the workgroups sharing a row's keys of one KV head
  // share that XCD's L2
  const int nb = (int)gridDim.x, xcd = (int)blockIdx.x & 7, per = nb >> 3, rem = nb & 7;
  const int L = xcd * per + min(xcd, rem) + ((int)blockIdx.x >> 3);
  const int ntl = nb / (4 * splits);
  const int g = L / (ntl * splits), h = 4 * g + w;
  const int lr = L - g * ntl * splits, sp = lr % splits;
  const int col = lane & 31, G = lane >> 5;   // query column; key / dim half
  // ---- row of this tile: last i with tile_off[i] <= t (tile_off[0] = 0)
  const int64_t t = lr / splits;
  const int64_t tx[1] = {t};
  int rows_to[1];
  upper(tile_off, (int)R, tx, rows_to);
  const int64_t row = max(rows_to[0], 1) - 1, lt = t - tile_off[row];
  const int64_t q0 = qsl[row] + lt * PQ;
  const int nq = (int)min((int64_t)PQ, qsl[row + 1] - q0);
  const int64_t p0 = qpos0[row] + (q0 - qsl[row]);
  const int64_t ks = ksl[row];
  const int S = (int)(ksl[row + 1] - ks);   // keys of 1 KB: a device holds fewer than 2^31
  const int32_t* kpr = kp ? kp + ks : nullptr;   // null: key j of the row at position j
  // ---- the wave's queries as the B operands of S^T = K . Q^T (8 k-steps of 16 dims)
  const bool qok = col < nq;
  const int qpos = (int)(p0 + col);
  u4v qb[8];
#pragma unroll
  for (int s = 0; s < 8; ++s)
    qb[s] = qok ? *reinterpret_cast<const u4v*>(q + ((q0 + col) * 16 + h) * 128 + 16 * s + 8 * G) : u4v{0, 0, 0, 0};
  // ---- key ranges: [0, sink_end) and [kbeg, kend)
  const int64_t pl = p0 + nq - 1;   // the tile's last query position
  int kend, kbeg = 0, sink_end = 0;
  if (kpr) {
    constexpr int NX = WIN ? 3 : 1;
    const int64_t xs[3] = {pl, p0 - window, nsink - 1};
    int64_t x[NX];
    int r[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) x[k] = xs[k];
    upper(kpr, S, x, r);
    kend = r[0];
    if (WIN) { kbeg = r[NX / 2]; sink_end = r[NX - 1]; }
  } else {                          // positions = indices 0 .. S - 1
    const auto first = [&](int64_t x) { return x < 0 ? 0 : (x + 1 < S ? (int)x + 1 : S); };
    kend = first(pl);
    if (WIN) { kbeg = first(p0 - window); sink_end = first(nsink - 1); }
  }
  sink_end = min(sink_end, kbeg);
  if (kbeg <= sink_end) { kbeg = 0; sink_end = 0; }
  // The keys as one list: entries [0, ns) the sinks, from ns on [kbeg, kend). A tile that holds both reaches from the row's
  // first key by 32-bit byte offsets; where these do not suffice, the sinks end with a tile of their own (entries
  // [sink_end, ns) empty). A window of 256 with 4 sinks takes 5 tiles of 64 per 32 queries instead of 6.
  const int ns = kbeg < (1 << 20) ? sink_end : (sink_end + PK - 1) / PK * PK;
  const int nt = (ns + (kend - kbeg) + PK - 1) / PK;
  // key split sp of `splits` takes tiles [i0, i1) of the nt (all of them without a split)
  const int per_sp = (nt + splits - 1) / splits, i0 = min(nt, sp * per_sp), i1 = min(nt, i0 + per_sp);
  f16v o[4];   // dims 32 j + 8 (v / 4) + 4 G + v % 4 of query col
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[j][v] = 0.f;
  float m = qok ? -1e30f : 1e30f, lsum = 0.f;   // columns without a query never ask for a rescale

  const float lazy = WIN || part ? 0.f : PLAZY;
  int32_t skp = 0;             // the next tile's key positions (lanes < 64), stored with the tile's last reads done
  auto fetch = [&](int i, PTile& T) {
    // tile i: list entries [c0, c0 + 64), entry c0 + j the key k0 + j, from j = cut on k0 + j + gap
    const int c0 = i * PK;
    const bool mixed = WIN && c0 < ns && c0 + PK > ns;
    const int k0 = !WIN ? c0 : c0 < ns ? (mixed ? 0 : c0) : kbeg + c0 - ns;
    const int cut = mixed ? ns - c0 : PK, gap = mixed ? kbeg - ns : 0, at = mixed ? c0 : 0;
    // the tile's K and V rows as buffers (base and size in SGPRs): a read past the row's S keys returns zeros, so every
    // staging load is issued unconditionally (keys past a range's end carry the position 0x7FFFFFFF and are masked)
    const int nbytes = min(S - k0, mixed ? kbeg + PK : PK) * 1024;
    const rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(K + (ks + k0) * 512), (short)0, nbytes,
                                                        RSRC_WORD3);
    const rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(V + (ks + k0) * 512), (short)0, nbytes,
                                                        RSRC_WORD3);
    // LDS-direct: instruction r of wave w fills key rows 16 r + 4 w .. + 3 (1 KB, lane l at byte 16 l); lane l
    // fetches the global piece that belongs in its slot
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * r + 4 * w + (lane >> 4), qs = lane & 15;
      const int base = (at + j + (j >= cut ? gap : 0)) * 1024 + g * 256;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)&T.k[(16 * r + 4 * w) * 128],
                                               16, base + 16 * kswz(j, qs), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)&T.v[(16 * r + 4 * w) * 128],
                                               16, base + 16 * vswz(j, qs), 0, 0, 0);
    }
    if (tid < PK) {
      const int key = k0 + at + tid + (tid >= cut ? gap : 0);
      const bool in = key < (WIN && c0 + tid < ns ? sink_end : kend);
      skp = in ? (kpr ? kpr[key] : key) : 0x7FFFFFFF;
    }
    // the loads write T behind the compiler's view of the buffer: its address escapes here
    asm volatile("" ::"s"((uint32_t)(uintptr_t)&T) : "memory");
  };

  if (i0 < i1) {
    fetch(i0, tA);
    if (tid < PK) tA.kp[tid] = skp;
  }
  __syncthreads();
  auto step = [&](int i, const PTile& T, PTile& Nx) {
    if (i + 1 < i1) fetch(i + 1, Nx);
    // ---- S^T = K . Q^T: 2 blocks of 32 keys; score register v of block nb: key 32 nb + 8 (v / 4) + 4 G + v % 4
    // wave priority by phase: of a SIMD's two waves the one in its softmax (2) or P.V (1) goes before one in QK (0)
    __builtin_amdgcn_s_setprio(0);
    f16v sc[2];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int po = 8 * kswz(col, 2 * s + G);   // rows col and 32 + col alike
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const u4v a = *reinterpret_cast<const u4v*>(&T.k[(nb * 32 + col) * 128 + po]);
        const f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        sc[nb] = mfma_bf(a, qb[s], s == 0 ? zero : sc[nb]);
      }
    }
    // ---- mask, scale, online softmax (the lane's 32 keys). No mask when every key of the tile is in range, precedes the
    // workgroup's first query and is a sink or inside the window of its last one.
    const int64_t kfirst = T.kp[0], klast = T.kp[PK - 1];   // ascending; klast is 0x7FFFFFFF if entries are missing
    const bool full = klast <= p0 && (!WIN || kfirst > pl - window || klast < nsink);
    if (!full) {
      const int wlo = WIN ? (int)max((int64_t)qpos - window, (int64_t)INT32_MIN) : INT32_MIN;
      const int nsk = WIN ? (int)nsink : 0;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int kpos = T.kp[nb * 32 + 8 * (v >> 2) + 4 * G + (v & 3)];
          const bool keep = qok & (kpos <= qpos) & ((kpos > wlo) | (kpos < nsk));
          sc[nb][v] = keep ? sc[nb][v] : -INFINITY;
        }
      }
    }
    __builtin_amdgcn_s_setprio(2);
    float tmax = -INFINITY;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int v = 0; v < 16; v += 2) tmax = fmaxf(fmaxf(tmax, sc[nb][v]), sc[nb][v + 1]);
    tmax = max2halves(tmax) * scale_log2;   // scale > 0: the max of the scaled scores
    // a query outgrows its state: its 16-query half of the columns rescales (the branch is wave-uniform)
    const uint64_t grow = __ballot(tmax > m + lazy);
    if (grow) {
      const float mnew = (grow & (col < 16 ? 0x0000FFFF0000FFFFull : 0xFFFF0000FFFF0000ull)) ? fmaxf(m, tmax) : m;
      const float alpha = __builtin_amdgcn_exp2f(m - mnew);
      m = mnew;
      lsum *= alpha;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] *= alpha;
    }
    // ---- O^T += V^T . P^T: 4 steps of 16 keys x 4 blocks of 32 dims. B = the step's 8 own probabilities (keys 4 G ..
    // 4 G + 3 and 8 + 4 G .. + 3), A = V^T (row = dim; the same keys) by two transposed reads: 16-lane group lane / 16
    // reads the key rows' dims 16 ((lane / 16) % 2) .. + 15 of the block
    const int n16 = lane & 15, vrow = 4 * G + (n16 >> 2), vpc = 2 * ((lane >> 4) & 1) + ((n16 >> 1) & 1);
    __builtin_amdgcn_s_setprio(1);
    float psum = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int nb = ks >> 1, v0 = 8 * (ks & 1);
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[nb][v0 + e], scale_log2, -m));   // masked: -inf -> 0
        psum += p[e];
      }
      const u4v b = {bfpk(p[0], p[1]), bfpk(p[2], p[3]), bfpk(p[4], p[5]), bfpk(p[6], p[7])};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int vo = 8 * vswz(vrow, 4 * j + vpc) + 4 * (n16 & 1);   // rows vrow and vrow + 8 alike
        const s4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s4*)const_cast<uint16_t*>(&T.v[(16 * ks + vrow) * 128 + vo]));
        const s4 t1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s4*)const_cast<uint16_t*>(&T.v[(16 * ks + vrow + 8) * 128 + vo]));
        const u4v a = {__builtin_bit_cast(uint32_t, __builtin_shufflevector(t0, t0, 0, 1)),
                       __builtin_bit_cast(uint32_t, __builtin_shufflevector(t0, t0, 2, 3)),
                       __builtin_bit_cast(uint32_t, __builtin_shufflevector(t1, t1, 0, 1)),
                       __builtin_bit_cast(uint32_t, __builtin_shufflevector(t1, t1, 2, 3))};
        o[j] = mfma_bf(a, b, o[j]);
      }
    }
    lsum += psum;
    // the next tile's positions into its buffer, whose last reads (tile i - 1) ended at the previous barrier; the
    // barrier waits for the tile's LDS-direct loads
    if (i + 1 < i1 && tid < PK) Nx.kp[tid] = skp;
    __syncthreads();
  };
  for (int i = i0; i < i1; i += 2) {
    step(i, tA, tB);
    if (i + 1 < i1) step(i + 1, tB, tA);
  }
  // ---- normalise and write: lane holds dims 32 j + 8 c + 4 G + 0..3 of query col. With a key split, the unnormalised
  // partial (o, m, l) of (query, head, split) instead: PPART floats, o relative to 2^m
  const float l = sum2halves(lsum);
  if (!qok) return;
  if (part) {
    float* pp = part + (((q0 + col) * 16 + h) * splits + sp) * PPART;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<f4*>(pp + 32 * j + 8 * c + 4 * G) =
            f4{o[j][4 * c], o[j][4 * c + 1], o[j][4 * c + 2], o[j][4 * c + 3]};
    if (G == 0) { pp[128] = m; pp[129] = l; }
    return;
  }
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  uint16_t* dst = out + ((q0 + col) * 16 + h) * 128 + 4 * G;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const u2v v2 = {bfpk(o[j][4 * c] * inv, o[j][4 * c + 1] * inv), bfpk(o[j][4 * c + 2] * inv, o[j][4 * c + 3] * inv)};
      *reinterpret_cast<u2v*>(dst + 32 * j + 8 * c) = v2;
    }
}

// ---------------------------------------------------------------- key-split merge
// W waves per (query, head). Lanes read the splits' (m, l) in parallel: M = max m_s and L = sum l_s 2^(m_s - M) by
// wave reductions; then lane holds dims 2 lane, 2 lane + 1 and sums o_s 2^(m_s - M) over its wave's splits, the first
// loads in flight during the reductions, the waves' sums added through LDS; out = bf16(O / L) (a split without keys has
// l = 0 and o = 0). Bound: latency, of the partials other XCDs wrote. 4 waves per pair where one would leave most CUs
// without a workgroup (up to 64 queries) and each of the 4 has several partials: whole attention call, 16 queries x 16K
// keys in 64 splits 22.0 -> 16.9 us (calls back to back: the kernels; one call at a time the host takes 34-35 us either
// way), 32 queries 24.9 -> 20.4, 64 queries x 4K keys in 32 splits 21.8 -> 21.1; but 128 queries x 4K in 8 splits 22.4 ->
// 26.3, 64 queries x 16K in 16 splits 30.9 -> 31.9, so these keep one wave.
constexpr int64_t MERGE_WIDE_PAIRS = 1024;
constexpr int MERGE_WIDE_SPLITS = 17;
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int k = 1; k < 64; k <<= 1) x = fmaxf(x, __shfl_xor(x, k, 64));
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int k = 1; k < 64; k <<= 1) x += __shfl_xor(x, k, 64);
  return x;
}
template <int W>   // waves per pair
__global__ void __launch_bounds__(256)
prefill_merge_kernel(const float* __restrict__ part, int64_t pairs, int splits, uint16_t* __restrict__ out) {
  constexpr int N = W == 1 ? 8 : 16;   // partials in flight per wave
  __shared__ float2 red[4][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = w % W;
  const int64_t pr = (int64_t)blockIdx.x * (4 / W) + w / W;
  if (W == 1 && pr >= pairs) return;   // uniform over the wave; with W = 4 the grid is exact
  const float* pp = part + pr * splits * PPART;
  float mv[N];
  float2 av[N];
  const auto load = [&](int s0) {   // splits s0 + W k
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int s = s0 + W * k, sk = s < splits ? s : 0;   // past the last split: a repeat, weighted 0 below
      mv[k] = s < splits ? pp[sk * PPART + 128] : -INFINITY;
      av[k] = *reinterpret_cast<const float2*>(pp + sk * PPART + 2 * lane);
    }
  };
  load(sub);
  float2 ml[PMAXSPLIT / 64];   // (m, l) of splits lane + 64 i
  float M = -INFINITY, Ls = 0.f;
#pragma unroll
  for (int i = 0; i < PMAXSPLIT / 64; ++i) {
    const int s = lane + 64 * i;
    ml[i] = s < splits ? *reinterpret_cast<const float2*>(pp + s * PPART + 128) : make_float2(-INFINITY, 0.f);
    M = fmaxf(M, ml[i].x);
  }
  M = wave_max(M);
#pragma unroll
  for (int i = 0; i < PMAXSPLIT / 64; ++i) Ls += __builtin_amdgcn_exp2f(ml[i].x - M) * ml[i].y;
  Ls = wave_sum(Ls);
  float o0 = 0.f, o1 = 0.f;
  for (int s0 = sub;;) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float wgt = __builtin_amdgcn_exp2f(mv[k] - M);
      o0 += wgt * av[k].x;
      o1 += wgt * av[k].y;
    }
    s0 += W * N;
    if (s0 >= splits) break;   // uniform over the wave
    load(s0);
  }
  if (W > 1) {
    red[w][lane] = make_float2(o0, o1);
    __syncthreads();
    if (sub) return;
#pragma unroll
    for (int k = 1; k < W; ++k) {
      o0 += red[w + k][lane].x;
      o1 += red[w + k][lane].y;
    }
  }
  const float inv = Ls > 0.f ? 1.0f / Ls : 0.f;
  *reinterpret_cast<uint32_t*>(out + pr * 128 + 2 * lane) = bfpk(o0 * inv, o1 * inv);
}

}  // namespace
}  // namespace kv800

using namespace kv800;

extern "C" {

int kv800_hip_rope_rows(const uint16_t* k, const int64_t* pos, int64_t S, const uint16_t* cos_t,
                        const uint16_t* sin_t, int64_t rope_rows, uint16_t* out, void* stream) {
  KV800_REQUIRE(S >= 0, "rope_rows: S < 0");
  if (S == 0) return KV800_OK;
  KV800_REQUIRE(k && pos && cos_t && sin_t && out, "rope_rows: null pointer");
  KV800_REQUIRE(rope_rows > 0, "rope_rows: empty RoPE tables");
  const int64_t n = S * 256;
  hipLaunchKernelGGL(rope_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, k, pos, S,
                     cos_t, sin_t, rope_rows, out);
  return check_launch("rope_rows");
}

int kv800_hip_prefill_split(const uint16_t* q, const int64_t* qsl, const int64_t* qpos0, const uint16_t* K,
                            const uint16_t* V, const int32_t* kp, const int64_t* ksl, const int64_t* tile_off,
                            int64_t R, int64_t ntiles, int64_t T, int64_t window, int64_t nsink, int64_t splits,
                            float* part, int64_t part_floats, uint16_t* out, void* stream) {
  KV800_REQUIRE(R >= 0 && ntiles >= 0 && T >= 0, "prefill: negative R, tile count or query count");
  if (R == 0 || ntiles == 0) return KV800_OK;
  KV800_REQUIRE(q && qsl && qpos0 && K && V && ksl && tile_off && out, "prefill: null pointer");
  KV800_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)K % 16) == 0 && ((uintptr_t)V % 16) == 0 &&
                ((uintptr_t)out % 8) == 0, "prefill: q, K, V need 16-byte and out 8-byte alignment");
  KV800_REQUIRE(window >= 0 && nsink >= 0, "prefill: negative window or sink count");
  KV800_REQUIRE(splits >= 1 && splits <= PMAXSPLIT, "prefill: splits must be in [1, %d]", PMAXSPLIT);
  KV800_REQUIRE(ntiles * 4 * splits < (1ll << 31), "prefill: too many query tiles x splits");
  KV800_REQUIRE(ntiles <= (T + PQ - 1) / PQ + R, "prefill: more query tiles than T queries can hold");
  if (splits > 1) {
    KV800_REQUIRE(part && ((uintptr_t)part % 16) == 0, "prefill: a key split needs a 16-byte aligned part buffer");
    KV800_REQUIRE(part_floats >= T * 16 * splits * PPART, "prefill: part holds %lld floats, the split needs %lld",
                  (long long)part_floats, (long long)(T * 16 * splits * PPART));
  }
  const float scale_log2 = 0.088388347648318440f * 1.4426950408889634f;   // 128^-0.5 * log2(e)
  hipLaunchKernelGGL(window > 0 ? prefill_kernel<true> : prefill_kernel<false>, dim3((unsigned)(ntiles * 4 * splits)),
                     dim3(256), 0, (hipStream_t)stream, q, qsl, qpos0, K, V, kp, ksl, tile_off, R, window, nsink,
                     scale_log2, out, (int)splits, splits > 1 ? part : (float*)nullptr);
  int rc = check_launch("prefill");
  if (rc != KV800_OK || splits == 1 || T == 0) return rc;
  const int64_t pairs = T * 16;
  const bool wide = pairs <= MERGE_WIDE_PAIRS && splits >= MERGE_WIDE_SPLITS;
  hipLaunchKernelGGL(wide ? prefill_merge_kernel<4> : prefill_merge_kernel<1>,
                     dim3((unsigned)(wide ? pairs : (pairs + 3) / 4)), dim3(256), 0, (hipStream_t)stream, part, pairs,
                     (int)splits, out);
  return check_launch("prefill_merge");
}

int kv800_hip_prefill(const uint16_t* q, const int64_t* qsl, const int64_t* qpos0, const uint16_t* K,
                      const uint16_t* V, const int32_t* kp, const int64_t* ksl, const int64_t* tile_off, int64_t R,
                      int64_t ntiles, int64_t window, int64_t nsink, uint16_t* out, void* stream) {
  KV800_REQUIRE(ntiles < (1ll << 29), "prefill: too many query tiles");
  return kv800_hip_prefill_split(q, qsl, qpos0, K, V, kp, ksl, tile_off, R, ntiles, ntiles * PQ, window, nsink, 1,
                                 nullptr, 0, out, stream);
}

}  // extern "C"
