// Split-K paged decode attention on the matrix cores (gfx950 MFMA), for
// 16-bit K/V pages with head_dim 64, 128 or 256 — the hot configurations of HELM's
// perform_streaming_attention (helm/runtime/kv_cache.py:468-555 masked
// online-softmax loop, :562-568 Path 1, :584-662 Path 3) and of the batched
// decode of _decode_batched (helm/runtime/kv_offload.py:152-174).
//
// Decode attention is bound by HBM: every K/V byte is read once.  The matrix
// cores are used here only to take the arithmetic off the vector ALU, so that
// the ALU work per 16-token block stays far below the time its 8 KiB take to
// arrive, at any GQA group size up to 16 query rows per KV head.
//
// Work decomposition: grid.x = split (<= kMfmaMaxPps pages), grid.y = KV head
// + Hkv * row tile, grid.z = sequence; NW waves per workgroup, wave w takes
// the 16-token blocks w, w+NW, ... of the split.  Per block, with q4 = lane/16 and
// n = lane%16:
//   * scores: S^T = K . Q^T with four 16x16x32 MFMAs (k = head dims).  Lane l
//     loads K of token tau(n) = 4*(n%4) + n/4 at dims chunk 4i + q4 (16 B, i =
//     0..3); Q^T's operand holds query row n at the same chunks.  The result
//     gives lane l the scores of query row n for tokens 4r + q4 (r = 0..3).
//   * online softmax per row on those four scores, in natural-log units as
//     HELM's loop; the running max is refreshed (wave-uniformly) only when a
//     score exceeds it by more than kMfmaSlack, otherwise the stale max keeps
//     every weight <= e^kMfmaSlack and O, L exact relative to it.
//   * O += P . V with eight 16x16x32 MFMAs (one per dim e of each lane's
//     8-dim column group): P's operand is {hi(p_r), lo(p_r)} — each weight
//     split into two 16-bit values whose sum carries 16 mantissa bits — and
//     V's operand the same four tokens 4j + q4 twice, so one MFMA adds
//     (hi + lo) . v.  Lane (q4, n) loads V rows 4j + q4 at dims 8n..8n+7: a
//     wave load is 1 KiB contiguous.  Products are exact and accumulate in
//     fp32.
// (Written for D = 128; D = 64 halves the K chunks and the dims a lane holds
// of a V row to four, D = 256 doubles both, the V row's halves apart: VRow.
// Against the vector-ALU kernel that served them before: f16 D = 64, four
// sequences of 3k-16k tokens, 45.6 -> 17.4 us; bf16 D = 256, 8,000 tokens
// soft-capped under a window mask, 37.9 -> 18.7 us.  Their weights' parts and
// scale: weight_parts, weight_shift.)
// No data moves between lanes in the loop; the split's per-wave states meet in
// LDS; the shared split epilogue (attn_kernel.h) merges the waves and then
// the splits.
#pragma once

#include <type_traits>

#include "attn_kernel.h"

namespace helm {

constexpr int kMfmaRows = 16;     // query rows per tile (MFMA M dimension)
// pages per split: page records live one per lane, in two windows of 64
constexpr int kMfmaMaxPps = 128;
constexpr int kMfmaMaxSplits = 4096;
constexpr float kMfmaSlack = 8.f;
// Register buffers of the block pipeline: with two, one block's loads are in
// flight while the wave computes the other (8 KiB per wave, 32 KiB per CU).
// Measured on the Qwen3-8B 32k call: 2 buffers 26.4-26.5 us, 3 buffers
// 26.7-27.0, 4 buffers 27.2-27.4 per call.
#ifndef HELM_MFMA_NBUF
#define HELM_MFMA_NBUF 2
#endif
// D = 64's blocks are half as large: two in flight (f16, four sequences of
// 3k-16k tokens, 32 / 8 heads: 2 buffers 18.0 us, 3 17.3, 4 17.5, 6 17.9; one of
// 700, 12 heads: 7.2, 7.1, 7.3, 7.7).
constexpr int mfma_bufs(int D) { return D == 64 ? 3 : HELM_MFMA_NBUF; }

// 16-bit parts a weight takes into P . V (the vector-ALU kernel multiplied by
// the fp32 weight).  f16: hi + lo, 22 bits.  bf16: hi + lo are 16 bits and, at
// the head dims that had the vector-ALU kernel, a third part holds the last
// eight, so that the fp32 weight enters exactly.  Without it a chunk's outputs
// were 1.7e-6 off before their rounding, with it 5e-7, as far as fp32 sums in
// two orders are.  It costs a decode call nothing and a chunk a third more
// matrix work: D = 256, 512 tokens over 4,700, soft-capped under a window mask,
// 99 -> 110 us; D = 64, 512 over 16k, 125 -> 146.
template <typename T>
constexpr int weight_parts(int D) { return std::is_same<T, bf16_t>::value && D != 128 ? 3 : 2; }

// f16 parts have a floor: what is below 2^-25 is lost.  At head dims 64 and 256
// (the vector-ALU kernel had no floor) f16 weights are taken times 2^9 and the
// row's reference max is refreshed once a weight passes 2^6, together below
// f16's 2^16: the floor lies at 2^-34 of the largest weight, where a million
// tokens at the floor weigh 2^-14 of the row.  (One key 17 nats above 65,536
// others, with the floor at 2^-25: the others, 2.7e-3 of the row, counted in its
// sum and not in its output.)  Chunk of 777 over 2,777, 14 / 2 heads, D = 64:
// 29.4 us without, 29.3 with; 2^11 and a refresh at 2^4 30.0.
template <typename T>
constexpr int weight_shift(int D) { return std::is_same<T, f16_t>::value && D != 128 ? 9 : 0; }
// the refresh threshold that goes with it, in base-2 units / in natural units
constexpr float chunk_slack(int shift) { return shift ? 6.f : 8.f; }
constexpr float decode_slack(int shift) { return shift ? 4.1588831f : kMfmaSlack; }   // 6 ln 2

// kFeatMask16: the mask is 16-bit (bf16 / fp16); the decode and 32-row chunk
// kernels read it at that width (the 16-row chunk kernel at run time)
enum MfmaFeat { kFeatMask = 1, kFeatCap = 2, kFeatCausal = 4, kFeatMask16 = 8 };

typedef __bf16 mf_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 mf_f16x8 __attribute__((ext_vector_type(8)));
typedef float mf_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t mf_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t mf_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t mf_u32x8 __attribute__((ext_vector_type(8)));

// One lane's share of a V row in the decode kernel, D / 16 dims in D / 32
// words: lane n of a row's 16 holds dims 4n .. 4n + 3 (D = 64), 8n .. 8n + 7
// (128) or those of both halves of the row (256: 8n .. and 128 + 8n ..), so
// every load instruction covers whole rows contiguously.
template <int D> struct VRow;
template <> struct VRow<64> { typedef mf_u32x2 type; };
template <> struct VRow<128> { typedef mf_u32x4 type; };
template <> struct VRow<256> { typedef mf_u32x8 type; };

// Low / high 16-bit halves of two words packed into one: (a.lo, b.lo), (a.hi, b.hi).
__device__ __forceinline__ uint32_t pack_lo(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

template <typename T> struct MfmaOps;

template <> struct MfmaOps<bf16_t> {
  __device__ static __forceinline__ mf_f32x4 mma(mf_u32x4 a, mf_u32x4 b, mf_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_bf16x8, a),
                                                   __builtin_bit_cast(mf_bf16x8, b), c, 0, 0, 0);
  }
  // Two weights as packed 16-bit hi and lo parts, hi = RNE(w), lo = RNE(w - hi)
  // (v_cvt_pk_bf16_f32 rounds to nearest even); element 0 in the low half.
  __device__ static __forceinline__ void split2(float w0, float w1, uint32_t& hi,
                                                uint32_t& lo) {
    hi = pk(w0, w1);
    lo = pk(w0 - __uint_as_float(hi << 16), w1 - __uint_as_float(hi & 0xffff0000u));
  }
  // The leading 8 bits of two weights packed into one word; what they leave of
  // each (exact) stays in w0 and w1.
  __device__ static __forceinline__ uint32_t lead(float& w0, float& w1) {
    const uint32_t u0 = __float_as_uint(w0), u1 = __float_as_uint(w1);
    w0 -= __uint_as_float(u0 & 0xffff0000u);
    w1 -= __uint_as_float(u1 & 0xffff0000u);
    return pack_hi(u0, u1);
  }
  // Two weights as three such parts: hi + mid + lo is the fp32 weight exactly.
  __device__ static __forceinline__ void split3(float w0, float w1, uint32_t& hi, uint32_t& mid,
                                                uint32_t& lo) {
    hi = lead(w0, w1);
    mid = lead(w0, w1);
    lo = pack_hi(__float_as_uint(w0), __float_as_uint(w1));
  }
  __device__ static __forceinline__ uint32_t pk(float a, float b) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, bf2));
  }
  // eight 16-bit ones (an MFMA operand)
  __device__ static __forceinline__ mf_u32x4 ones8() {
    return mf_u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  }
};

template <> struct MfmaOps<f16_t> {
  __device__ static __forceinline__ mf_f32x4 mma(mf_u32x4 a, mf_u32x4 b, mf_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mf_f16x8, a),
                                                  __builtin_bit_cast(mf_f16x8, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pk(float a, float b) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, h2));
  }
  // eight 16-bit ones (an MFMA operand)
  __device__ static __forceinline__ mf_u32x4 ones8() {
    return mf_u32x4{0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
  }
  // hi = RNE(w), lo = RNE(w - hi) in fp16, packed two per word (v_cvt_pk_f16_f32)
  __device__ static __forceinline__ void split2(float w0, float w1, uint32_t& hi,
                                                uint32_t& lo) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    const h2 h = __builtin_convertvector((f2){w0, w1}, h2);
    hi = __builtin_bit_cast(uint32_t, h);
    const f2 back = __builtin_convertvector(h, f2);
    lo = pk(w0 - back[0], w1 - back[1]);
  }
  // The same with w - hi (exact) by v_fma_mix_f32, which reads the f16 half in
  // place: one conversion less per weight (D = 64 chunk of 777 over 2,777,
  // 14 / 2 heads: 30.1 -> 29.2 us).  Not in the decode kernel, where the asm
  // holds the scheduler back (D = 128, 2,048 tokens: 8.07 us, with it 8.12).
  __device__ static __forceinline__ void split2_mix(float w0, float w1, uint32_t& hi,
                                                    uint32_t& lo) {
    hi = pk(w0, w1);
    float r0, r1;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(hi), "v"(w0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=v"(r1)
        : "v"(hi), "v"(w1));
    lo = pk(r0, r1);
  }
};

// 16-byte buffer load with the non-temporal hint: K/V are read exactly once.
__device__ __forceinline__ mf_u32x4 buf_load16_nt(__amdgpu_buffer_rsrc_t r, int off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2);
  return mf_u32x4{v[0], v[1], v[2], v[3]};
}

// A lane's share of a V row (VRow) at byte offset row of the resource.
template <int D>
__device__ __forceinline__ typename VRow<D>::type buf_load_vrow_nt(__amdgpu_buffer_rsrc_t r,
                                                                   int row, int n) {
  if constexpr (D == 64) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, row + 8 * n, 0, 2);
    return mf_u32x2{v[0], v[1]};
  } else if constexpr (D == 128) {
    return buf_load16_nt(r, row + 16 * n);
  } else {
    const mf_u32x4 a = buf_load16_nt(r, row + 16 * n);
    const mf_u32x4 b = buf_load16_nt(r, row + 256 + 16 * n);
    return mf_u32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  }
}

// 16 bytes at any alignment (one load: the target takes unaligned vector loads).
__device__ __forceinline__ mf_u32x4 load16_any(const char* p) {
  struct __attribute__((packed)) Any { mf_u32x4 v; };
  return reinterpret_cast<const Any*>(p)->v;
}

// x = cap tanh(x k) with k = scale / cap and cap in the caller's log units, for
// the N scores of a lane.  Logits far below the cap (|x k| <= 2^-2.5 for every
// score of the wave, |logit| <= 8.8 at a cap of 50: the usual case) take the
// odd Taylor polynomial of tanh through y^7, whose first left-out term is below
// 2.1e-8 of the result there, a third of an fp32 half ulp; k and cap sit in its
// coefficients (x times a polynomial in x^2: five instructions a score), which
// holds while their powers stay in fp32's range: |k| in [2^-20, 2^8], far around
// every head dim and cap in use.  Any other step takes tanhf (for every step it
// had cost as much as the softmax: bf16 chunk of 512 over 8,192, 32 / 8 heads,
// 4,096-token window, capped: 236 us, now 135).
template <int N>
__device__ __forceinline__ void softcap_scores(float (&x)[N], float k, float cap) {
  float top = fabsf(x[0]);
#pragma unroll
  for (int r = 1; r < N; ++r) top = fmaxf(top, fabsf(x[r]));
  const float ak = fabsf(k);
  const bool in_range = ak >= 0x1p-20f && ak <= 0x1p8f;
  if (__builtin_expect(in_range && !__builtin_amdgcn_ballot_w64(!(top * ak <= 0.1767767f)), 1)) {
    const float kk = k * k, a0 = k * cap;
    const float a1 = a0 * kk * (-1.f / 3.f), a2 = a0 * kk * kk * (2.f / 15.f);
    const float a3 = a0 * kk * kk * kk * (-17.f / 315.f);
#pragma unroll
    for (int r = 0; r < N; ++r) {
      const float z = x[r] * x[r];
      x[r] *= fmaf(z, fmaf(z, fmaf(z, a3, a2), a1), a0);
    }
  } else {
#pragma unroll
    for (int r = 0; r < N; ++r) x[r] = tanhf(x[r] * k) * cap;
  }
}

// LDS transpose read of 16-bit elements (ds_read_b64_tr_b16): within each
// 16-lane group, lane c = 4a + b receives element b of the 8 bytes that
// lanes a, a + 4, a + 8 and a + 12 address, in that order.
__device__ __forceinline__ uint2 ld_tr16(const char* lds_addr) {
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) v4i16*)(lds_addr));
  return __builtin_bit_cast(uint2, r);
}

// ---- page records held one per lane ------------------------------------------
// Lane i holds the record of page pg0 + i of the split; a block reads its
// page's record with v_readlane (a uniform lane index), so no memory access
// sits between a block's turn and the issue of its loads.
struct PoolLanes {
  int slot;
};
struct DescLanes {
  uint32_t klo, khi, vlo, vhi;
  int used, tok_off, head_stride;
};

// Issued before the sequence length is known: the pool's table row is read
// up to its declared width, so the first K/V loads wait for one memory trip.
__device__ __forceinline__ PoolLanes lane_pages(const PoolSrc& s, int b, int pg0, int lane) {
  PoolLanes L;
  L.slot = s.max_pages > 0
               ? s.table[(int64_t)b * s.table_stride + min(pg0 + lane, s.max_pages - 1)]
               : 0;
  return L;
}
__device__ __forceinline__ DescLanes lane_pages(const DescSrc& s, int b, int pg0, int lane) {
  const helm_page* base = s.base(b);
  const int cnt = s.n_pages(b);
  helm_page d{};
  if (cnt > 0) d = base[max(0, min(pg0 + lane, cnt - 1))];
  DescLanes L;
  L.klo = static_cast<uint32_t>(d.k);
  L.khi = static_cast<uint32_t>(d.k >> 32);
  L.vlo = static_cast<uint32_t>(d.v);
  L.vhi = static_cast<uint32_t>(d.v >> 32);
  L.used = s.used_of(d, b);
  L.tok_off = d.tok_off;
  L.head_stride = d.head_stride;
  return L;
}

// Page i of the split (uniform): head-hk K / V bases, used tokens, token offset.
__device__ __forceinline__ PageView lane_page_view(const PoolSrc& s, const PoolLanes& L, int b,
                                                   int pg, int i, int hk) {
  const int slot = __builtin_amdgcn_readlane(L.slot, i);
  const int T = sload(s.seq_lens + b);
  PageView pv;
  const int64_t off = (int64_t)slot * s.slot_stride_b + hk * s.head_stride_b;
  pv.k = s.k_pool + off;
  pv.v = s.v_pool + off;
  pv.tok_off = pg * s.page_size;
  pv.used = min(s.page_size, T - pv.tok_off);
  pv.head_stride_b = 0;
  return pv;
}
__device__ __forceinline__ PageView lane_page_view(const DescSrc& s, const DescLanes& L, int,
                                                   int, int i, int hk) {
  const uint64_t k = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(L.khi, i) << 32) |
                     (uint32_t)__builtin_amdgcn_readlane(L.klo, i);
  const uint64_t v = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(L.vhi, i) << 32) |
                     (uint32_t)__builtin_amdgcn_readlane(L.vlo, i);
  const int hs = __builtin_amdgcn_readlane(L.head_stride, i);
  // (head strides are >= 0: one 32 x 32 -> 64-bit product)
  const uint64_t off = (uint64_t)(uint32_t)hs * (uint32_t)(hk * s.elem_bytes);
  PageView pv;
  pv.k = reinterpret_cast<const char*>(k) + off;
  pv.v = reinterpret_cast<const char*>(v) + off;
  pv.used = __builtin_amdgcn_readlane(L.used, i);
  pv.tok_off = __builtin_amdgcn_readlane(L.tok_off, i);
  pv.head_stride_b = 0;
  return pv;
}

// The page `pg` (per lane) whose record this lane holds: head-hk K / V bases,
// used tokens, token offset.
__device__ __forceinline__ PageView lane_own_view(const PoolSrc& s, const PoolLanes& L, int b,
                                                  int pg, int hk) {
  PageView pv;
  const int64_t off = (int64_t)L.slot * s.slot_stride_b + hk * s.head_stride_b;
  pv.k = s.k_pool + off;
  pv.v = s.v_pool + off;
  pv.tok_off = pg * s.page_size;
  pv.used = min(s.page_size, sload(s.seq_lens + b) - pv.tok_off);
  pv.head_stride_b = 0;
  return pv;
}
__device__ __forceinline__ PageView lane_own_view(const DescSrc& s, const DescLanes& L, int, int,
                                                  int hk) {
  const uint64_t off = (uint64_t)(uint32_t)L.head_stride * (uint32_t)(hk * s.elem_bytes);
  PageView pv;
  pv.k = reinterpret_cast<const char*>((((uint64_t)L.khi << 32) | L.klo) + off);
  pv.v = reinterpret_cast<const char*>((((uint64_t)L.vhi << 32) | L.vlo) + off);
  pv.used = L.used;
  pv.tok_off = L.tok_off;
  pv.head_stride_b = 0;
  return pv;
}

// One 16-token block of the online-softmax recurrence on the matrix cores:
// k / v are the block's K and V operands (K token tau(n) at dim chunks
// q4 + 4i; V tokens q4 + 4j at dims 8n..8n+7), mk the additive mask of the
// lane's row for tokens 4r + q4, ntok the block's valid tokens, tok0 the
// HELM token cursor of its first token.  Updates the row max m, this lane's
// share of the row sum, and O (rows 4 q4 + r, dims 8n + e).
// q . k of the lane's row n for tokens 4r + q4 of a block (K operand k).
template <class Ops, int NK>
__device__ __forceinline__ mf_f32x4 mfma_qk(const mf_u32x4 (&k)[NK], const mf_u32x4 (&qop)[NK]) {
  mf_f32x4 sc = mf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NK; ++i) sc = Ops::mma(k[i], qop[i], sc);
  return sc;
}

// Logits of those four tokens: scale, soft-cap, additive mask, causal limit
// (tokens past s_vis, the row's last visible token), and -inf past the
// block's ntok valid tokens.
template <bool kMask, bool kCap, bool kCausal>
__device__ __forceinline__ void mfma_logits(mf_f32x4 sc, const float (&mk)[4], int ntok, int tok0,
                                            float scale, float cap, float inv_cap, int s_vis,
                                            int q4, float (&x)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) x[r] = kCap ? sc[r] : sc[r] * scale;
  if constexpr (kCap) softcap_scores<4>(x, scale * inv_cap, cap);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if constexpr (kMask) x[r] += mk[r];
    if constexpr (kCausal)
      if (tok0 + 4 * r + q4 > s_vis) x[r] = -INFINITY;
  }
  if (ntok < kBlockTok) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * r + q4 >= ntok) x[r] = -INFINITY;
  }
}

// The lazy online-softmax reference update for a block max bm: when bm
// exceeds the row max by more than the slack anywhere in the wave, the row
// max is refreshed and l and the O rows rescaled.
template <int SHIFT, int NO>
__device__ __forceinline__ void mfma_refresh_max(float bm, float& m, float& lsum,
                                                 mf_f32x4 (&o)[NO], int q4) {
  if (__builtin_amdgcn_ballot_w64(bm > m + decode_slack(SHIFT))) {
    // refresh the row max (uniform across the row's four lanes)
    float rm = fmaxf(bm, __shfl_xor(bm, 16, 64));
    rm = fmaxf(rm, __shfl_xor(rm, 32, 64));
    const float mn = fmaxf(m, rm);
    const float a = fexp(m - ((mn == -INFINITY) ? 0.f : mn));
    lsum *= a;
    m = mn;
    // O rows of this lane are 4*q4 + r: fetch their factors
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float ar = __shfl(a, 4 * q4 + r, 64);
#pragma unroll
      for (int e = 0; e < NO; ++e) o[e][r] *= ar;
    }
  }
}

// Weights exp(x - m) of the four tokens into l and, as PARTS 16-bit parts (2:
// hi + lo, 3: all 24 bits of a bf16 call's weights), P . V into O (V operand v:
// tokens q4 + 4j at the lane's dims of the row).
template <int PARTS, int SHIFT, class Ops, class V, int NO>
__device__ __forceinline__ void mfma_pv(const float (&x)[4], const V (&v)[4], float m,
                                        float& lsum, mf_f32x4 (&o)[NO]) {
  const float base = (m == -INFINITY) ? 0.f : m;
  float wt[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    wt[r] = fexp(x[r] - base);
    if constexpr (SHIFT) wt[r] *= static_cast<float>(1 << SHIFT);
    if constexpr (!(SHIFT || PARTS == 3)) lsum += wt[r];
  }
  // (the block's sum first: weights below an ulp of the row's sum add up)
  if constexpr (SHIFT || PARTS == 3) lsum += (wt[0] + wt[1]) + (wt[2] + wt[3]);
  uint32_t h01, l01, h23, l23, e01 = 0u, e23 = 0u;
  if constexpr (PARTS == 3) {
    Ops::split3(wt[0], wt[1], h01, l01, e01);
    Ops::split3(wt[2], wt[3], h23, l23, e23);
  } else {
    Ops::split2(wt[0], wt[1], h01, l01);
    Ops::split2(wt[2], wt[3], h23, l23);
  }
  const mf_u32x4 pop = mf_u32x4{h01, h23, l01, l23};
#pragma unroll
  for (int w = 0; w < NO / 2; ++w) {
    const uint32_t a01 = pack_lo(v[0][w], v[1][w]);
    const uint32_t a23 = pack_lo(v[2][w], v[3][w]);
    const uint32_t b01 = pack_hi(v[0][w], v[1][w]);
    const uint32_t b23 = pack_hi(v[2][w], v[3][w]);
    o[2 * w] = Ops::mma(pop, mf_u32x4{a01, a23, a01, a23}, o[2 * w]);
    o[2 * w + 1] = Ops::mma(pop, mf_u32x4{b01, b23, b01, b23}, o[2 * w + 1]);
    if constexpr (PARTS == 3) {
      // (the same shape with half of P zero: a 16x16x16 product right after the
      // 16x16x32 one has read O before its result was there)
      const mf_u32x4 pex = mf_u32x4{e01, e23, 0u, 0u};
      o[2 * w] = Ops::mma(pex, mf_u32x4{a01, a23, a01, a23}, o[2 * w]);
      o[2 * w + 1] = Ops::mma(pex, mf_u32x4{b01, b23, b01, b23}, o[2 * w + 1]);
    }
  }
}

// One 16-token block of the recurrence: q . k, logits, max refresh, P . V.
template <class Ops, int PARTS, int SHIFT, bool kMask, bool kCap, bool kCausal, class V, int NK,
          int NO>
__device__ __forceinline__ void mfma_block_step(const mf_u32x4 (&k)[NK], const V (&v)[4],
                                                const float (&mk)[4], int ntok, int tok0,
                                                const mf_u32x4 (&qop)[NK], float& m, float& lsum,
                                                mf_f32x4 (&o)[NO], float scale, float cap,
                                                float inv_cap, int s_vis, int q4) {
  float x[4];
  mfma_logits<kMask, kCap, kCausal>(mfma_qk<Ops>(k, qop), mk, ntok, tok0, scale, cap, inv_cap,
                                    s_vis, q4, x);
  mfma_refresh_max<SHIFT>(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), m, lsum, o, q4);
  mfma_pv<PARTS, SHIFT, Ops>(x, v, m, lsum, o);
}

// True where any O of the wave is NaN.
template <int NO, class O>
__device__ __forceinline__ bool any_nan(const O (&o)[NO]) {
  float t = 0.f;
#pragma unroll
  for (int e = 0; e < NO; ++e)
#pragma unroll
    for (int r = 0; r < (int)(sizeof(O) / 4); ++r) t = fmaf(o[e][r], 0.f, t);
  return __builtin_amdgcn_ballot_w64(!(t == 0.f)) != 0;
}

// The arguments of a kernel (AttnParams p, Src src), read again from where the
// launch put them: a rare path that goes through here keeps none of them in
// registers beside the loop before it.
template <class Src>
struct KernelArgs {
  const char* base;
  __device__ __forceinline__ KernelArgs() {
    auto ka = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
    base = (const char*)ka;
  }
  __device__ __forceinline__ const AttnParams& p() const {
    return *reinterpret_cast<const AttnParams*>(base);
  }
  __device__ __forceinline__ const Src& src() const {
    constexpr size_t at = (sizeof(AttnParams) + alignof(Src) - 1) / alignof(Src) * alignof(Src);
    return *reinterpret_cast<const Src*>(base + at);
  }
};

// Infinite values.  A weight times an infinite value is infinite, but the sum
// of its 16-bit parts' products is NaN where a part is zero or of the other
// sign (1.0 has hi = 1, lo = 0).  At the head dims that had the vector-ALU kernel
// a wave whose O holds a NaN at the end of its walk comes here, a rare path
// kept short and out of the loop (a second walk with parts above zero instead
// slowed the chunks by 2 to 7% and the soft-capped decode by 8%): it looks
// through V of the wave's blocks (blk, blk + step, ...) again and, per token
// with an infinity or NaN, takes the weight of each row in fp32, from the same
// logit and the row's final max m (natural units, row (g, s) in this lane), and
// hands it with the token's V row to add, which corrects O with the fp32 product.
template <typename T, class Src, int FEAT, int D, class Add>
__device__ __forceinline__ void infinite_values(const AttnParams& p, const Src& src, int b, int hk,
                                                int pg0, int blk, int nblk, int step, int g, int s,
                                                float m, int lane, Add&& add) {
  constexpr int kRow = 2 * D;
  constexpr uint32_t kExp = std::is_same<T, bf16_t>::value ? 0x7f80u : 0x7c00u;
  const int h = hk * p.G + g;
  const char* qp = reinterpret_cast<const char*>(p.q) + ((int64_t)(b * p.Hq + h) * p.S + s) * kRow;
  const float base = (m == -INFINITY) ? 0.f : m;
#pragma unroll 1
  for (; blk < nblk; blk += step) {
    const int pi = blk / p.bpp;
    const int tok_in = (blk - pi * p.bpp) * kBlockTok;
    const PageView pv = src.page(b, pg0 + pi, hk);
    const int ntok = sclamp(pv.used - tok_in, 0, kBlockTok);
    const char* vb = pv.v + tok_in * kRow;
    const auto rv = make_rsrc(vb, ntok * kRow);
    bool bad = false;
#pragma unroll
    for (int c = 0; c < kBlockTok * kRow / 1024; ++c) {
      const mf_u32x4 v = buf_load16_nt(rv, 1024 * c + 16 * lane);   // (zero past the tokens)
#pragma unroll
      for (int w = 0; w < 4; ++w)
        bad = bad || (v[w] & kExp) == kExp || ((v[w] >> 16) & kExp) == kExp;
    }
    if (!__builtin_amdgcn_ballot_w64(bad)) continue;
#pragma unroll 1
    for (int t = 0; t < ntok; ++t) {
      const char* kp = pv.k + (tok_in + t) * kRow;
      float x = 0.f;
#pragma unroll 1
      for (int i = 0; i < kRow; i += 4)
        x = dot2<T>(*reinterpret_cast<const uint32_t*>(qp + i),
                    *reinterpret_cast<const uint32_t*>(kp + i), x);
      x *= p.scale;
      // (tanh to 1e-6: only whether the weight is zero matters)
      if constexpr ((FEAT & kFeatCap) != 0)
        x = (1.f - 2.f / (fexp(2.f * x / p.softcap) + 1.f)) * p.softcap;
      const int tok = pv.tok_off + tok_in + t;
      if constexpr ((FEAT & kFeatMask) != 0) x += mask_row(p, b, h, s)[tok];
      if constexpr ((FEAT & kFeatCausal) != 0)
        if (tok > s + p.causal - 1) x = -INFINITY;
      add(fexp(x - base), reinterpret_cast<const uint16_t*>(vb + t * kRow));
    }
  }
}

// O with the product of weight w and value bits v: left alone where it or v is
// finite; the NaN of the parts' products (any but `done`) gives way to w v.
template <typename T>
__device__ __forceinline__ float with_infinite(float o, float w, uint16_t v) {
  constexpr uint32_t kDone = 0x7fc0dead;   // a NaN that stays
  Raw<2> raw;
  raw.w[0] = v;
  const float term = w * elem_f32<T>(raw, 0);
  if (fabsf(o) < INFINITY || fabsf(elem_f32<T>(raw, 0)) < INFINITY) return o;
  const float sum = (o != o && __float_as_uint(o) != kDone) ? term : o + term;
  return sum != sum ? __uint_as_float(kDone) : sum;
}

template <class Src> struct LanesOf;
template <> struct LanesOf<PoolSrc> { using type = PoolLanes; };
template <> struct LanesOf<DescSrc> { using type = DescLanes; };

// The decode kernel of head dim D (64, 128 or 256); the entry points below
// launch it.
template <typename T, class Src, int FEAT, int NW, int D>
__device__ __forceinline__ void decode_mfma_body(const AttnParams& p, const Src& src) {
  using Ops = MfmaOps<T>;
  using V = typename VRow<D>::type;
  constexpr int NT = 64 * NW;
  constexpr int kRow = 2 * D;     // bytes per token row
  constexpr int NK = D / 32;      // K (and Q) operand chunks of a lane
  constexpr int NO = D / 16;      // O column groups (MFMAs of P . V per block)
  constexpr bool kMask = (FEAT & kFeatMask) != 0;
  constexpr bool kCap = (FEAT & kFeatCap) != 0;
  constexpr bool kCausal = (FEAT & kFeatCausal) != 0;
  constexpr bool kMask16 = (FEAT & kFeatMask16) != 0;

  __shared__ Smem<NW, kMfmaRows, D> sm;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int q4 = lane >> 4;
  const int n = lane & 15;
  // profiling stamps of this workgroup (helm_profile_workgroup_stamps)
  uint64_t* const stp =
      p.stamps ? p.stamps + 4 * (blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z))
               : nullptr;
  if (stp && tid == 0) {
    stp[0] = stamp_now();
    stp[3] = stamp_place();
  }

  int split_local = blockIdx.x, b = blockIdx.z;
  if (src.compact) {
    // the last sequence whose first split is at or before blockIdx.x
    int bb = 0;
#pragma unroll
    for (int j = 1; j < kSeqArgs; ++j)
      if (j < src.n_seq && (int)blockIdx.x >= src.seq_split0[j]) bb = j;
    b = bb;
    split_local = blockIdx.x - src.seq_split0[bb];
  }
  const int hk = blockIdx.y % p.Hkv;
  // the waves share one 16-row tile and split its blocks (query chunks with
  // more tiles run in chunk_mfma_kernel)
  const int qt = blockIdx.y / p.Hkv;
  const int tile = (b * p.Hkv + hk) * p.n_qtiles + qt;
  const int S = p.S;
  const int G = p.G;
  const int r0 = qt * kMfmaRows;
  const int nrows = min(kMfmaRows, G * S - r0);

  // ---- loads that need no sequence length: page records, query rows --------
  // (pg0 below equals this whenever the workgroup has pages to process)
  const typename LanesOf<Src>::type lanes =
      lane_pages(src, b, p.lo + split_local * p.pps, lane);
  // a split of more than 64 pages: the records of its pages 64 .. 127
  typename LanesOf<Src>::type lanes_hi{};
  if (p.pps > 64 && !(D == 128 && p.dyn)) lanes_hi = lane_pages(src, b, p.lo + split_local * p.pps + 64, lane);
  // ---- query operand: row n of the tile at dim chunks 4i + q4 ---------------
  const bool row_ok = n < nrows;
  const int rr = r0 + (row_ok ? n : 0);
  const RowCoord rc = row_coord(rr, G);
  const int g_row = rc.g;
  const int s_row = rc.s;
  // causal: query position s sees tokens 0 .. s + causal - 1
  const int s_vis = s_row + (kCausal ? p.causal - 1 : 0);
  mf_u32x4 qop[NK];
  {
    const int h = hk * G + g_row;
    const char* qp = reinterpret_cast<const char*>(p.q) +
                     ((int64_t)(b * p.Hq + h) * S + s_row) * kRow;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(qp + 16 * (4 * i + q4));
      qop[i] = row_ok ? mf_u32x4{v.x, v.y, v.z, v.w} : mf_u32x4{0u, 0u, 0u, 0u};
    }
  }
  // ---- this workgroup's page range -------------------------------------------
  const int np = src.n_pages(b);
  const int lo = min(p.lo, np);
  const int hi = min(p.hi, np);
  const int nsplit_launch = (hi - lo + p.pps - 1) / p.pps;
  const int total = p.total_splits > 0 ? p.total_splits : nsplit_launch;
  // split 0 publishes the tile's split count; a tile without pages gets
  // zeros (HELM kv_cache.py:441-442): from split 0 in fused mode, from
  // merge_splits_kernel otherwise
  if (split_local == 0 && tid == 0) p.counts[tile] = total;
  const bool active = total > 0 && split_local < nsplit_launch;
  if (!active) {
    if (total == 0 && p.fused && split_local == 0) {
      for (int idx = tid; idx < nrows * D; idx += NT) {
        const int zr = r0 + idx / D;
        const RowCoord rc = row_coord(zr, G);
        const int h = hk * G + rc.g, s = rc.s;
        const int64_t o_off = ((int64_t)(b * p.Hq + h) * S + s) * D + idx % D;
        store_elem<T>(reinterpret_cast<char*>(p.out) + o_off * 2, 0.f);
      }
    }
    if (stp && tid == 0) stp[1] = stp[2] = stamp_now();
    return;
  }
  const int split = p.split_base + split_local;
  const int pg0 = lo + split_local * p.pps;
  const int npg = min(pg0 + p.pps, hi) - pg0;  // 1..kMfmaMaxPps
  if constexpr (D == 128 && std::is_same<Src, DescSrc>::value) {
    // a call that carries the sequences' new tokens: each workgroup whose
    // split holds the sequence's last page writes its head's token into that
    // page's last used slot (16 lanes K, 16 lanes V, 16 bytes each), and the
    // stores are complete before any wave of the workgroup reads the page.
    // Workgroups of other query tiles of the same head write the same bytes.
    if (!p.dyn && b < src.app_n && pg0 + npg == np) {
      if (wave == 0) {
        const PageView tv = src.page(b, np - 1, hk);
        if (lane < 32 && tv.used > 0) {
          const int c = lane & 15;
          const bool isv = lane >= 16;
          const char* from = (isv ? src.app_v[b] : src.app_k[b]) + hk * src.app_hs[b] * 2 + 16 * c;
          char* to = const_cast<char*>(isv ? tv.v : tv.k) + (int64_t)(tv.used - 1) * kRow + 16 * c;
          *reinterpret_cast<uint4*>(to) = *reinterpret_cast<const uint4*>(from);
        }
        __builtin_amdgcn_s_waitcnt(0);
      }
      __syncthreads();
    }
  }

  MaskRow mrow{nullptr, HELM_F32};
  if constexpr (kMask) mrow = mask_row(p, b, hk * G + g_row, s_row);

  const float scale = p.scale;
  const float cap = p.softcap;
  const float inv_cap = kCap ? 1.f / cap : 0.f;

  float m = -INFINITY;  // running max of row n (same in the 4 lanes of the row)
  float lsum = 0.f;     // this lane's share of row n's weight sum
  mf_f32x4 o[NO];
#pragma unroll
  for (int e = 0; e < NO; ++e) o[e] = mf_f32x4{0.f, 0.f, 0.f, 0.f};

  const int bpp = p.bpp;
  const int nblk = npg * bpp;
  // lane offsets inside a block: K token tau(n) at chunk q4 (+64 B per i),
  // V token q4 (+4 rows per j)
  const int voff_k = (4 * (n & 3) + (n >> 2)) * kRow + 16 * q4;

  struct Blk {
    mf_u32x4 k[NK];
    V v[4];
    // mask elements as loaded, at their width (a 16-bit mask kept as 16-bit
    // values: zero-extending them would be an instruction on each loaded
    // register, placed where the next step's loads must have completed)
    typename std::conditional<kMask16, uint16_t, uint32_t>::type mk[4];
    int ntok;   // valid tokens of the block (0: past the end)
    int tok0;   // HELM token cursor of the block's first token
  };

  auto load_block = [&](int bi, Blk& B) {
    const bool valid = bi < nblk;
    const int pi = valid ? (p.bpp_log2 >= 0 ? bi >> p.bpp_log2 : bi / bpp) : 0;
    const int sub = valid ? bi - pi * bpp : 0;
    const PageView pv = pi < 64 ? lane_page_view(src, lanes, b, pg0 + pi, pi, hk)
                                : lane_page_view(src, lanes_hi, b, pg0 + pi, pi - 64, hk);
    const int tok_in = sub * kBlockTok;
    const int ntok = valid ? sclamp(pv.used - tok_in, 0, kBlockTok) : 0;
    B.ntok = ntok;
    B.tok0 = pv.tok_off + tok_in;
    const auto rk = make_rsrc(pv.k + tok_in * kRow, ntok * kRow);
    const auto rv = make_rsrc(pv.v + tok_in * kRow, ntok * kRow);
#pragma unroll
    for (int i = 0; i < NK; ++i) B.k[i] = buf_load16_nt(rk, voff_k + 64 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j) B.v[j] = buf_load_vrow_nt<D>(rv, (q4 + 4 * j) * kRow, n);
    if constexpr (kMask) {
      // token 4r + q4 of the block for row n; clamped inside the block's
      // tokens (a block past its page's tokens reads the row's first key:
      // its scores are -inf whatever the mask holds)
      const int mbase = ntok > 0 ? B.tok0 : 0;
      const int last = max(ntok - 1, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        B.mk[r] = mrow.bits<kMask16>(mbase + min(4 * r + q4, last));
    }
  };

  auto compute_block = [&](const Blk& B) {
    float mk[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) mk[r] = kMask ? mrow.widen<kMask16>(B.mk[r]) : 0.f;
    mfma_block_step<Ops, weight_parts<T>(D), weight_shift<T>(D), kMask, kCap, kCausal>(
        B.k, B.v, mk, B.ntok, B.tok0, qop, m, lsum, o, scale, cap, inv_cap, s_vis, q4);
  };

  // ---- dynamic block claiming (p.dyn): the waves of every workgroup of the
  // tile share the tile's blocks through one counter -------------------------
  // Block k of the tile is page lo + k / bpp, 16-token block k % bpp of it.
  // The Wt waves of the tile's workgroups take blocks w, w + Wt, w + 2 Wt
  // first (w = the wave's index among them), then claim one block at a time
  // (block 3 Wt + the counter's old value), so a wave that streams faster
  // takes more blocks and every wave's last block ends at about the same
  // time.  Per step a wave reads the result of the claim it issued one step
  // before, issues the next claim, fetches the page record of the block two
  // ahead (scalar load) and the K / V of the block one ahead, then computes
  // the current block: each of the three latencies hides behind one step.
  // Claims only grow, so a wave is done at its first block past the tile.
  if (D == 128 && p.dyn) {
    const int Wt = nsplit_launch * NW;
    const int np_t = hi - lo;
    const int nblk_t = np_t * bpp;
    const int kbase = 3 * Wt;
    uint32_t* const ctr = p.claims + (int64_t)tile * kClaimStride;
    const int w0 = split_local * NW + wave;
    // the block whose last slot takes the step's new token (-1: none)
    int k_tok = -1;
    const char* tok_from = nullptr;
    if constexpr (std::is_same<Src, DescSrc>::value) {
      if (b < src.app_n && np_t > 0) {
        const PageView tv = src.page(b, hi - 1, hk);
        if (tv.used > 0) {
          k_tok = (np_t - 1) * bpp + (tv.used - 1) / kBlockTok;
          tok_from = (lane >= 16 ? src.app_v[b] : src.app_k[b]) + hk * src.app_hs[b] * 2 +
                     16 * (lane & 15);
        }
      }
    }
    // block k's page record, fetched a step before it is used (scalar loads
    // whose wait falls in the next step), and its view; past the tile: none
    struct Rec {
      typename Src::Raw r;
      int k;
    };
    const typename Src::Ctx sc = src.ctx(b);
    auto fetch = [&](int k) {
      Rec d;
      d.k = __builtin_amdgcn_readfirstlane(k);  // uniform: scalar loads, not vector ones
      // (past the tile: the last page's record, not used)
      const int kk = min(d.k, nblk_t - 1);
      const int pi = p.bpp_log2 >= 0 ? kk >> p.bpp_log2 : kk / bpp;
      d.r = src.raw(sc, lo + pi);
      return d;
    };
    auto view = [&](Rec d) {
      PageView pv;
      if (d.k < nblk_t) {
        const int pi = p.bpp_log2 >= 0 ? d.k >> p.bpp_log2 : d.k / bpp;
        Src::pin(d.r);
        pv = src.view(sc, d.r, lo + pi, hk);
        const int tok_in = (d.k - pi * bpp) * kBlockTok;
        pv.k += tok_in * kRow;
        pv.v += tok_in * kRow;
        pv.tok_off += tok_in;
        pv.used -= tok_in;
      } else {
        pv.k = pv.v = reinterpret_cast<const char*>(p.q);
        pv.used = 0;
        pv.tok_off = 0;
      }
      // (uniform; said so, so that the values stay in scalar registers)
      pv.k = reinterpret_cast<const char*>(uniform64(reinterpret_cast<uint64_t>(pv.k)));
      pv.v = reinterpret_cast<const char*>(uniform64(reinterpret_cast<uint64_t>(pv.v)));
      pv.used = __builtin_amdgcn_readfirstlane(pv.used);
      pv.tok_off = __builtin_amdgcn_readfirstlane(pv.tok_off);
      pv.head_stride_b = 0;
      return pv;
    };
    // K / V (and mask) loads of block k through its record
    auto load_dyn = [&](int k, const PageView& pv, Blk& B) {
      k = __builtin_amdgcn_readfirstlane(k);
      if constexpr (std::is_same<Src, DescSrc>::value) {
        if (k == k_tok) {
          // this wave is the one that reads the new token's block: write the
          // token into its slot first (16 lanes K, 16 lanes V)
          if (lane < 32) {
            char* to = const_cast<char*>(lane >= 16 ? pv.v : pv.k) +
                       (int64_t)(pv.used - 1) * kRow + 16 * (lane & 15);
            *reinterpret_cast<uint4*>(to) = *reinterpret_cast<const uint4*>(tok_from);
          }
          __builtin_amdgcn_s_waitcnt(0);
        }
      }
      const int ntok = sclamp(pv.used, 0, kBlockTok);
      B.ntok = ntok;
      B.tok0 = pv.tok_off;
      const auto rk = make_rsrc(pv.k, ntok * kRow);
      const auto rv = make_rsrc(pv.v, ntok * kRow);
#pragma unroll
      for (int i = 0; i < NK; ++i) B.k[i] = buf_load16_nt(rk, voff_k + 64 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) B.v[j] = buf_load_vrow_nt<D>(rv, (q4 + 4 * j) * kRow, n);
      if constexpr (kMask) {
        const int mbase = ntok > 0 ? B.tok0 : 0;
        const int last = max(ntok - 1, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) B.mk[r] = mrow.bits<kMask16>(mbase + min(4 * r + q4, last));
      }
    };
    auto claim = [&]() {
      uint32_t v = 0;
      if (lane == 0) v = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return v;
    };
    bool dry = kbase >= nblk_t;  // no block left to claim
    uint32_t cl = dry ? 0u : claim();
    int kc = w0, kn = w0 + Wt, kr = w0 + 2 * Wt;
    Rec rn = fetch(kn);
    Blk buf[2];
    load_dyn(kc, view(fetch(kc)), buf[0]);
    auto step = [&](Blk& cur, Blk& nxt) {
      int kq = nblk_t;
      if (!dry) {
        kq = kbase + (int)__builtin_amdgcn_readfirstlane(cl);
        if (kq >= nblk_t) {
          kq = nblk_t;
          dry = true;
        } else {
          cl = claim();
        }
      }
      // (the record fetch after the view of the one fetched a step before:
      // scalar loads return out of order, so a wait for that one would also
      // wait for this one)
      load_dyn(kn, view(rn), nxt);
      const Rec rr = fetch(kr);
      compute_block(cur);
      kc = kn;
      kn = kr;
      rn = rr;
      kr = kq;
    };
    while (kc < nblk_t) {
      step(buf[0], buf[1]);
      if (kc >= nblk_t) break;
      step(buf[1], buf[0]);
    }
    // the claim still in flight (its result is not needed)
    __builtin_amdgcn_s_waitcnt(0);
  } else
  // ---- main loop: a ring of mfma_bufs(D) register buffers, all but one
  // blocks' loads in flight while one block is computed ----------------------
  {
    constexpr int NB = mfma_bufs(D);
    // this wave's blocks: wave, wave + NW, ...
    const int nmine = nblk > wave ? (nblk - wave + NW - 1) / NW : 0;
    Blk buf[NB];
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) load_block(wave + i * NW, buf[i]);
    // Whole rounds of NB blocks, then the remaining blocks: an exit inside
    // the unrolled round would join register states the compiler can only
    // reconcile by waiting for every load in flight.  The scheduling barrier
    // keeps each step's loads ahead of its compute, so the wait for the
    // block computed covers that block's loads only.
    int k = 0;
    for (; k + NB <= nmine; k += NB) {
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        load_block(wave + (k + u + NB - 1) * NW, buf[(u + NB - 1) % NB]);
        __builtin_amdgcn_sched_barrier(0);
        compute_block(buf[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < NB - 1; ++u) {
      if (k + u >= nmine) break;
      load_block(wave + (k + u + NB - 1) * NW, buf[(u + NB - 1) % NB]);
      compute_block(buf[u]);
    }
    if constexpr (D != 128) {
      if (__builtin_expect(any_nan<NO>(o), 0))
        infinite_values<T, Src, FEAT, D>(
            p, src, b, hk, pg0, wave, nblk, NW, g_row, s_row, m, lane,
            [&](float w, const uint16_t* v) {
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float wr = __shfl(w, 4 * q4 + r, 64);
#pragma unroll
                for (int e = 0; e < NO; ++e)
                  o[e][r] = with_infinite<T>(
                      o[e][r], wr, v[(D == 64 ? 4 : 8) * n + (e >> 3) * 128 + (e & 7)]);
              }
            });
    }
  }

  // ---- per-wave state to LDS ---------------------------------------------------
  if constexpr (weight_shift<T>(D) != 0) {   // the weights' scale taken back (exact)
    constexpr float kUnit = 1.f / (1 << weight_shift<T>(D));
    lsum *= kUnit;
#pragma unroll
    for (int e = 0; e < NO; ++e)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[e][r] *= kUnit;
  }
  float lrow = lsum + __shfl_xor(lsum, 16, 64);
  lrow += __shfl_xor(lrow, 32, 64);
  if (q4 == 0) {
    sm.m[wave][n] = m;
    sm.l[wave][n] = lrow;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    // the lane's dims: D = 64 4n .. 4n + 3, else 8n .. 8n + 7 of each 128
    float* dst = &sm.o[wave][4 * q4 + r][(D == 64 ? 4 : 8) * n];
#pragma unroll
    for (int e = 0; e < NO; e += 4)
      *reinterpret_cast<float4*>(dst + (e >> 3) * 128 + (e & 7)) =
          make_float4(o[e][r], o[e + 1][r], o[e + 2][r], o[e + 3][r]);
  }
  __syncthreads();
  if (stp && tid == 0) stp[1] = stamp_now();
  split_epilogue_mfma<T, NW, kMfmaRows, D>(sm, p, tid, tile, split, total, nrows, r0, b, hk);
  if (stp && tid == 0) stp[2] = stamp_now();
}

template <typename T, class Src, int FEAT, int NW>
__global__ __launch_bounds__(64 * NW) void decode_mfma_kernel(AttnParams p, Src src) {
  decode_mfma_body<T, Src, FEAT, NW, 128>(p, src);
}
template <typename T, class Src, int FEAT, int D>
__global__ __launch_bounds__(256) void decode_mfma_dim_kernel(AttnParams p, Src src) {
  decode_mfma_body<T, Src, FEAT, 4, D>(p, src);
}

// ---- query chunks: K/V blocks staged through LDS ----------------------------
// For q_len > 1 with more than one 16-row tile per KV head.  A workgroup of
// four waves owns four 16-row tiles (one per wave) and walks the split's
// blocks in stages of four: wave w loads block w of the stage (K and V,
// 4 KiB each) from HBM / L2 into registers one stage ahead, writes it to LDS,
// and after one barrier every wave computes all four blocks from LDS.  K and
// V sit in LDS as 16-byte chunks with chunk c of token t at slot c ^ (t % 16),
// so the operand reads of a wave (16 tokens x one chunk for K, one token x
// 16 chunks for V) are free of bank conflicts.  The per-block arithmetic is
// mfma_block_step, as in the decode kernel.  A split may span any number of
// pages: the page records sit one per lane in windows of 64 pages, the next
// window loaded when the current one is entered.  Each wave writes its own
// split partial (merged by merge_splits_d128_kernel), or, when the call has a
// single split (p.direct_out), its normalized output rows.
constexpr int kChunkStage = 4;        // blocks per stage = waves per workgroup
constexpr int kRecWindow = 64;        // page records held per lane window

template <typename T, class Src, int FEAT>
__global__ __launch_bounds__(256) void chunk_mfma_kernel(AttnParams p, Src src) {
  using Ops = MfmaOps<T>;
  constexpr int kRow = 256;            // bytes per token row (128 dims x 2 B)
  constexpr int kBlk = kBlockTok * kRow;  // 4 KiB per block of K (or V)
  constexpr bool kMask = (FEAT & kFeatMask) != 0;
  constexpr bool kCap = (FEAT & kFeatCap) != 0;
  constexpr bool kCausal = (FEAT & kFeatCausal) != 0;
  // [buffer][K, V][block of the stage][16-byte chunk]
  __shared__ mf_u32x4 lds[2][2][kChunkStage][kBlk / 16];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int q4 = lane >> 4;
  const int n = lane & 15;

  const int split_local = blockIdx.x;
  const int hk = blockIdx.y % p.Hkv;
  const int qt_w = (blockIdx.y / p.Hkv) * kChunkStage + wave;
  const bool wave_rows = qt_w < p.n_qtiles;
  const int qt = wave_rows ? qt_w : p.n_qtiles - 1;
  const int b = blockIdx.z;
  const int tile = (b * p.Hkv + hk) * p.n_qtiles + qt;
  const int S = p.S;
  const int G = p.G;
  const int r0 = qt * kMfmaRows;
  const int nrows = min(kMfmaRows, G * S - r0);

  // output row of this lane's accumulator row 4 q4 + r (direct output)
  auto out_row = [&](int r) -> char* {
    const RowCoord c = row_coord(r0 + 4 * q4 + r, G);
    return reinterpret_cast<char*>(p.out) +
           (((int64_t)(b * p.Hq + hk * G + c.g) * S + c.s) * 128 + n) * 2;
  };

  const int np = src.n_pages(b);
  const int lo = min(p.lo, np);
  const int hi = min(p.hi, np);
  const int nsplit_launch = (hi - lo + p.pps - 1) / p.pps;
  const int total = p.total_splits > 0 ? p.total_splits : nsplit_launch;
  if (split_local == 0 && lane == 0 && wave_rows) p.counts[tile] = total;
  if (!(total > 0 && split_local < nsplit_launch)) {      // uniform per workgroup
    if (p.direct_out && total == 0 && split_local == 0 && wave_rows) {
      // no keys: HELM's zeros
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * q4 + r < nrows) {
          uint16_t* dst = reinterpret_cast<uint16_t*>(out_row(r));
#pragma unroll
          for (int e = 0; e < 8; ++e) dst[16 * e] = 0;
        }
    }
    return;
  }
  const int split = p.split_base + split_local;
  const int pg0 = lo + split_local * p.pps;
  const int npg = min(pg0 + p.pps, hi) - pg0;

  const bool row_ok = n < nrows;
  const int rr = r0 + (row_ok ? n : 0);
  const RowCoord rc = row_coord(rr, G);
  const int g_row = rc.g;
  const int s_row = rc.s;
  // causal: query position s sees tokens 0 .. s + causal - 1
  const int s_vis = s_row + (kCausal ? p.causal - 1 : 0);
  mf_u32x4 qop[4];
  {
    const int h = hk * G + g_row;
    const char* qp = reinterpret_cast<const char*>(p.q) +
                     ((int64_t)(b * p.Hq + h) * S + s_row) * kRow;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(qp + 16 * (4 * i + q4));
      qop[i] = row_ok ? mf_u32x4{v.x, v.y, v.z, v.w} : mf_u32x4{0u, 0u, 0u, 0u};
    }
  }
  MaskRow mrow{nullptr, HELM_F32};
  if constexpr (kMask) mrow = mask_row(p, b, hk * G + g_row, s_row);
  const float scale = p.scale;
  const float cap = p.softcap;
  const float inv_cap = kCap ? 1.f / cap : 0.f;

  float m = -INFINITY;
  float lsum = 0.f;
  mf_f32x4 o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = mf_f32x4{0.f, 0.f, 0.f, 0.f};

  const int bpp = p.bpp;
  const int nblk = npg * bpp;
  const int nstage = (nblk + kChunkStage - 1) / kChunkStage;

  // page records: window [win, win + 64) of the split's pages, and the next
  typename LanesOf<Src>::type lanes = lane_pages(src, b, pg0, lane);
  typename LanesOf<Src>::type lanes_next = lane_pages(src, b, pg0 + kRecWindow, lane);
  int win = 0;
  // the page (relative to pg0) and sub-block of the next block to be viewed
  int cur_pi = 0, cur_sub = 0;

  // The four blocks of a stage, viewed once, in order: valid tokens and HELM
  // token cursor of each (uniform), and this wave's own block's K / V bases.
  struct StageView {
    int ntok[kChunkStage], tok0[kChunkStage];
    int own_ntok;
    const char *kb, *vb;
  };
  auto view_stage = [&](int st, StageView& sv) {
#pragma unroll
    for (int j = 0; j < kChunkStage; ++j) {
      if (cur_pi - win >= kRecWindow) {   // uniform: the page lies in the next window
        lanes = lanes_next;
        win += kRecWindow;
        lanes_next = lane_pages(src, b, pg0 + win + kRecWindow, lane);
      }
      const PageView pv = lane_page_view(src, lanes, b, pg0 + cur_pi, cur_pi - win, hk);
      const int tok_in = cur_sub * kBlockTok;
      const int nt = st * kChunkStage + j < nblk ? sclamp(pv.used - tok_in, 0, kBlockTok) : 0;
      sv.ntok[j] = nt;
      sv.tok0[j] = pv.tok_off + tok_in;
      if (j == wave) {
        sv.own_ntok = nt;
        sv.kb = pv.k + tok_in * kRow;
        sv.vb = pv.v + tok_in * kRow;
      }
      if (++cur_sub == bpp) {
        cur_sub = 0;
        ++cur_pi;
      }
    }
  };

  // additive mask of the lane's row for the four blocks of a stage (tokens
  // 4r + q4 of each block), loaded a stage ahead like the K/V chunks
  float mcur[kChunkStage][4], mnext[kChunkStage][4];
  auto load_mask = [&](const StageView& sv, float (&mk)[kChunkStage][4]) {
    if constexpr (kMask) {
#pragma unroll
      for (int j = 0; j < kChunkStage; ++j) {
        const int last = max(sv.ntok[j] - 1, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          mk[j][r] = sv.ntok[j] > 0 ? mrow[sv.tok0[j] + min(4 * r + q4, last)] : 0.f;
      }
    }
  };

  // this wave's share of a stage: block (stage * 4 + wave), 4 chunks of K and
  // 4 of V per lane (chunk lane + 64 u of the block)
  mf_u32x4 gk[4], gv[4];
  auto load_stage = [&](const StageView& sv) {
    const auto rk = make_rsrc(sv.kb, sv.own_ntok * kRow);
    const auto rv = make_rsrc(sv.vb, sv.own_ntok * kRow);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      gk[u] = buf_load16_nt(rk, (lane + 64 * u) * 16);
      gv[u] = buf_load16_nt(rv, (lane + 64 * u) * 16);
    }
  };
  auto store_stage = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = lane + 64 * u;          // chunk index in the block
      const int t = c >> 4;                 // token
      const int slot = t * 16 + ((c & 15) ^ t);
      lds[buf][0][wave][slot] = gk[u];
      lds[buf][1][wave][slot] = gv[u];
    }
  };

  // LDS address this lane supplies to the transpose read of V dim group e of
  // block j: token 4 (n >> 2) + q4, dims 16 e + 4 (n & 3) .. + 3 (8 bytes of
  // the swizzled row); the read hands lane n dim 16 e + n of the four tokens
  // 4r + q4 supplied by lanes n >> 2, + 4, + 8, + 12 of its 16-lane group
  const int vt = 4 * (n >> 2) + q4;
  auto vaddr = [&](int buf, int j, int e) -> const char* {
    const int chunk = 2 * e + ((n & 3) >> 1);
    return reinterpret_cast<const char*>(&lds[buf][1][j][vt * 16 + (chunk ^ vt)]) + 8 * (n & 1);
  };
  const int tau = 4 * (n & 3) + (n >> 2);   // K token of this lane in a block
  StageView sv_cur, sv_next;
  if (nstage > 0) {
    view_stage(0, sv_cur);
    load_stage(sv_cur);
    if (wave_rows) load_mask(sv_cur, mcur);
  }
  for (int st = 0; st < nstage; ++st) {
    const int buf = st & 1;
    store_stage(buf);
    if (st + 1 < nstage) {
      view_stage(st + 1, sv_next);
      load_stage(sv_next);
      if (wave_rows) load_mask(sv_next, mnext);
    }
    __syncthreads();
    if (wave_rows) {
      // blocks in pairs: one P . V MFMA takes 32 tokens (block jp's four of
      // this lane in k 0-3, block jp + 1's in k 4-7), once with the hi parts
      // of the weights and once with the lo parts, against the same V
      // operand; an empty block of a pair holds zeros (bounded loads) and
      // -inf logits, so it adds nothing
#pragma unroll
      for (int jp = 0; jp < kChunkStage; jp += 2) {
        if (sv_cur.ntok[jp] == 0 && sv_cur.ntok[jp + 1] == 0) continue;   // uniform
        float x[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int j = jp + h;
          mf_u32x4 k[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) k[i] = lds[buf][0][j][tau * 16 + ((q4 + 4 * i) ^ tau)];
          float mk[4] = {0.f, 0.f, 0.f, 0.f};
          if constexpr (kMask) {
#pragma unroll
            for (int r = 0; r < 4; ++r) mk[r] = mcur[j][r];
          }
          mfma_logits<kMask, kCap, kCausal>(mfma_qk<Ops>(k, qop), mk, sv_cur.ntok[j],
                                            sv_cur.tok0[j], scale, cap, inv_cap, s_vis, q4, x[h]);
        }
        mfma_refresh_max<0>(fmaxf(fmaxf(fmaxf(x[0][0], x[0][1]), fmaxf(x[0][2], x[0][3])),
                               fmaxf(fmaxf(x[1][0], x[1][1]), fmaxf(x[1][2], x[1][3]))),
                         m, lsum, o, q4);
        const float base = (m == -INFINITY) ? 0.f : m;
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float wt[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            wt[r] = fexp(x[h][r] - base);
            lsum += wt[r];
          }
          Ops::split2(wt[0], wt[1], hw[2 * h], lw[2 * h]);
          Ops::split2(wt[2], wt[3], hw[2 * h + 1], lw[2 * h + 1]);
        }
        const mf_u32x4 phi = mf_u32x4{hw[0], hw[1], hw[2], hw[3]};
        const mf_u32x4 plo = mf_u32x4{lw[0], lw[1], lw[2], lw[3]};
        // V operand of dim group e: lane n gets dim 16 e + n of tokens
        // 4r + q4 (r = 0..3) of each block, by the LDS transpose read
        mf_u32x4 vop[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint2 a = ld_tr16(vaddr(buf, jp, e));
          const uint2 c = ld_tr16(vaddr(buf, jp + 1, e));
          vop[e] = mf_u32x4{a.x, a.y, c.x, c.y};
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = Ops::mma(phi, vop[e], o[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = Ops::mma(plo, vop[e], o[e]);
      }
    }
    sv_cur = sv_next;
    if constexpr (kMask) {
#pragma unroll
      for (int j = 0; j < kChunkStage; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) mcur[j][r] = mnext[j][r];
    }
  }

  if (!wave_rows) return;
  float lrow = lsum + __shfl_xor(lsum, 16, 64);
  lrow += __shfl_xor(lrow, 32, 64);
  if (p.direct_out) {
    // the call's only split: normalized rows straight to the output
    // (HELM's final out / max(sum, 1e-12), kv_cache.py:554-555)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float l = __shfl(lrow, 4 * q4 + r, 64);   // lane 4 q4 + r holds that row's sum
      const float inv = 1.f / fmaxf(l, 1e-12f);
      if (4 * q4 + r < nrows) {
        uint16_t* dst = reinterpret_cast<uint16_t*>(out_row(r));
#pragma unroll
        for (int e = 0; e < 8; ++e)                              // dim 16 e + n
          dst[16 * e] = static_cast<uint16_t>(Ops::pk(o[e][r] * inv, 0.f));
      }
    }
    return;
  }
  // the wave's own partial (m, l, o[128]) per row, straight from registers
  const int64_t part = ((int64_t)tile * p.max_splits + split) * p.rows_per_tile;
  if (q4 == 0 && n < nrows)
    *reinterpret_cast<float2*>(&p.ws_ml[(part + n) * 2]) = make_float2(m, lrow);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 4 * q4 + r;
    if (row < nrows) {
      float* dst = &p.ws_o[(part + row) * 128 + n];
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[16 * e] = o[e][r];      // dim 16 e + n
    }
  }
}

}  // namespace helm
