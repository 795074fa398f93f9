// Query chunks on 32 x 32 matrix-core tiles (v_mfma_f32_32x32x16_{bf16,f16}).
//
// The same page walk and LDS staging as chunk_mfma_kernel (stages of four
// 16-token blocks swizzled into LDS, two stage buffers, one barrier per stage;
// here the blocks go from memory straight into LDS by buffer loads with the
// LDS destination, shared out over the workgroup's waves), but each wave owns
// 32 query rows (two 16-row tiles of the partial layout) and computes 32
// tokens (two blocks) per step, so the softmax of a step covers 1024 scores
// instead of 256 and its fixed costs (max refresh check, weight rounding,
// scalar bookkeeping) are shared by four times the matrix work.  A workgroup
// has four waves (128 rows; two workgroups per CU) or eight (256 rows; one
// per CU, half the stage loads per row).
//
// Lane l = 32 hh + j (j = l % 32):
//   q . k   S^T = K Q^T: A = K (row m = token tau(m), dims 16i + 8hh .. + 7),
//           B = Q^T (column j = query row j), one MFMA per 16 dims.
//           The result gives lane l, for its query row j, register
//           r = 4g + t <-> output row m = 8g + 4hh + t, and with
//           tau(8g + 4h + t) = 16 (g >> 1) + 8h + 4 (g & 1) + t register r holds
//           token 8hh + (r & 7) of block r >> 3 of the step.
//   P . V   O += P V: A = the weights of row j for tokens 8hh .. 8hh + 7 of a
//           block (exactly registers 8u .. 8u + 7 above), rounded once to the
//           16-bit type; B = V of those tokens at dim 32e + j, fetched by LDS
//           transpose reads; O register 4g + t of dim group e is row
//           8g + 4hh + t, dim 32e + j.  The row sums add
//           exactly the weights P . V used (packed dot products with ones), so
//           that each output row is an exact weighted mean of V under the
//           rounded weights (their rounding perturbs the weights by <= 2^-9
//           relative, bf16, and the mean by that times the spread of V).
//           (D = 128; HELM_CHUNK32_HILO=1 builds hi + lo there, weights to
//           ~2^-17, one more MFMA per group.  At D = 64 and 256 the weights
//           enter in weight_parts parts, one MFMA per part and group.)
// Online softmax per query row with the lazy rescale of the decode kernel, in
// base-2 units (logits scaled by log2(e) with the softmax scale, weights
// 2^(x - m); the partials' max goes out in natural units).
#pragma once

#include <type_traits>

#include "attn_mfma.h"

namespace helm {

typedef float mf_f32x16 __attribute__((ext_vector_type(16)));

template <typename T> struct Mfma32;
template <> struct Mfma32<bf16_t> {
  __device__ static __forceinline__ mf_f32x16 mma(mf_u32x4 a, mf_u32x4 b, mf_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mf_bf16x8, a),
                                                   __builtin_bit_cast(mf_bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma32<f16_t> {
  __device__ static __forceinline__ mf_f32x16 mma(mf_u32x4 a, mf_u32x4 b, mf_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mf_f16x8, a),
                                                  __builtin_bit_cast(mf_f16x8, b), c, 0, 0, 0);
  }
};

constexpr int kChunk32Rows = 32;   // query rows per wave

// LDS swizzle of a staged block: chunk c (16 B) of token t (0..15) sits at
// slot c ^ swz(t) of the token's row.  The q . k reads (one chunk, 16 tokens
// per 16 lanes) meet 16 distinct slots mod 16, and so do the V transpose reads
// (chunks c0 .. c0 + 3, c0 a multiple of 4, of four consecutive tokens
// 4a .. 4a + 3 per 32 lanes): each group of accesses covers every 16-byte bank
// group once.  Rows of 256 bytes or more (D = 128, 256): swz(4a + b) = 4b + a.
// D = 64, two tokens per 256 bytes: the eight tokens of one parity take eight
// different XORs, t and t + 2 differing in bit 2, swz(4a + 2b + p) = 4b + a.
template <int D>
__device__ __forceinline__ int swz(int t) {
  return D == 64 ? ((t & 2) << 1) | (t >> 2) : ((t & 3) << 2) | (t >> 2);
}
// P . V with the weights in 16-bit parts (weight_parts) or, at D = 128, rounded
// once to 16 bits (a query chunk is bound by the matrix cores, and the single
// rounding stays far inside the tolerance; HELM_CHUNK32_HILO=1 builds hi + lo
// there too)
#ifndef HELM_CHUNK32_HILO
#define HELM_CHUNK32_HILO 0
#endif
template <typename T>
constexpr int chunk32_parts(int D) {
  return D != 128 ? weight_parts<T>(D) : HELM_CHUNK32_HILO ? 2 : 1;
}
constexpr float kLog2E = 1.4426950408889634f;   // log2(e)
constexpr float kLn2 = 0.6931471805599453f;     // ln(2)

// 16 bytes per lane from a buffer straight into LDS: lane i writes
// lds_dst + 16 i (the address must be the same in every lane); loads past the
// buffer's size write zeros
__device__ __forceinline__ void buf_load16_lds(__amdgpu_buffer_rsrc_t r, void* lds_dst, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds_dst, 16,
                                           off, 0, 0, 0);
}

// The workgroup's block of query rows.  Under a causal limit a block's walk
// grows with its index; p.qb_round > 0 (blocks per head that the device's CUs
// take in one round of workgroups, in launch order) hands the blocks out
// longest first, every second round in reverse, so that the workgroups that
// share a CU add up to about the same walk and the shortest come last (bf16
// first prompt of 2,048, 40 / 8 heads: in index order 83, longest first 65 us;
// 32 / 32 heads: 67, longest first 61.5, with the reversal 59.6).
__device__ __forceinline__ int query_block(const AttnParams& p) {
  const int j = blockIdx.y / p.Hkv;
  if (p.qb_round <= 0) return j;
  const int n = gridDim.y / p.Hkv;
  const int r = j / p.qb_round, first = r * p.qb_round;
  const int last = min(n, first + p.qb_round) - 1;
  return n - 1 - ((r & 1) ? last - (j - first) : j);
}

// NW waves per workgroup (4: two workgroups per CU; 8: one, which halves the
// stage loads per query row), 32 query rows each.
template <typename T, class Src, int FEAT, int NW, int D>
__device__ __forceinline__ void chunk32_mfma_body(const AttnParams& p, const Src& src) {
  static_assert(NW == 4 || NW == 8, "waves per workgroup");
  constexpr int SB = kChunkStage;   // 16-token blocks per stage
  constexpr int kParts = chunk32_parts<T>(D);
  constexpr int kShift = weight_shift<T>(D);
  constexpr float kSlack = chunk_slack(kShift), kUnit = 1.f / (1 << kShift);
  // a window's page records are read one window ahead, except with a mask at
  // D = 256, whose masks, O and query operand leave no registers for them: there
  // they are read when the window is entered, once in 64 blocks
  constexpr bool kAhead = !((FEAT & kFeatMask) && D == 256);
  constexpr int NK = D / 16;        // 16-dim steps of q . k
  constexpr int NE = D / 32;        // 32-dim groups of P . V
  constexpr int CPR = D / 8;        // 16-byte chunks per token row
  using Ops = MfmaOps<T>;
  using M32 = Mfma32<T>;
  constexpr int kRow = 2 * D;              // bytes per token row
  constexpr int kBlk = kBlockTok * kRow;   // bytes per 16-token block of K (or V)
  constexpr bool kMask = (FEAT & kFeatMask) != 0;
  constexpr bool kCap = (FEAT & kFeatCap) != 0;
  constexpr bool kCausal = (FEAT & kFeatCausal) != 0;
  constexpr bool kMask16 = (FEAT & kFeatMask16) != 0;
  // 16-byte-per-lane loads (1 KiB each) a wave issues per stage: a stage is
  // SB blocks of K and of V, kBlkLoads loads each, shared out over the NW
  // waves in order (wave w takes loads w * kLoads ..), all in one block per wave
  constexpr int kBlkLoads = kBlk / 1024;
  constexpr int kLoads = 2 * kBlkLoads * SB / NW;
  // two stage buffers as two objects, so that the compiler sees that the
  // loads filling one never touch the reads of the other:
  // [K, V][block of the stage][16-byte chunk], chunk c of token t at slot
  // t * CPR + (c ^ swz(t)) (see swz)
  typedef mf_u32x4 StageBuf[2][SB][kBlk / 16];
  __shared__ StageBuf lds0, lds1;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int jr = lane & 31;
  const int hh = lane >> 5;

  const int split_local = blockIdx.x;
  const int hk = blockIdx.y % p.Hkv;
  const int n32 = (p.n_qtiles + 1) / 2;                 // 32-row groups of the head
  const int wt = query_block(p) * NW + wave;
  const bool wave_rows = wt < n32;
  const int wtc = wave_rows ? wt : n32 - 1;
  const int b = blockIdx.z;
  const int S = p.S;
  const int G = p.G;
  const int rbase = wtc * kChunk32Rows;
  const int nrows = min(kChunk32Rows, G * S - rbase);
  const int tile0 = (b * p.Hkv + hk) * p.n_qtiles + 2 * wtc;   // this wave's first 16-row tile
  const bool two_tiles = 2 * wtc + 1 < p.n_qtiles;

  // output element of O register 4g + t of dim group e
  auto out_elem = [&](int g, int t, int e) -> uint16_t* {
    const RowCoord c = row_coord(rbase + 8 * g + 4 * hh + t, G);
    return reinterpret_cast<uint16_t*>(p.out) +
           ((int64_t)(b * p.Hq + hk * G + c.g) * S + c.s) * D + 32 * e + jr;
  };

  const int np = src.n_pages(b);
  const int lo = min(p.lo, np);
  const int hi = min(p.hi, np);
  const int nsplit_launch = (hi - lo + p.pps - 1) / p.pps;
  const int total = p.total_splits > 0 ? p.total_splits : nsplit_launch;
  if (split_local == 0 && lane == 0 && wave_rows) {
    p.counts[tile0] = total;
    if (two_tiles) p.counts[tile0 + 1] = total;
  }
  if (!(total > 0 && split_local < nsplit_launch)) {        // uniform per workgroup
    if (p.direct_out && total == 0 && split_local == 0 && wave_rows) {
      // no keys: HELM's zeros
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (8 * g + 4 * hh + t < nrows)
#pragma unroll
            for (int e = 0; e < NE; ++e) *out_elem(g, t, e) = 0;
    }
    return;
  }
  const int split = p.split_base + split_local;
  const int pg0 = lo + split_local * p.pps;
  const int npg = min(pg0 + p.pps, hi) - pg0;

  // ---- query operand: row jr of the wave, dims 16i + 8hh .. + 7 ----------------
  const bool row_ok = jr < nrows;
  const RowCoord rc = row_coord(rbase + (row_ok ? jr : 0), G);
  const int s_row = rc.s;
  // causal: query position s sees tokens 0 .. s + coff (coff = causal - 1)
  const int coff = kCausal ? p.causal - 1 : 0;
  const int s_vis = s_row + coff;                      // row jr's last visible token
  const int s_last = (rbase + nrows - 1) / G + coff;   // the wave's last visible token
  const int s_first = rbase / G + coff;                // and its first row's
  // causal: the workgroup's last query position; stages starting past it
  // add nothing for any of its rows (a causal call lists a launch's pages in
  // token order, so tokens only grow along the walk), and the walk ends
  // there (uniform across the workgroup)
  const int qrow_end = min(G * S, (query_block(p) + 1) * NW * kChunk32Rows);
  const int s_last_wg = (qrow_end - 1) / G + coff;
  mf_u32x4 qop[NK];
  {
    const char* qp = reinterpret_cast<const char*>(p.q) +
                     ((int64_t)(b * p.Hq + hk * G + rc.g) * S + s_row) * kRow;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(qp + 16 * (2 * i + hh));
      qop[i] = row_ok ? mf_u32x4{v.x, v.y, v.z, v.w} : mf_u32x4{0u, 0u, 0u, 0u};
    }
  }
  MaskRow mrow{nullptr, HELM_F32};
  if constexpr (kMask) mrow = mask_row(p, b, hk * G + rc.g, s_row);
  const float scale = p.scale;
  const float cap = p.softcap;
  const float inv_cap = kCap ? 1.f / cap : 0.f;
  // logits, running max and weights in base-2 units: one multiply per score
  // turns q . k into x = s * scale * log2(e), and each weight is 2^(x - m)
  const float scale2 = scale * kLog2E;
  const float cap2 = cap * kLog2E;
  auto sexp = [](float v) { return __builtin_amdgcn_exp2f(v); };

  float m = -INFINITY;   // running max of row jr (same in both halves)
  // this lane's share of row jr's weight sum: of the fp32 weights where P . V
  // takes them in parts, else of exactly the rounded weights it takes (packed
  // dot products with ones: half the matrix-core time that a ones column of
  // P . V takes, and no accumulator tile; bf16 512 tokens over 32k, 32 / 8 heads:
  // 303 -> 299 us)
  float lsum = 0.f;
  mf_f32x16 o[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[e][r] = 0.f;

  const int bpp = p.bpp;
  const int nblk = npg * bpp;
  const int nstage = (nblk + SB - 1) / SB;

  // The walk's blocks, viewed 64 at a time: lane i holds block win + i of the
  // split, its K / V addresses, valid tokens and first token offset, and ballots
  // over the window say which blocks are partial (or empty), add nothing to any
  // row of the wave, reach a row's causal limit, or lie past every row of the
  // workgroup.  A stage then takes its four blocks' bits and one address by
  // v_readlane, where walking pages and sub-blocks in scalar code took ~120
  // scalar instructions per stage of every wave's serial path (bf16 512 tokens
  // over 32k: 296 -> 271; D = 64, 512 over 16k: 144 -> 128 us).
  struct Window {
    uint32_t klo, khi, vlo, vhi;
    int nt, t0;
    uint64_t part, none, limit, end;
  } win;
  auto block_page = [&](int blk) -> int {
    return min(p.bpp_log2 >= 0 ? blk >> p.bpp_log2 : blk / bpp, npg - 1);
  };
  // the record of the page of block w0 + lane (lane 0's position of a lane window)
  auto load_records = [&](int w0) {
    return lane_pages(src, b, pg0 + block_page(w0 + lane), 0);
  };
  typename LanesOf<Src>::type recs = load_records(0);
  auto enter_window = [&](int w0) {
    if (!kAhead && w0 > 0) recs = load_records(w0);
    const int blk = w0 + lane;
    const int pi = block_page(blk);
    const int tok_in = (blk - pi * bpp) * kBlockTok;
    const PageView pv = lane_own_view(src, recs, b, pg0 + pi, hk);
    win.nt = blk < nblk ? max(0, min(pv.used - tok_in, kBlockTok)) : 0;
    win.t0 = pv.tok_off + tok_in;
    const uint64_t ka = reinterpret_cast<uint64_t>(pv.k) + (int64_t)tok_in * kRow;
    const uint64_t va = reinterpret_cast<uint64_t>(pv.v) + (int64_t)tok_in * kRow;
    win.klo = static_cast<uint32_t>(ka);
    win.khi = static_cast<uint32_t>(ka >> 32);
    win.vlo = static_cast<uint32_t>(va);
    win.vhi = static_cast<uint32_t>(va >> 32);
    win.part = __builtin_amdgcn_ballot_w64(win.nt < kBlockTok);
    win.none = __builtin_amdgcn_ballot_w64(win.nt == 0 || (kCausal && win.t0 > s_last));
    win.limit =
        kCausal ? __builtin_amdgcn_ballot_w64(win.nt > 0 && win.t0 + kBlockTok - 1 > s_first) : 0;
    // (an empty block, past the used tokens of a page shorter than the longest,
    // says nothing: the next page's tokens may lie before its offset)
    win.end = kCausal ? __builtin_amdgcn_ballot_w64(win.nt > 0 && win.t0 > s_last_wg) : 0;
    if (kAhead) recs = load_records(w0 + kRecWindow);
  };

  // a stage's four blocks: their bits of the window's ballots, and (where a
  // step needs them: a mask, a partial block or a causal limit) their valid
  // tokens and first token offsets; kept for the stage's compute, one stage
  // after its loads were issued
  struct StageBits {
    uint32_t part, none, limit;
    bool end;
  } bits[2];
  int vnt[2][SB], vt0[2][SB];
  struct OwnBlock {
    int ntok;
    const char *kb, *vb;
  };
  const int own_blk = (wave * kLoads) / (2 * kBlkLoads);
  static_assert(kRecWindow % SB == 0, "windows start at stage boundaries");
  auto view_stage = [&](int st, StageBits& sb, int (&ntok)[SB], int (&tok0)[SB], OwnBlock& ob) {
    const int at = (st * SB) % kRecWindow;
    if (at == 0) enter_window(st * SB);   // uniform
    constexpr uint32_t kAll = (1u << SB) - 1;
    sb.part = static_cast<uint32_t>(win.part >> at) & kAll;
    sb.none = static_cast<uint32_t>(win.none >> at) & kAll;
    sb.limit = static_cast<uint32_t>(win.limit >> at) & kAll;
    sb.end = (win.end >> at) & 1;
    if (kMask || (sb.part | sb.limit)) {
#pragma unroll
      for (int j = 0; j < SB; ++j) {
        ntok[j] = __builtin_amdgcn_readlane(win.nt, at + j);
        tok0[j] = __builtin_amdgcn_readlane(win.t0, at + j);
      }
    }
    const int own = at + own_blk;
    ob.ntok = __builtin_amdgcn_readlane(win.nt, own);
    ob.kb = reinterpret_cast<const char*>(
        ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(win.khi, own) << 32) |
        (uint32_t)__builtin_amdgcn_readlane(win.klo, own));
    ob.vb = reinterpret_cast<const char*>(
        ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(win.vhi, own) << 32) |
        (uint32_t)__builtin_amdgcn_readlane(win.vlo, own));
  };

  // this wave's loads of a stage straight from memory into LDS (no VGPRs):
  // load i = wave * kLoads + k covers K (the block's first kBlkLoads) or V of
  // the wave's block, slots 64u .. 64u + 63 with u = i % kBlkLoads, lane l slot
  // 64u + l of token t = (64u + l) / CPR, which holds chunk (l % CPR) ^ swz(t)
  // (the swizzle), so each lane fetches that chunk; loads past the block's
  // tokens write zeros
  auto dma_stage = [&](const OwnBlock& ob, StageBuf& dst) {
    const auto rk = make_rsrc(ob.kb, ob.ntok * kRow);
    const auto rv = make_rsrc(ob.vb, ob.ntok * kRow);
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
      const int i = wave * kLoads + k;
      const int u = i % kBlkLoads;
      const int t = (64 / CPR) * u + lane / CPR;
      const int off = t * kRow + 16 * ((lane % CPR) ^ swz<D>(t));
      if ((i / kBlkLoads) & 1)
        buf_load16_lds(rv, &dst[1][own_blk][64 * u], off);
      else
        buf_load16_lds(rk, &dst[0][own_blk][64 * u], off);
    }
  };

  // K row this lane supplies to the q . k MFMAs: token tau(jr) of the step
  const int g_a = jr >> 3, h_a = (jr >> 2) & 1, t_a = jr & 3;
  const int tau = 16 * (g_a >> 1) + 8 * h_a + 4 * (g_a & 1) + t_a;
  const int kblk = tau >> 4, ktok = tau & 15;
  // transpose-read address of V: token 8hh + 4z + (n >> 2) of a block, dims
  // 32e + 16 (jr >> 4) + 4 (n & 3) .. + 3, with n = lane % 16
  const int nl = lane & 15;
  auto vaddr = [&](const StageBuf& cur, int blk, int z, int e) -> const char* {
    const int vtok = 8 * hh + 4 * z + (nl >> 2);
    const int chunk = 4 * e + 2 * (jr >> 4) + ((nl & 3) >> 1);
    return reinterpret_cast<const char*>(&cur[1][blk][vtok * CPR + (chunk ^ swz<D>(vtok))]) +
           8 * (nl & 1);
  };

  // additive mask of row jr for a stage's blocks: tokens 8hh .. 8hh + 7 of
  // each, bounded by its valid tokens, as loaded: eight words for an fp32 mask,
  // four (two tokens each) for a 16-bit one.  A whole block's tokens are 16-byte
  // loads at the mask's own alignment; a partial block's go one by one, the index
  // clamped to its last valid token.  A stage's masks are loaded with its K / V, one
  // stage ahead, or, where the registers for two stages' are not there (fp32
  // masks; D = 128 soft-capped), at the stage's start before the next stage's
  // K / V: a load after those would have to wait for them too.  Element loads of every step, converted and added
  // even where zero, had bound the masked chunk (bf16 512 over 8,192 tokens under
  // a 4,096-token window, 32 / 8 heads: 187 us, now 109; D = 256, 512 over 4,700,
  // soft-capped: 203, now 108).
  typedef typename std::conditional<kMask16, mf_u32x4, mf_u32x8>::type MaskWords;
  constexpr bool kMaskAhead = kMask16 && !(kCap && D == 128);
  MaskWords mkw[kMaskAhead ? 2 : 1][SB];
  auto load_block_mask = [&](int nt, int tok0) -> MaskWords {
    const MaskRow mb = mrow + tok0;
    if (__builtin_expect(nt == kBlockTok, 1)) {
      const char* src = (mb + 8 * hh).base;
      const mf_u32x4 a = load16_any(src);
      if constexpr (kMask16) {
        return a;
      } else {
        const mf_u32x4 c = load16_any(src + 16);
        return mf_u32x8{a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
      }
    }
    if (nt == 0) return MaskWords(0u);
    auto at = [&](int i) -> uint32_t {
      return mb.template bits<kMask16>(min(8 * hh + i, nt - 1));
    };
    if constexpr (kMask16)
      return mf_u32x4{at(0) | at(1) << 16, at(2) | at(3) << 16, at(4) | at(5) << 16,
                      at(6) | at(7) << 16};
    else
      return mf_u32x8{at(0), at(1), at(2), at(3), at(4), at(5), at(6), at(7)};
  };
  auto load_stage_mask = [&](const int (&ntok)[SB], const int (&tok0)[SB], MaskWords (&w)[SB]) {
    if constexpr (kMask) {
#pragma unroll
      for (int j = 0; j < SB; ++j) w[j] = load_block_mask(ntok[j], tok0[j]);
    }
  };
  // any bit of the mask words set (a zero mask adds nothing to any score)
  auto mask_bits = [&](const MaskWords& w) -> uint32_t {
    uint32_t any = w[0] | w[1] | w[2] | w[3];
    if constexpr (!kMask16) any |= w[4] | w[5] | w[6] | w[7];
    return any;
  };
  // a block's eight mask values in fp32
  auto mask_values = [&](const MaskWords& w, float* mk) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (kMask16)
        mk[i] = mrow.template widen<true>((i & 1) ? w[i >> 1] >> 16 : w[i >> 1] & 0xffffu);
      else
        mk[i] = __uint_as_float(w[i]);
    }
  };

  // the first stage's loads
  {
    OwnBlock ob;
    if (nstage > 0) {
      view_stage(0, bits[0], vnt[0], vt0[0], ob);
      dma_stage(ob, lds0);
      if (kMaskAhead && wave_rows) load_stage_mask(vnt[0], vt0[0], mkw[0]);
    }
  }
  bool done = false;
  // stage st (view slot K = st % 2) computes from `cur` while the loads of
  // stage st + 1 go into `nxt` (the buffer stage st - 1 computed from)
  auto stage = [&](int st, auto kslot, const StageBuf& cur, StageBuf& nxt) {
    constexpr int K = decltype(kslot)::value;
    const int (&ntok_c)[SB] = vnt[K];
    const int (&tok0_c)[SB] = vt0[K];
    if constexpr (kCausal) {
      if (bits[K].end) {
        __builtin_amdgcn_s_waitcnt(0x0F70);   // this stage's loads land before the exit
        done = true;
        return;
      }
    }
    // stage st is in LDS (this wave's loads done, then everyone's), and every
    // wave is done with the other buffer, which the next stage's loads fill
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    __syncthreads();
    if (!kMaskAhead && wave_rows) load_stage_mask(ntok_c, tok0_c, mkw[0]);
    if (st + 1 < nstage) {
      OwnBlock ob;
      view_stage(st + 1, bits[K ^ 1], vnt[K ^ 1], vt0[K ^ 1], ob);
      dma_stage(ob, nxt);
      if constexpr (kMaskAhead)
        if (wave_rows) load_stage_mask(vnt[K ^ 1], vt0[K ^ 1], mkw[K ^ 1]);
    }
    if (wave_rows) {
      // q . k of the step of blocks bp, bp + 1: S^T for the wave's 32 rows
      auto qk = [&](int bp) -> mf_f32x16 {
        mf_f32x16 sc;
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = 0.f;
        // every K operand read issued before the first MFMA (one LDS wait,
        // then the MFMAs back to back), registers allowing: with a mask
        // operand its prefetched values take them, and the compiler's order
        // stays
        mf_u32x4 ka[NK];
#pragma unroll
        for (int i = 0; i < NK; ++i)
          ka[i] = cur[0][bp + kblk][ktok * CPR + ((2 * i + hh) ^ swz<D>(ktok))];
        if constexpr (!kMask && D == 128)
          __builtin_amdgcn_sched_barrier(0);   // (keeps the reads ahead of the MFMAs)
#pragma unroll
        for (int i = 0; i < NK; ++i) sc = M32::mma(ka[i], qop[i], sc);
        return sc;
      };
      // steps that add exactly nothing for any row of the wave are skipped
      // (uniform tests): both blocks empty (an empty block holds zeros and
      // -inf logits), or, causal, every token past the wave's last query
      // position
      auto idle_step = [&](int bp) -> bool { return ((bits[K].none >> bp) & 3) == 3; };
      // logits, online softmax and P . V of one step
      auto finish = [&](int bp, const mf_f32x16& sc, bool add_mask, const float (&mk)[16]) {
        float x[16];
        if constexpr (kCap) {
#pragma unroll
          for (int r = 0; r < 16; ++r) x[r] = sc[r];
          softcap_scores<16>(x, scale * inv_cap, cap2);
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) x[r] = sc[r] * scale2;
        }
        // finfo.min masks stay finite, as in natural units (a row masked
        // everywhere gets equal weights, as HELM's loop gives it).  A zero mask
        // and an added one follow one rule, so that a key's NaN or -inf logit does
        // not depend on its neighbours' masks.  D = 128 (kBound): every masked
        // logit is at least -FLT_MAX, NaN and -inf among them (with a zero mask
        // bounded where the step's maximum asks for it).
        // Else (as the vector-ALU kernel): NaN stays, and -inf hides a key, also
        // where it leaves a row with none; a key masked to -1e30 or below takes
        // its mask as its logit, as the skipped steps have it: lowered by
        // 1e30 (log2(e) - 1), so that the masks' order holds across -1e30.
        constexpr bool kBound = kMask && D == 128;
        if constexpr (kBound) {
          if (add_mask)
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = fmaxf(fmaf(mk[r], kLog2E, x[r]), -__FLT_MAX__);
        } else if constexpr (kMask) {
          if (add_mask)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              x[r] = mk[r] <= -1e30f ? mk[r] - 0.442695e30f : fmaf(mk[r], kLog2E, x[r]);
        }
        if constexpr (kBound) {
          float top = x[0];   // (NaN passes through)
#pragma unroll
          for (int r = 1; r < 16; ++r) top = __builtin_elementwise_maximum(top, x[r]);
          // (a token hidden below may stand above the visible ones here)
          const bool limits = (((bits[K].part | bits[K].limit) >> bp) & 3) != 0;
          if (__builtin_expect(limits || __builtin_amdgcn_ballot_w64(!(top > -INFINITY)) != 0, 0))
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = fmaxf(x[r], -__FLT_MAX__);
        }
        // the per-token limits, only where a step reaches them (uniform tests):
        // the causal limit when a block's last token is past the wave's first
        // query position, the valid-token limit when a block is partial
        if constexpr (kCausal) {
          if (__builtin_expect((bits[K].limit >> bp) & 3, 0)) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (tok0_c[bp + (r >> 3)] + 8 * hh + (r & 7) > s_vis) x[r] = -INFINITY;
          }
        }
        if (__builtin_expect((bits[K].part >> bp) & 3, 0)) {
          const int nt0 = ntok_c[bp], nt1 = ntok_c[bp + 1];
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (8 * hh + (r & 7) >= ((r >> 3) ? nt1 : nt0)) x[r] = -INFINITY;
        }
        float bm = x[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) bm = fmaxf(bm, x[r]);
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(bm > m + kSlack) != 0, 0)) {
          // refresh the row max (both halves of the row agree); with scaled
          // weights to the integer above, so that m - kShift is exact
          float mn = fmaxf(m, fmaxf(bm, __shfl_xor(bm, 32, 64)));
          if constexpr (kShift) mn = ceilf(mn);
          const float a = sexp(m - ((mn == -INFINITY) ? 0.f : mn));
          lsum *= a;
          m = mn;
          // O register 4g + t is row 8g + 4hh + t: that row's factor
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const float ar = __shfl(a, 8 * g + 4 * hh + t, 64);
#pragma unroll
              for (int e = 0; e < NE; ++e) o[e][4 * g + t] *= ar;
            }
        }
        const float base = (m == -INFINITY) ? 0.f : m - kShift;
        uint32_t hw[8], lw[8], ew[8];
        float ws[8];   // (weights below an ulp of the row's sum add up first)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float w0 = sexp(x[2 * q] - base), w1 = sexp(x[2 * q + 1] - base);
          if constexpr (kParts == 3) {
            ws[q] = w0 + w1;
            Ops::split3(w0, w1, hw[q], lw[q], ew[q]);
          } else if constexpr (kParts == 2) {
            ws[q] = w0 + w1;
            if constexpr (std::is_same<T, f16_t>::value) Ops::split2_mix(w0, w1, hw[q], lw[q]);
            else Ops::split2(w0, w1, hw[q], lw[q]);
          } else {
            hw[q] = Ops::pk(w0, w1);
            lsum = dot2<T>(hw[q], Ops::ones8()[0], lsum);
          }
        }
        if constexpr (kParts >= 2)
          lsum += ((ws[0] + ws[1]) + (ws[2] + ws[3])) + ((ws[4] + ws[5]) + (ws[6] + ws[7]));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          auto pop = [&](const uint32_t (&w)[8]) {
            return mf_u32x4{w[4 * u], w[4 * u + 1], w[4 * u + 2], w[4 * u + 3]};
          };
          mf_u32x4 vop[NE];
#pragma unroll
          for (int e = 0; e < NE; ++e) {
            const uint2 a0 = ld_tr16(vaddr(cur, bp + u, 0, e));
            const uint2 a1 = ld_tr16(vaddr(cur, bp + u, 1, e));
            vop[e] = mf_u32x4{a0.x, a0.y, a1.x, a1.y};
          }
#pragma unroll
          for (int e = 0; e < NE; ++e) o[e] = M32::mma(pop(hw), vop[e], o[e]);
          if constexpr (kParts >= 2)
#pragma unroll
            for (int e = 0; e < NE; ++e) o[e] = M32::mma(pop(lw), vop[e], o[e]);
          if constexpr (kParts == 3)
#pragma unroll
            for (int e = 0; e < NE; ++e) o[e] = M32::mma(pop(ew), vop[e], o[e]);
        }
      };
      {
#pragma unroll
        for (int bp = 0; bp < SB; bp += 2) {     // the step's blocks bp, bp + 1
          if (__builtin_expect(idle_step(bp), 0)) continue;
          // masked, a step whose every mask value is <= -1e30 while every
          // row's max is already above -1e20 adds exactly nothing (each
          // weight underflows to 0 and the max stays)
          float mk[16];
          bool add_mask = false;
          if constexpr (kMask) {
            const MaskWords &w0 = mkw[kMaskAhead ? K : 0][bp], &w1 = mkw[kMaskAhead ? K : 0][bp + 1];
            add_mask = __builtin_amdgcn_ballot_w64(mask_bits(w0 | w1) != 0u) != 0;
            if (add_mask) {
              mask_values(w0, mk);
              mask_values(w1, mk + 8);
              float mm = mk[0];
#pragma unroll
              for (int r = 1; r < 16; ++r) mm = fmaxf(mm, mk[r]);
              if (!__builtin_amdgcn_ballot_w64(mm > -1e30f) &&
                  !__builtin_amdgcn_ballot_w64(m <= -1e20f))
                continue;
            }
          }
          finish(bp, qk(bp), add_mask, mk);
        }
      }
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  for (int st = 0; st < nstage && !done; st += 2) {
    stage(st, I0{}, lds0, lds1);
    if (st + 1 < nstage && !done) stage(st + 1, I1{}, lds1, lds0);
  }

  if (!wave_rows) return;
  if constexpr (D != 128) {
    if (__builtin_expect(any_nan<NE>(o), 0)) {
      // everything uniform is read from the kernel arguments again: kept in
      // scalar registers for this rare path it spilled others in the loop
      // (D = 256, 512 over 4,700, soft-capped under a window: 105.1 us without the
      // path, 106.7 with it, 108.0 with the arguments kept)
      const KernelArgs<Src> ka;
      const AttnParams& pc = ka.p();
      const Src& sc = ka.src();
      const int hkc = blockIdx.y % pc.Hkv;
      const int lo_c = min(pc.lo, sc.n_pages(blockIdx.z));
      const int first = lo_c + (int)blockIdx.x * pc.pps;
      const int last = min(min(pc.hi, sc.n_pages(blockIdx.z)), first + pc.pps);
      const int row0 = (query_block(pc) * NW + (int)(threadIdx.x >> 6)) * kChunk32Rows;
      const RowCoord rw = row_coord(row0 + (row0 + jr < pc.G * pc.S ? jr : 0), pc.G);
      infinite_values<T, Src, FEAT, D>(
          pc, sc, blockIdx.z, hkc, first, 0, (last - first) * pc.bpp, 1, rw.g, rw.s, m * kLn2, lane,
          [&](float w, const uint16_t* v) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float wr = __shfl(w, 8 * (r >> 2) + 4 * hh + (r & 3), 64);
#pragma unroll
              for (int e = 0; e < NE; ++e) o[e][r] = with_infinite<T>(o[e][r], wr, v[32 * e + jr]);
            }
          });
    }
  }
  const float lrow = (lsum + __shfl_xor(lsum, 32, 64)) * kUnit;   // row jr's sum
  if (p.direct_out) {
    // the call's only split: normalized rows straight to the output
    // (HELM's final out / max(sum, 1e-12), kv_cache.py:554-555)
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = 8 * g + 4 * hh + t;
        const float inv = kUnit / fmaxf(__shfl(lrow, i, 64), 1e-12f);
        if (i < nrows)
#pragma unroll
          for (int e = 0; e < NE; ++e)
            *out_elem(g, t, e) = static_cast<uint16_t>(Ops::pk(o[e][4 * g + t] * inv, 0.f));
      }
    return;
  }
  // partials (m, l, o[D]) of the wave's rows in their 16-row tiles
  auto part_row = [&](int i) -> int64_t {
    return ((int64_t)(tile0 + (i >> 4)) * p.max_splits + split) * p.rows_per_tile + (i & 15);
  };
  const float m_nat = m * kLn2;   // the partials' max in natural units
  if (hh == 0 && jr < nrows)
    *reinterpret_cast<float2*>(&p.ws_ml[part_row(jr) * 2]) = make_float2(m_nat, lrow);
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int i = 8 * g + 4 * hh + t;
      if (i < nrows) {
        float* dst = &p.ws_o[part_row(i) * D + jr];
#pragma unroll
        for (int e = 0; e < NE; ++e) dst[32 * e] = o[e][4 * g + t] * kUnit;
      }
    }
}

template <typename T, class Src, int FEAT, int NW>
__global__ __launch_bounds__(NW * 64, 2) void chunk32_mfma_kernel(AttnParams p, Src src) {
  chunk32_mfma_body<T, Src, FEAT, NW, 128>(p, src);
}
// D = 64: 32 KiB of LDS and under 128 registers.  D = 256: the 128 KiB of its
// two stage buffers leave one workgroup per CU, and its 32 x 256 O tile and
// 32 x 256 query operand take 192 registers before any score: one wave per
// SIMD, which may use all 512.  Against the vector-ALU kernel, which read K
// and V once per four rows: f16 D = 64, 777 tokens over 2,777 (14 / 2 heads),
// 436 -> 29 us; bf16 D = 256, 512 over 4,700 soft-capped under a window mask
// (16 / 8 heads), 3,033 -> 108 us.
template <typename T, class Src, int FEAT, int NW, int D>
__global__ __launch_bounds__(NW * 64, D == 256 ? 1 : 2) void chunk32_mfma_dim_kernel(AttnParams p,
                                                                                     Src src) {
  chunk32_mfma_body<T, Src, FEAT, NW, D>(p, src);
}

}  // namespace helm
