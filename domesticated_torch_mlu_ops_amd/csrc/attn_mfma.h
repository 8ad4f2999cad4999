// attn_mfma: the MFMA kernel of single_query_cached_kv_attn (reference _ops.py:777-900) for gfx950;
// decode_attn.hip states the op and chooses the kernel, attn_mfma_*.hip instantiate it per kind of
// cache.
//
// bf16 or f16 operands, fp32 accumulation; K and V head sizes and cache rows all 64 / 128 / 256,
// block_size a multiple of 16, per-token or per-channel scales.  The query columns of a (sequence,
// KV head) are its (token, query head) pairs, c = s * g + head-in-group (g = Hq / Hkv), in blocks
// of 16.  A workgroup of four wavefronts owns one (sequence, KV head, split, column block) and its
// wavefronts take every fourth 16-token tile.  Per tile:
//   * S^T = K Q^T with v_mfma_f32_16x16x16 (tokens are the rows, the block's query columns the
//     columns, zero-padded to 16): lane (t = l % 16, c = l / 16) holds a quarter of token t's
//     row (one run of channels, or every fourth 16-byte vector: k_channel), and MFMA m takes
//     channels 4m .. + 3 of every lane group's own (a permutation of the reduction order).
//     Int8 codes enter as exact f16 values 1152 + code (two byte permutes per four codes) against
//     a power-of-two scaled f16 q, and 1152 * sum(q) is subtracted from the fp32 result; the
//     per-token scale and softmax_scale * log2(e) then multiply it.  Int4 codes enter as
//     3 + code / 8 (int4_f16), 3 * sum(q) is subtracted and the factor 8 joins the scale.
//   * The result layout (lane holds tokens 4c .. 4c + 3 of query column l % 16) IS the B
//     operand layout of O^T = V^T P^T, so the probabilities feed the second product without a
//     shuffle.  V^T's operand needs four tokens of one channel per lane: lane (n, c) reads
//     D/16 bytes of tokens 4c .. 4c + 3 at channels n D/16 .., and MFMA j uses channel
//     n D/16 + j of them, so lane (q, c) accumulates channels [4c D/16, (4c + 4) D/16) -- one
//     contiguous run of the output row.
//   * p (times the per-token V scale) is split into hi + lo bf16 operands (16 significant
//     bits) and two products accumulate, against V codes converted to bf16 exactly; q gets a
//     lo operand too when it is folded with per-channel key scales.
//   * Online softmax in base 2 per query column, each column masked to its own key range; a
//     lane keeps a partial sum over its own four tokens, summed over the lane groups at the
//     end.  The sink joins the denominator when the output is written.
// The four wavefronts combine through LDS; with more than one split per (sequence, KV head)
// the partials (max, sum, normalised row) go to a caller-provided workspace and a combine
// kernel merges them.
#pragma once

#include "attn_common.h"

namespace tmo {
namespace {

// kKind: 0 int8 caches (f16 QK, bf16 PV), 1 bf16 caches, 2 f16 caches, 3 float8_e4m3fn caches
// (as int8: f16 QK against the exact code values, no bias; bf16 PV), 4 int4 pairs (K pairing
// channels, V pairing the rows of a page; f16 QK through int4_f16, bf16 PV of the exact
// codes).  kQLo: q needs a lo operand.  kSB: the scale tensors are bf16 (else fp32).  kMask:
// a mask is given (its terms are added in the tiles that reach the last mask_len keys; the
// instances without one carry none of that code and its registers).  kPacked: the workgroups are
// numbered live ones first (work_of).
// Workgroups per CU the register allocation must allow: three (168 registers per lane) for
// the quantised-cache kernels up to head_size 128, fewer where that would spill.
constexpr bool attn_quant(int kind) { return kind == 0 || kind == 3 || kind == 4; }
constexpr int attn_min_blocks(int d, int kind) {
  return d == 256 ? 1 : (!attn_quant(kind) && d == 128 ? 2 : 3);
}

#ifndef TMO_ATTN_DEPTH
#define TMO_ATTN_DEPTH 2
#endif

template <int kD, int kKind, bool kQLo, bool kSB, bool kMask, bool kPacked>
__global__ __launch_bounds__(256, (attn_min_blocks(kD, kKind))) void attn_mfma(AttnParams p) {
  constexpr bool kQuant = attn_quant(kKind);  // codes with per-token / per-channel scales
  // tiles in flight per wavefront: three register sets where they fit the register budget of
  // attn_min_blocks (the quantised-cache kernels up to head_size 128)
  constexpr int kDepth = (kQuant && kD <= 128 && !kQLo) ? TMO_ATTN_DEPTH : 2;
  constexpr bool kF16 = kKind == 2;
  using M = Mfma<kF16>;
  using V4 = typename M::V4;
  constexpr int kDC = kD / 4;       // channels per lane group in the K layout
  constexpr int kDV = kD / 16;      // channels per lane in the V layout
  constexpr int kQK = kD / 16;      // QK MFMAs per tile
  constexpr int kEs = kQuant ? 1 : 2;  // cache element bytes
  constexpr bool kInt4 = kKind == 4;
  // Channel c of a lane's kDC is channel k_channel(c) of the row: runs of kKV channels, the lane
  // groups' runs in turn.  Rows of more than 128 bytes take runs of one 16-byte vector, so one
  // load of the wavefront covers 64 contiguous bytes of each token; with one run per lane it strode
  // over them, a quarter (bf16, 128 channels) of each 64-byte line at a time: 8 sequences of
  // 128..4096 keys, 32 / 8 heads x 128 bf16: 39.5 -> 34.0 us, 32 sequences of 512..4096 keys: 95 ->
  // 77 us.  Shorter rows take one run per lane: int8 and float8 rows of 128 bytes measured 0.2 to
  // 0.5 us longer in alternating vectors (4 sequences of up to 250 keys: 12.9 and 12.5 us against
  // 12.7 and 12.0).
  constexpr bool kAlt = !kInt4 && kD * kEs > 128;  // (int4 rows: 128 bytes at most)
  constexpr int kKV = kAlt ? 16 / kEs : kDC;

  const int lane = threadIdx.x & (kWave - 1);
  // wave-uniform (readfirstlane): the tile indices, page numbers and page offsets derived from it
  // stay in scalar registers, and the tile loads take a scalar base plus a per-lane offset
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane & 15;        // query column within the block / token row
  const int grp = lane >> 4;        // lane group c
  auto k_channel = [&](int c) -> int { return (c / kKV * 4 + grp) * kKV + c % kKV; };
  Work wk;
  if (!work_of<kPacked>(p, p.ncb, wk)) return;
  const int64_t i = wk.i;
  const int hk = wk.hk, split = wk.split;
  const int cb = wk.cb;  // column block
  const Seq sq = wk.sq;
  const Range rg = token_range(p, sq, split);
  // An empty split (past the sequence's keys) writes no partial; the combine skips it.  With
  // one split the (zero) output and lse are still written below.
  if (p.splits > 1 && rg.begin >= rg.end) return;
  // column c = token s * g + head hc: query head hk * g + hc of token s at position P
  const int c = cb * 16 + col;
  const int tok = c / p.g;
  const int hq = hk * p.g + (c - tok * p.g);
  const bool qvalid = c < p.ncols && token_valid(p, sq, tok);
  const int64_t qrow = sq.row0 + tok;

  // ---- Q operand (B of S^T = K Q^T): column `col`, channels k_channel(4m .. 4m + 3).  The QK
  // product runs on f16 operands: int8 codes as 1152 + code (codes_f16), q scaled by a power
  // of two sigma that puts the column's largest |q| in [2^14, 2^15) (an f16 holds every bf16
  // and f16 value of that column exactly down to 2^-29 of the largest), with a second (lo)
  // operand when q is folded with per-channel key scales.  Plain caches use their own type.
  using MQ = Mfma<kQuant ? true : kF16>;
  using VQ = typename MQ::V4;
  VQ qhi[kQK], qlo[kQLo ? kQK : 1];
  float qx[kQK][4];
  float qabs = 0.0f;
  // token positions fit in 32 bits (context lengths are int32).  Column keys: [klo, khi]
  // within the split, khi < klo when the column has none (or is padding).
  const int32_t pos = (int32_t)(sq.L - sq.nq) + tok;                 // the column's P
  int32_t klo = (int32_t)rg.begin, khi = (int32_t)rg.end - 1;
  if (p.window >= 0 && pos - (int32_t)p.window > klo) klo = pos - (int32_t)p.window;
  if (pos < khi) khi = pos;
  if (!qvalid) khi = klo - 1;
  // Tiles inside every valid column's keys need no per-key range test: [t0, t0 + 15] within
  // [wklo, wkhi], the largest klo and the smallest khi over the block's valid columns
  // (wave-uniform; the 16 columns are the lanes of each row, order-preserving u32 maxima).
  // Padding columns then carry scores of keys outside their range, which no output reads.
  int32_t wklo, wkhi;
  {
    const uint32_t lo = qvalid ? ((uint32_t)klo ^ 0x80000000u) : 0u;
    const uint32_t hi = qvalid ? ~((uint32_t)khi ^ 0x80000000u) : 0u;
    wklo = (int32_t)((uint32_t)__builtin_amdgcn_readfirstlane((int)group_max_u32<16>(lo)) ^
                     0x80000000u);
    wkhi = (int32_t)(~(uint32_t)__builtin_amdgcn_readfirstlane((int)group_max_u32<16>(hi)) ^
                     0x80000000u);
  }
  // The block's tiles: from its first valid token's window start to its last token's P
  // (wave-uniform: every lane computes the same numbers)
  int64_t bbeg = rg.begin, bend = rg.end;
  {
    const int64_t ntok = sq.nq < p.S ? sq.nq : p.S;
    const int64_t s_first = (int64_t)cb * 16 / p.g;
    int64_t s_last = ((int64_t)cb * 16 + 15) / p.g;
    if (s_last > ntok - 1) s_last = ntok - 1;
    const int64_t p_first = sq.L - sq.nq + s_first, p_last = sq.L - sq.nq + s_last;
    if (p.window >= 0 && p_first - p.window > bbeg) bbeg = p_first - p.window;
    if (p_last + 1 < bend) bend = p_last + 1;
    if (s_last < s_first || bend <= bbeg) bbeg = bend = 0;   // no key for the block: no tile
  }
  const int32_t first_tile = (int32_t)(bbeg >> 4);
  const int32_t end_tile = (int32_t)((bend + 15) >> 4);
  // the MFMA kernel takes tables of one row per sequence or per KV head
  const int32_t* bt_row = p.bt + (p.bt_heads ? i * p.bt_heads + hk : i) * p.max_blocks;
  auto page_of = [&](int32_t tl) -> int32_t {
    const int32_t t0 = tl * 16;
    return p.bs_shift >= 0 ? t0 >> p.bs_shift : t0 / p.BS;
  };
  // The wave's tiles are first_tile + wave + 4n.  Lane l holds the block of the window's
  // tile n = l (64 tiles per refill), read per tile with v_readlane.
  int32_t lane_blk = -1;
  int32_t win_base = first_tile + wave;
  auto refill = [&]() {
    const int32_t tl = win_base + 4 * lane;
    lane_blk = tl < end_tile ? bt_row[page_of(tl)] : -1;
  };
  // Start-up: the q row (and per-channel key scales) and the first block-table window are
  // independent reads, issued together -- q first, so the q arithmetic waits for q only and
  // the block ids arrive meanwhile; the first tile loads wait for the block ids alone.
  if (p.q_vec) {  // 16-byte aligned q rows of a 2-byte type: kDC / 8 vectors per lane
    constexpr int kQV = kDC / 8;
    u32x4 qraw[kQV];
    const uint16_t* qp = static_cast<const uint16_t*>(p.q) + i * p.q_sb + qrow * p.q_ss +
                         (int64_t)hq * p.q_sh;
#pragma unroll
    for (int v = 0; v < kQV; ++v)
      qraw[v] = qvalid ? *reinterpret_cast<const u32x4*>(qp + k_channel(8 * v))
                       : u32x4{0u, 0u, 0u, 0u};
    // per-channel key scales of the lane's channels, raw: fp32 (4 per vector) or bf16 (8)
    constexpr int kCS = kQuant ? (kSB ? kDC / 8 : kDC / 4) : 1;
    u32x4 kcs[kCS];
    if (kQuant && p.smode == 2) {
      const int64_t e0 = (int64_t)hk * kD;
#pragma unroll
      for (int v = 0; v < kCS; ++v)
        kcs[v] = kSB ? *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.ks) + e0 +
                                                       k_channel(8 * v))
                     : *reinterpret_cast<const u32x4*>(static_cast<const float*>(p.ks) + e0 +
                                                       k_channel(4 * v));
    }
    refill();
    const bool bf = p.q_dtype == TMO_DTYPE_BF16;
#pragma unroll
    for (int m = 0; m < kQK; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = qk_channel(kInt4, m, e);  // channel within the lane's run
        const uint32_t w = qraw[c / 8][(c % 8) / 2];
        const uint32_t h = (c & 1) ? (w >> 16) : (w & 0xffffu);
        float x = bf ? __uint_as_float(h << 16) : f16_bits_to_f32(h);
        if (kQuant && p.smode == 2) {
          if constexpr (kSB) {
            const uint32_t sw = kcs[c / 8][(c % 8) / 2];
            x *= __uint_as_float((c & 1) ? (sw & 0xffff0000u) : (sw << 16));
          } else {
            x *= __uint_as_float(kcs[c / 4][c % 4]);
          }
        }
        qx[m][e] = x;
        qabs = fmaxf(qabs, fabsf(x));
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < kQK; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = k_channel(qk_channel(kInt4, m, e));
        float x = qvalid ? load_q(p, i * p.q_sb + qrow * p.q_ss + (int64_t)hq * p.q_sh + d) : 0.0f;
        if (kQuant && p.qs_mode == 3 && qvalid)  // group-wise q scales (kQLo holds the rest)
          x *= q_group_scale(p, i * p.qs_sb + qrow * p.qs_ss + (int64_t)hq * p.qs_sh, d);
        if (kQuant && p.smode == 2) x *= scale_at(p.ks, (int64_t)hk * kD + d, kSB);
        qx[m][e] = x;
        qabs = fmaxf(qabs, fabsf(x));
      }
    }
    refill();
  }
  float inv_sigma = 1.0f, qk_off = 0.0f;
  if constexpr (kQuant) {
    qabs = col_max(qabs);
    // a column's largest |q| in [2^(ex-1), 2^ex); no lower than 2^-100, so that sigma stays finite
    const int ex = qabs > 0.0f ? max(__builtin_amdgcn_frexp_expf(qabs), -100) : 1;
    const float sigma = __builtin_ldexpf(1.0f, 15 - ex);
    inv_sigma = __builtin_ldexpf(1.0f, ex - 15);
    float qsum = 0.0f;
#pragma unroll
    for (int m = 0; m < kQK; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = qx[m][e] * sigma;
        const _Float16 h = (_Float16)y;
        qhi[m][e] = h;
        qsum += (float)h;
        if constexpr (kQLo) {
          const _Float16 l = (_Float16)(y - (float)h);
          qlo[m][e] = l;
          qsum += (float)l;
        }
      }
    }
    if constexpr (kKind == 0) qk_off = kCodeBias * col_sum(qsum);
    if constexpr (kInt4) qk_off = kInt4Bias * col_sum(qsum);
  } else {
#pragma unroll
    for (int m = 0; m < kQK; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kF16) {
          qhi[m][e] = (_Float16)qx[m][e];
        } else {
          qhi[m][e] = M::bits(qx[m][e]);
        }
      }
    }
  }
  const float alibi = (p.alibi && qvalid) ? p.alibi[i * p.Hq + hq] * kLog2e : 0.0f;
  // inv_sigma: an exact power of two; int4 operands carry the codes / 8; a per-tensor or
  // per-token q scale multiplies the column's scores (its q operand holds the exact codes)
  const float q_rs = (kQuant && qvalid && p.qs_mode)
                         ? q_row_scale(p, i * p.qs_sb + qrow * p.qs_ss + (int64_t)hq * p.qs_sh)
                         : 1.0f;
  const float score_scale = p.scale_log2 * inv_sigma * (kInt4 ? 8.0f : 1.0f) * q_rs;
  // mask: terms for keys [mask_lo, L), element mask_row + m for key mask_lo + m
  const int32_t mask_lo = (int32_t)sq.L - p.mask_len;

  float mrun = -__builtin_inff();   // running max (base 2) of this lane's column
  float lpart = 0.0f;               // this lane's share of the running sum
  f32x4 acc[kDV];
#pragma unroll
  for (int j = 0; j < kDV; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const char* kbase = static_cast<const char*>(p.kc);
  const char* vbase = static_cast<const char*>(p.vc);
  // cache row bytes: K rows of kD elements (int4: kD / 2 bytes of channel pairs); V rows of kD
  // elements (int4: pair rows of kD bytes, each two tokens, so a page is BS / 2 of them and
  // the same bytes as a K page)
  constexpr int kKRow = kInt4 ? kD / 2 : kD * kEs;
  constexpr int kVRow = kInt4 ? kD : kD * kEs;
  constexpr int kVRows = kInt4 ? 2 : 4;                     // V rows per lane: tokens 4 grp .. + 3
  const int64_t page_bytes = (int64_t)p.BS * kKRow;         // one head's page
  // per-lane offsets inside a 16-row piece of a page: K token `col`, the lane group's first run of
  // channels; V tokens 4 grp .. + 3, channels col * kDV ..
  constexpr int kKStep = kInt4 ? kKV / 2 : kKV * kEs;       // bytes of one run
  const int32_t k_lane = col * kKRow + grp * kKStep;
  const int32_t v_lane = kVRows * grp * kVRow + col * kDV * (kInt4 ? 1 : kEs);
  constexpr int kKW = kInt4 ? kDC / 8 : kDC * kEs / 4;      // dwords per lane
  constexpr int kVW = kInt4 ? kDV / 4 : kDV * kEs / 4;

  // Raw tile: this lane's K piece, its V pieces of four tokens, the per-token scales.
  // The per-token scales stay raw until the tile is computed (fp32 words, or bf16 pairs in
  // ks[0..1] / vs[0..1]): widening them at load time would wait for the loads there.
  struct Raw {
    uint32_t kw[kKW];
    uint32_t vw[kVRows][kVW];
    uint32_t ks[4], vs[4];
  };
  auto raw_scale = [](const uint32_t (&w)[4], int e) -> float {
    if constexpr (kSB) return __uint_as_float((e & 1) ? (w[e / 2] & 0xffff0000u) : (w[e / 2] << 16));
    return __uint_as_float(w[e]);
  };
  auto load_tile = [&](Raw& r, int32_t tl, int64_t blk) {
    const int32_t t0 = tl * 16;
    const int32_t row0 = t0 - page_of(tl) * p.BS;
    // the piece's offset in a K page; in an int4 V page (pair rows of kD bytes) row0 / 2 * kD
    // is the same number
    const int64_t piece = (blk * p.Hkv + hk) * page_bytes + (int64_t)row0 * kKRow;
    const char* krow = kbase + piece + k_lane;
    if constexpr (kKW >= 4) {
#pragma unroll
      for (int u = 0; u < kKW / 4; ++u) {
        const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(krow) + (kAlt ? 4 * u : u));
#pragma unroll
        for (int e = 0; e < 4; ++e) r.kw[4 * u + e] = w[e];
      }
    } else if constexpr (kKW == 2) {
      const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(krow));
      r.kw[0] = w[0];
      r.kw[1] = w[1];
    } else {
      r.kw[0] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(krow));
    }
#pragma unroll
    for (int e = 0; e < kVRows; ++e) {
      const char* vrow = vbase + piece + v_lane + e * kVRow;
      if constexpr (kVW == 4) {
        const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vrow));
#pragma unroll
        for (int u = 0; u < 4; ++u) r.vw[e][u] = w[u];
      } else if constexpr (kVW == 2) {
        const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(vrow));
        r.vw[e][0] = w[0];
        r.vw[e][1] = w[1];
      } else if constexpr (kVW == 1) {
        r.vw[e][0] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(vrow));
      } else {  // 32 bytes
        const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vrow));
        const u32x4 b = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vrow) + 1);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          r.vw[e][u] = a[u];
          r.vw[e][4 + u] = b[u];
        }
      }
    }
    constexpr uint32_t kOne = kSB ? 0x3f803f80u : 0x3f800000u;  // 1.0 (a bf16 pair)
#pragma unroll
    for (int e = 0; e < 4; ++e) r.ks[e] = r.vs[e] = kOne;
    if (kQuant && p.smode == 1) {
      const int32_t so = row0 + 4 * grp;
      const int64_t ka = blk * p.ks_sb + hk * p.ks_sh + so, va = blk * p.vs_sb + hk * p.vs_sh + so;
      if constexpr (kSB) {
        const u32x2 a = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p.ks) + ka);
        const u32x2 b = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p.vs) + va);
        r.ks[0] = a[0];
        r.ks[1] = a[1];
        r.vs[0] = b[0];
        r.vs[1] = b[1];
      } else {
        const u32x4 a = *reinterpret_cast<const u32x4*>(static_cast<const float*>(p.ks) + ka);
        const u32x4 b = *reinterpret_cast<const u32x4*>(static_cast<const float*>(p.vs) + va);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          r.ks[e] = a[e];
          r.vs[e] = b[e];
        }
      }
    }
  };

  // Arithmetic of one loaded tile (the whole wavefront: the MFMAs need every lane).
  auto compute_tile = [&](const Raw& r, int32_t tile) {
      const int32_t t0 = tile * 16;
      // ---- S^T = K Q^T
      f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int m = 0; m < kQK; ++m) {
        VQ a;
        if constexpr (kKind == 0) {
          a = codes_f16(r.kw[m]);
        } else if constexpr (kInt4) {
          a = int4_f16(r.kw[m >> 1], m & 1);
        } else if constexpr (kKind == 3) {
          a = fp8_f16(r.kw[m]);
        } else {
          u32x2 w;
          w[0] = r.kw[2 * m];
          w[1] = r.kw[2 * m + 1];
          a = __builtin_bit_cast(VQ, w);
        }
        s = MQ::run(a, qhi[m], s);
        if constexpr (kQLo) s = MQ::run(a, qlo[m], s);
      }

      // ---- scores (base 2), masking, online softmax
      float sc[4];
      float tmax = -__builtin_inff();
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[e] = (s[e] - qk_off) * (raw_scale(r.ks, e) * score_scale);
      // ALiBi and the key-range test as wave-uniform branches (if-converted, both ran on
      // every tile: ~36 VALU per tile, a tenth of the int4 kernel's)
      if (p.alibi) {
        keep_branch();
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[e] += alibi * (float)(t0 + 4 * grp + e - pos);
      }
      if (t0 < wklo || t0 + 15 > wkhi) {
        keep_branch();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int32_t j = t0 + 4 * grp + e;
          if (j < klo || j > khi) sc[e] = -__builtin_inff();
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) tmax = fmaxf(tmax, sc[e]);
      // mask terms of the last mask_len keys: only the tiles that reach them (wave-uniform)
      if (kMask && t0 + 15 >= mask_lo) {
        // the column's row of terms (recomputed here: nothing stays live across the tiles;
        // a padding column reads token S - 1's row, in bounds, and its scores stay -inf)
        const int ct = (cb * 16 + col) / p.g;
        const int64_t mask_row = i * p.m_sb + (int64_t)(ct < p.S ? ct : p.S - 1) * p.m_ss;
        tmax = -__builtin_inff();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int32_t j = t0 + 4 * grp + e;
          if (j >= mask_lo) sc[e] += mask_value(p, mask_row + (j - mask_lo)) * kLog2e;
          tmax = fmaxf(tmax, sc[e]);
        }
      }
      tmax = col_max(tmax);
      // No branch on the column's state: the MFMAs below need the whole wavefront.  The
      // reference maximum moves only when a score exceeds it by more than kLazy (base 2), so
      // the probabilities stay below 2^kLazy and the accumulators are rarely rescaled; the
      // first finite score sets it.
      const bool was_empty = mrun == -__builtin_inff();
      const bool raise = tmax > mrun + kLazy || (was_empty && tmax != -__builtin_inff());
      const float mnew = raise ? tmax : mrun;
      const bool live = mnew != -__builtin_inff();          // some key of this column so far
      const float corr = raise ? __builtin_amdgcn_exp2f(mrun - mnew) : 1.0f;  // -inf -> 0
      mrun = mnew;
      float pe[4];
      float psum = 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pe[e] = live ? __builtin_amdgcn_exp2f(sc[e] - mnew) : 0.0f;  // masked: -inf -> 0
        psum += pe[e];
      }
      lpart = lpart * corr + psum;
      if (__ballot(corr != 1.0f && !was_empty)) {  // an empty column's accumulators are zero
#pragma unroll
        for (int j = 0; j < kDV; ++j) acc[j] *= corr;
      }

      // ---- P^T operands (hi + lo) with the per-token V scale folded in
      V4 phi, plo;
      if constexpr (!kF16) {
        // bf16 pairs: one v_cvt_pk_bf16_f32 rounds two probabilities (hi), the hi values are
        // read back from the packed bits, and one more rounds the two remainders (lo)
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        u32x2 hv, lv;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const f2 a = {pe[2 * k] * raw_scale(r.vs, 2 * k), pe[2 * k + 1] * raw_scale(r.vs, 2 * k + 1)};
          const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(a, bf2));
          const f2 l = {a[0] - __uint_as_float(h << 16), a[1] - __uint_as_float(h & 0xffff0000u)};
          hv[k] = h;
          lv[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(l, bf2));
        }
        phi = __builtin_bit_cast(V4, hv);
        plo = __builtin_bit_cast(V4, lv);
      } else
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pv = pe[e] * raw_scale(r.vs, e);
        if constexpr (kF16) {
          const _Float16 h = (_Float16)pv;
          phi[e] = h;
          plo[e] = (_Float16)(pv - (float)h);
        } else {
          const short hb = M::bits(pv);
          phi[e] = hb;
          plo[e] = M::bits(pv - M::value(hb));
        }
      }

      // int4 V: the nibbles of token 4 grp + e moved into the high half of their bytes, so
      // each byte read as signed is 16 x the code (the low nibble shifted up, the other half
      // cleared; one mask per dword, kept whole in a register -- left to the combiner, the
      // masks were split into per-byte shifts and extractions)
      uint32_t vm[kInt4 ? 4 : 1][kInt4 ? kVW : 1];
      if constexpr (kInt4) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int u = 0; u < kVW; ++u) {
            const uint32_t w = r.vw[e >> 1][u];
            uint32_t m = ((e & 1) ? (w << 4) : w) & 0xF0F0F0F0u;
            asm("" : "+v"(m));
            vm[e][u] = m;
          }
      }

      // ---- O^T += V^T P^T: MFMA j takes channel col * kDV + j of tokens 4 grp .. + 3
#pragma unroll
      for (int j = 0; j < kDV; ++j) {
        typedef short s4 __attribute__((ext_vector_type(4)));
        s4 b4;
        if constexpr (kKind == 0) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int8_t code = (int8_t)(r.vw[e][j >> 2] >> (8 * (j & 3)));
            b4[e] = (short)(__float_as_uint((float)code) >> 16);
          }
        } else if constexpr (kInt4) {
          // channel j's byte of pair row e / 2 holds tokens 4 grp + e (high nibble, e even)
          // and + 1 (low nibble); byte j & 3 of the masked dword is 16 x the code: one
          // sign-extending byte conversion, as for int8 codes, exact as bf16.  The factor 16
          // leaves with the normalisation (exactly: a power of two).
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int8_t c16 = (int8_t)(vm[e][j >> 2] >> (8 * (j & 3)));
            b4[e] = (short)(__float_as_uint((float)c16) >> 16);
          }
        } else if constexpr (kKind == 3) {
          // the e4m3fn value's fp32 pattern truncated to bf16 is exact (<= 4 significant bits)
#pragma unroll
          for (int e = 0; e < 4; ++e) b4[e] = (short)(__float_as_uint(fp8_value(r.vw[e][j >> 2], j & 3)) >> 16);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) b4[e] = (short)(r.vw[e][j >> 1] >> (16 * (j & 1)));
        }
        const V4 a = __builtin_bit_cast(V4, b4);
        acc[j] = M::run(a, phi, acc[j]);
        acc[j] = M::run(a, plo, acc[j]);
      }
  };

  // Register sets rotate: while one tile is computed the loads of the next kDepth - 1 tiles
  // are in flight (no copies between the sets).
  int32_t slot = 0;  // index in the window of the most recently loaded tile
  Raw ra, rb;
  int32_t tile = first_tile + wave;
  // Every call issues a tile's loads: a tile past the wave's range or on a missing page (its
  // keys masked) re-reads the wave's last valid tile (in bounds and just read; page 0 before
  // any) and is not computed.  With the loads under a branch, the register set was assigned
  // on one path only, and the copies that merged it waited for the loads just issued -- the
  // next tile's -- before the current tile was computed.
  int32_t safe_tl = first_tile + wave;
  int64_t safe_blk = 0;
  auto try_load = [&](Raw& r, int32_t tl) -> bool {
    const int64_t blk = __builtin_amdgcn_readlane(lane_blk, slot);
    const bool ok = tl < end_tile && blk >= 0 && blk < p.NB;  // wave-uniform
    if (ok) {
      safe_tl = tl;
      safe_blk = blk;
    }
    load_tile(r, safe_tl, safe_blk);
    return ok;
  };
  auto advance = [&]() {
    if (++slot == kWave) {
      win_base += 4 * kWave;
      refill();
      slot = 0;
    }
  };
  bool ok_a = try_load(ra, tile);
  if constexpr (kDepth == 3) {
    Raw rc;
    advance();
    bool ok_b = try_load(rb, tile + 4);
    while (tile < end_tile) {
      advance();
      const bool ok_c = try_load(rc, tile + 8);
      if (ok_a) compute_tile(ra, tile);
      tile += 4;
      if (tile >= end_tile) break;
      advance();
      ok_a = try_load(ra, tile + 8);
      if (ok_b) compute_tile(rb, tile);
      tile += 4;
      if (tile >= end_tile) break;
      advance();
      ok_b = try_load(rb, tile + 8);
      if (ok_c) compute_tile(rc, tile);
      tile += 4;
    }
  } else {
    while (tile < end_tile) {
      advance();
      const bool ok_b = try_load(rb, tile + 4);
      if (ok_a) compute_tile(ra, tile);
      tile += 4;
      if (tile >= end_tile) break;
      advance();
      ok_a = try_load(ra, tile + 4);
      if (ok_b) compute_tile(rb, tile);
      tile += 4;
    }
  }

  // ---- combine the four wavefronts: waves 1..3 leave (max, sum, accumulators) in LDS in
  // their lane layout, wave 0 merges them into its own registers lane by lane and writes
  const float lsum = col_sum(lpart);
  __shared__ float lds_m[4][16];
  __shared__ float lds_l[4][16];
  // lane-major partial rows, padded by one float: lane l's value k at l * (4 kDV + 1) + k, so
  // the 64 lanes of one store or load hit 64 different banks (a [col][channel] layout put the
  // 16 columns of a wavefront on one bank)
  constexpr int kRow = 4 * kDV + 1;
  __shared__ float lds_o[3][kWave * kRow];
  if (grp == 0) {
    lds_m[wave][col] = mrun;
    lds_l[wave][col] = lsum;
  }
  if (wave > 0) {
#pragma unroll
    for (int j = 0; j < kDV; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) lds_o[wave - 1][lane * kRow + e * kDV + j] = acc[j][e];
  }
  __syncthreads();
  if (wave != 0) return;
  float mx = -__builtin_inff();
#pragma unroll
  for (int w = 0; w < 4; ++w) mx = fmaxf(mx, lds_m[w][col]);
  float f[4];
  float lt = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    f[w] = mx == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(lds_m[w][col] - mx);
    lt += lds_l[w][col] * f[w];
  }
  if (!qvalid) return;
  const bool direct = p.splits == 1;
  float lse_v;
  // int4 V operands carry 16 x the codes: the power-of-two factor is exact, so the outputs
  // are those of the codes themselves bit for bit
  const float inv = (direct ? finish(p, hq, mx, lt, &lse_v) : (lt > 0.0f ? 1.0f / lt : 0.0f)) *
                    (kInt4 ? 0.0625f : 1.0f);
  float* ws_row = p.ws + ((((i * p.Hkv + hk) * p.splits + split) * p.ncols + c) * (int64_t)(kD + 2));
  if (!direct && grp == 0) {
    ws_row[0] = mx;
    ws_row[1] = lt;
  }
  const int64_t orow = i * p.o_sb + qrow * p.o_ss + (int64_t)hq * p.o_sh;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int j = 0; j < kDV; ++j) {
      const int d = kDV * (4 * grp + e) + j;
      float o = acc[j][e] * f[0];
#pragma unroll
      for (int w = 1; w < 4; ++w) o += lds_o[w - 1][lane * kRow + e * kDV + j] * f[w];
      o *= inv;
      if (kQuant && p.smode == 2) o *= scale_at(p.vs, (int64_t)hk * kD + d, kSB);  // per-channel V
      if (direct) {
        store_out(p, orow + d, o);
      } else {
        ws_row[2 + d] = o;
      }
    }
  }
  if (direct && grp == 0 && p.lse) p.lse[i * p.lse_sb + qrow * p.lse_ss + (int64_t)hq * p.lse_sh] = lse_v;
}

template <int kD, int kKind, bool kQLo, bool kSB>
int launch_mfma_q(const AttnParams& p, hipStream_t st) {
  const dim3 grid = attn_grid(p, p.ncb), block(256);
  if (p.packed)
    return p.mask ? launch_kernel(attn_mfma<kD, kKind, kQLo, kSB, true, true>, grid, block, st, p)
                  : launch_kernel(attn_mfma<kD, kKind, kQLo, kSB, false, true>, grid, block, st, p);
  return p.mask ? launch_kernel(attn_mfma<kD, kKind, kQLo, kSB, true, false>, grid, block, st, p)
                : launch_kernel(attn_mfma<kD, kKind, kQLo, kSB, false, false>, grid, block, st, p);
}

template <int kD, int kKind, bool kSB>
int launch_mfma_d(const AttnParams& p, bool qlo, hipStream_t st) {
  if constexpr (attn_quant(kKind)) {  // q of 16-bit caches is their own type: no lo operand
    if (qlo) return launch_mfma_q<kD, kKind, true, kSB>(p, st);
  }
  return launch_mfma_q<kD, kKind, false, kSB>(p, st);
}

template <int kKind, bool kSB>
int launch_mfma(const AttnParams& p, bool qlo, hipStream_t st) {
  switch (p.D) {
    case 64: return launch_mfma_d<64, kKind, kSB>(p, qlo, st);
    case 128: return launch_mfma_d<128, kKind, kSB>(p, qlo, st);
    default: return launch_mfma_d<256, kKind, kSB>(p, qlo, st);
  }
}

// Caches of kind kKind, their scales of either type (16-bit caches have none).
template <int kKind>
int launch_mfma(const AttnParams& p, bool qlo, hipStream_t st) {
  if constexpr (attn_quant(kKind)) {
    if (p.s_bf16) return launch_mfma<kKind, true>(p, qlo, st);
  }
  return launch_mfma<kKind, false>(p, qlo, st);
}

}  // namespace
}  // namespace tmo
