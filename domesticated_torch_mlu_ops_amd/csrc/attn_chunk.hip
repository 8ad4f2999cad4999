// Attention of many query columns per (sequence, KV head) over paged caches, for gfx950:
// chunked prefill and several query tokens per sequence (single_query_cached_kv_attn, reference
// _ops.py:777-900; the forms and softmax are those of decode_attn.hip; ALiBi and mask terms are
// left to attn_mfma).
//
// What bounds it: with hundreds of query columns per KV head the keys and values come from L2 and
// the work is arithmetic.  attn_mfma gives 16 columns a workgroup, so each 16 columns unpacked
// every key and value code again (about 300 VALU instructions per 16 keys, against 24 MFMAs).
// Here a workgroup of four wavefronts owns 64 * kC columns (kC blocks of 16 per wavefront) and a
// tile of keys and values is unpacked once, into LDS, for all of them:
//   * The raw rows of the next tile are loaded into registers while a tile is computed, then
//     converted (int8 / int4 / float8_e4m3fn codes to exact f16 for K and exact bf16 for V) and
//     written to the other LDS buffer; one barrier per tile.
//   * K is the operand of S^T = K Q^T (v_mfma_f32_16x16x32), V of O^T = V^T P^T
//     (ds_read_b64_tr_b16 transposes it); each operand read from LDS serves kC column blocks.
//     The 16-byte chunk index is XORed with the row's low four bits (three for 128-byte rows),
//     as in attn_latent.hip.
//   * The softmax costs as much as the MFMAs, so it is kept short: scores meet the token's scale
//     once, the column's scale and maximum in the exponential's FMA, and the maximum over the
//     lane groups uses the permlane swaps.
// 8 chunks of up to 512 tokens over 1019..8192 int8 keys, 32 query and 8 KV heads x 128 (0.24
// TFLOP): 1205 us on attn_mfma, 437 us here (550 TFLOP/s).  Per wavefront and 64 keys that is
// about 500 VALU instructions, 64 exponentials' cycles and 96 MFMAs, which overlap little.  What
// it took: no spilled register inside the loop (a reload waits for the rows in flight), hence
// the scheduling barriers and no ALiBi path; operands read from LDS a step ahead.
// p stays hi + lo operands (16 significant bits), q gets a lo operand when folded with
// per-channel scales, as in attn_mfma.
#include "attn_common.h"

namespace tmo {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// Maximum over the four lane groups of a column (lanes l, l ^ 16, l ^ 32, l ^ 48), in VALU.
__device__ __forceinline__ float col_max_swap(float v) {
  const uint32_t u = __float_as_uint(v);
  auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const float m = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const uint32_t w = __float_as_uint(m);
  auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Four bytes u (a code plus kBias - 1024, unsigned) -> four f16 codes: 0x6400 | u is 1024 + u
// exactly, and the subtraction of kBias is exact.
template <int kBias>
__device__ __forceinline__ u32x2 bytes_f16(uint32_t u) {
  u32x2 r;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t w = __builtin_amdgcn_perm(0x64646464u, u, k ? 0x04030402u : 0x04010400u);
    const h2 x = __builtin_bit_cast(h2, w) - h2{(_Float16)kBias, (_Float16)kBias};
    r[k] = __builtin_bit_cast(uint32_t, x);
  }
  return r;
}

// Four signed bytes -> four bf16 values (exact).
__device__ __forceinline__ u32x2 bytes_bf16(uint32_t w) {
  u32x2 r;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float a = (float)(int8_t)(w >> (16 * k)), b = (float)(int8_t)(w >> (16 * k + 8));
    r[k] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
  }
  return r;
}
__device__ __forceinline__ u32x2 fp8_bf16(uint32_t w) {
  u32x2 r;
#pragma unroll
  for (int k = 0; k < 2; ++k)
    r[k] = __builtin_amdgcn_perm(__float_as_uint(fp8_value(w, 2 * k + 1)),
                                 __float_as_uint(fp8_value(w, 2 * k)), 0x07060302u);
  return r;
}

constexpr bool chunk_quant(int kind) { return kind == 0 || kind == 3 || kind == 4; }

// Geometry of head size kD over caches of kind kKind (attn_mfma's kinds).
template <int kD, int kKind, bool kQLo>
struct Geo {
  static constexpr bool kQuant = chunk_quant(kKind);
  static constexpr bool kInt4 = kKind == 4;
  static constexpr int kT = kD > 128 ? 32 : 64;             // keys per tile
  // column blocks per wavefront (256 registers per lane: two workgroups per CU)
  static constexpr int kC = kD > 128 || kQLo ? 1 : 2;
  static constexpr int kQM = (kD + 31) / 32;                // QK MFMAs per 16 keys
  static constexpr int kVB = kD / 16;                       // value channel blocks
  static constexpr int kPitch = kD <= 64 ? 128 : (kD <= 128 ? 256 : 512);  // LDS row bytes
  static constexpr int kX = kPitch >= 256 ? 15 : 7;         // row bits XORed into the chunk index
  static constexpr int kKRow = kInt4 ? kD / 2 : kD * (kQuant ? 1 : 2);     // cache row bytes
  static constexpr int kVRow = kD * (kQuant ? 1 : 2);       // (int4: a pair row of two tokens)
  static constexpr int kKU = kKRow / 16, kVU = kVRow / 16;  // 16-byte units per row
  static constexpr int kVRows = kInt4 ? kT / 2 : kT;
  static constexpr int kKL = (kT * kKU + 255) / 256;        // units per thread and tile
  static constexpr int kVL = (kVRows * kVU + 255) / 256;
};

// Workgroups per CU: two, and three where they fit (16-bit caches, head size 64: 191 us with two
// for 8 chunks of up to 256 tokens over 8192 keys, 171 with three).
// kFit: splits as long as the contexts present need (fitted_split).  That costs a workgroup's start
// 0.5 to 1 us, so head sizes 80 and 96, whose calls had no faster kernel, keep the announced ones.
template <int kD, int kKind, bool kQLo, bool kFit>
__global__ __launch_bounds__(256, kD <= 64 && !chunk_quant(kKind) ? 3 : 2) void attn_chunk(AttnParams p) {
  using G = Geo<kD, kKind, kQLo>;
  constexpr bool kQuant = G::kQuant, kInt4 = G::kInt4;
  constexpr bool kF16K = kQuant || kKind == 2, kF16V = kKind == 2;
  constexpr int kT = G::kT, kC = G::kC, kQM = G::kQM, kVB = G::kVB, kTT = kT / 16;
  constexpr int kPitch = G::kPitch;
  __shared__ __align__(128) char lds_k[2][kT * kPitch];
  __shared__ __align__(128) char lds_v[2][kT * kPitch];
  __shared__ __align__(16) float lds_ks[2][kT], lds_vs[2][kT];

  touch_params();
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int col = lane & 15, grp = lane >> 4;
  // Longest sequences first, and of each the last column groups, which see the most keys: 707
  // -> 437 us for 8 chunks of up to 512 tokens over 1019..8192 int8 keys.  The KV heads of a
  // group are consecutive workgroups: with 8 of them, one per XCD and its L2.
  const int32_t own = lane_length(p);
  const int64_t i = seq_by_length(p, (int)blockIdx.y, own);
  const int hk = (int)(blockIdx.x % (unsigned)p.Hkv);
  const unsigned yr = (gridDim.x - 1 - blockIdx.x) / (unsigned)p.Hkv;
  const int cbg = (int)(yr / (unsigned)p.splits);  // group of 4 kC column blocks
  const int split = (int)yr - cbg * p.splits;
  const Seq sq = seq_of(p, i);
  const int64_t per = kFit ? fitted_split(p, own) : p.split_tokens;
  const Range rg = token_range(p, sq, split, per);
  if (p.splits > 1 && rg.begin >= rg.end) return;  // an empty split writes no partial
  const bool direct = live_splits(p, sq, per) <= 1;  // no merge: the only split writes the output

  // the workgroup's keys: from its first token's window start to its last token's position
  constexpr int kCols = 64 * kC;
  const int64_t ntok = sq.nq < p.S ? sq.nq : p.S;
  const int64_t s_first = (int64_t)cbg * kCols / p.g;
  if (s_first >= ntok) return;                     // no query token (workgroup-uniform)
  int64_t bbeg = rg.begin, bend = rg.end;
  int32_t all_lo, all_hi;  // all of its tokens see the keys from all_lo to all_hi
  {
    int64_t s_last = ((int64_t)cbg * kCols + kCols - 1) / p.g;
    if (s_last > ntok - 1) s_last = ntok - 1;
    const int64_t p_first = sq.L - sq.nq + s_first, p_last = sq.L - sq.nq + s_last;
    if (p.window >= 0 && p_first - p.window > bbeg) bbeg = p_first - p.window;
    if (p_last + 1 < bend) bend = p_last + 1;
    if (bend <= bbeg) bbeg = bend = 0;
    all_lo = (int32_t)(p.window >= 0 && p_last - p.window > bbeg ? p_last - p.window : bbeg);
    all_hi = (int32_t)(p_first < bend - 1 ? p_first : bend - 1);
  }
  const int32_t kbeg = (int32_t)bbeg & ~15, kend = (int32_t)bend;  // tiles on 16-key boundaries
  const int32_t tiles = (kend - kbeg + kT - 1) / kT;
  // Tiles before rag_lo and from rag_hi on hold keys that some token does not see.  p = 0 does not
  // remove a value that is no number, so the values of these tiles are checked in LDS: those that
  // are none become zeros, and the columns that see them get them after the loop.  Only tiles at
  // the causal edge and at a window's start are (none of one token without a window): 0.2 to 1.4%
  // of the times of 512-token chunks, up to 5% of short calls (16 tokens of 32 sequences of 512
  // bf16 keys x 128: 28.4 -> 29.3 us).
  const int32_t rag_lo = (all_lo - kbeg + kT - 1) / kT;
  const int32_t rag_hi = all_hi >= kend - 1 ? INT32_MAX : all_hi < kbeg ? 0 : (all_hi - kbeg + 1) / kT;

  // ---- staging
  const int32_t* bt_row = p.bt + (p.bt_heads ? i * p.bt_heads + hk : i) * p.max_blocks;
  auto page_index = [&](int32_t t) -> int32_t { return p.bs_shift >= 0 ? t >> p.bs_shift : t / p.BS; };
  // Lane l holds, for the 16 keys kbeg + 16 (win + l) .. (one page), the cache row of the first
  // key and of its scales, -1 when there is no page; bit l of `bad` is set then.
  int32_t win = 0, lane_row = -1, lane_ks = 0, lane_vs = 0;
  uint64_t bad = 0;
  auto refill = [&]() {
    const int32_t t = kbeg + (win + lane) * 16;
    const int32_t pg = page_index(t), off = t - pg * p.BS;
    const int32_t blk = t < kend ? bt_row[pg] : -1;
    const bool ok = blk >= 0 && blk < p.NB;
    lane_row = ok ? (int32_t)((blk * (int64_t)p.Hkv + hk) * p.BS + off) : -1;
    if (kQuant && p.smode == 1) {
      lane_ks = ok ? (int32_t)(blk * p.ks_sb + hk * p.ks_sh + off) : 0;
      lane_vs = ok ? (int32_t)(blk * p.vs_sb + hk * p.vs_sh + off) : 0;
    }
    bad = __ballot(!ok);
  };
  u32x4 kw[G::kKL], vw[G::kVL];
  uint32_t kok = 0, vok = 0;       // bit j: unit j holds keys
  uint16_t sc_hi = 0, sc_lo = 0;   // raw scale of key `lane` (even wavefronts) or value (odd)
  bool sc_ok = false;
  uint32_t bad_next = 0;           // missing 16-key groups of the tile in flight
  const char* sc_base = static_cast<const char*>((wave & 1) ? p.vs : p.ks);
  const int sc_shift = p.s_bf16 ? 1 : 2;
  auto issue = [&](int32_t tile) {
    if (tile * kTT >= win + kWave) {
      win += kWave;
      refill();
    }
    const int slot0 = tile * kTT - win;
    const int32_t left = kend - (kbeg + tile * kT);  // keys of the tile
    bad_next = (uint32_t)(bad >> slot0) & ((1u << kTT) - 1u);
    kok = vok = 0;
    // Lane shuffles first, then the loads, all unconditional: a row without a key reads row 0.
    // int4 V: pair row r holds keys 2r and 2r + 1 of one page (row even).
    int32_t kg[G::kKL], vg[G::kVL], e = 0;
    auto key_of_k = [&](int j) { const int r = (tid + 256 * j) / G::kKU; return r < kT ? r : kT - 1; };
    auto key_of_v = [&](int j) {
      const int r = (tid + 256 * j) / G::kVU * (kInt4 ? 2 : 1);
      return r < kT ? r : kT - (kInt4 ? 2 : 1);
    };
    const int rs = lane < kT ? lane : kT - 1;
#pragma unroll
    for (int j = 0; j < G::kKL; ++j) kg[j] = __shfl(lane_row, slot0 + (key_of_k(j) >> 4), kWave);
#pragma unroll
    for (int j = 0; j < G::kVL; ++j) vg[j] = __shfl(lane_row, slot0 + (key_of_v(j) >> 4), kWave);
    if constexpr (kQuant) e = __shfl((wave & 1) ? lane_vs : lane_ks, slot0 + (rs >> 4), kWave);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kQuant) {
      sc_ok = rs < left && !(bad_next >> (rs >> 4) & 1);
      const int64_t at = sc_ok && p.smode == 1 ? (int64_t)(e + (rs & 15)) << sc_shift : 0;
      sc_hi = *reinterpret_cast<const uint16_t*>(sc_base + at + (sc_shift == 2 ? 2 : 0));
      sc_lo = *reinterpret_cast<const uint16_t*>(sc_base + at);
    }
#pragma unroll
    for (int j = 0; j < G::kKL; ++j) {
      const int u = tid + 256 * j, r = key_of_k(j);
      kok |= (uint32_t)(kg[j] >= 0 && r < left) << j;
      const int64_t row = kg[j] >= 0 ? kg[j] + (r & 15) : 0;
      kw[j] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(p.kc) + row * G::kKRow +
                                              (u % G::kKU) * 16);
    }
#pragma unroll
    for (int j = 0; j < G::kVL; ++j) {
      const int u = tid + 256 * j, r = key_of_v(j);
      vok |= (uint32_t)(vg[j] >= 0 && r < left) << j;
      const int64_t row = vg[j] >= 0 ? vg[j] + (r & 15) : 0;
      vw[j] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(p.vc) +
                                              (kInt4 ? row >> 1 : row) * G::kVRow + (u % G::kVU) * 16);
    }
  };
  auto put = [&](char* base, int r, int chunk, u32x4 w) {
    *reinterpret_cast<u32x4*>(base + r * kPitch + ((chunk ^ (r & G::kX)) << 4)) = w;
  };
  // Convert the rows in flight and write them to LDS buffer `buf`; rows without a key are zeros,
  // or integer codes with scale 0.  float8 values of no key are cleared too: whatever row 0 or a
  // page's rest holds there may be NaN codes, and p = 0 would not remove those (K's scores of no
  // key are replaced).
  auto stage = [&](int buf) {
#pragma unroll
    for (int j = 0; j < G::kKL; ++j) {
      const int u = tid + 256 * j, r = u / G::kKU, c = u - r * G::kKU;
      if (kT * G::kKU % 256 != 0 && u >= kT * G::kKU) continue;
      u32x4 w = kw[j];
      if (!kQuant && !(kok >> j & 1)) w = u32x4{0u, 0u, 0u, 0u};
      if constexpr (!kQuant) {
        put(lds_k[buf], r, c, w);
      } else if constexpr (kInt4) {
        // byte b of a dword: channels 2b (high nibble), 2b + 1 (low): bytes u = code + 8
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint32_t x = w[h] ^ 0x88888888u;
          const uint32_t hi = (x >> 4) & 0x0f0f0f0fu, lo = x & 0x0f0f0f0fu;
          const u32x2 a = bytes_f16<1032>(__builtin_amdgcn_perm(lo, hi, 0x05010400u));
          const u32x2 b = bytes_f16<1032>(__builtin_amdgcn_perm(lo, hi, 0x07030602u));
          put(lds_k[buf], r, 4 * c + h, u32x4{a[0], a[1], b[0], b[1]});
        }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          u32x2 a, b;
          if constexpr (kKind == 3) {
            a = __builtin_bit_cast(u32x2, fp8_f16(w[2 * h]));
            b = __builtin_bit_cast(u32x2, fp8_f16(w[2 * h + 1]));
          } else {
            a = bytes_f16<1152>(w[2 * h] ^ 0x80808080u);
            b = bytes_f16<1152>(w[2 * h + 1] ^ 0x80808080u);
          }
          put(lds_k[buf], r, 2 * c + h, u32x4{a[0], a[1], b[0], b[1]});
        }
      }
    }
#pragma unroll
    for (int j = 0; j < G::kVL; ++j) {
      const int u = tid + 256 * j, r = u / G::kVU, c = u - r * G::kVU;
      if (G::kVRows * G::kVU % 256 != 0 && u >= G::kVRows * G::kVU) continue;
      u32x4 w = vw[j];
      if ((!kQuant || kKind == 3) && !(vok >> j & 1)) w = u32x4{0u, 0u, 0u, 0u};
      if constexpr (!kQuant) {
        put(lds_v[buf], r, c, w);
      } else {
        // int4: the nibbles of key 2r (high) and 2r + 1 as 16 x code bytes; the factor leaves
        // with the normalisation
#pragma unroll
        for (int k = 0; k < (kInt4 ? 2 : 1); ++k)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            u32x2 a, b;
            if constexpr (kKind == 3) {
              a = fp8_bf16(w[2 * h]);
              b = fp8_bf16(w[2 * h + 1]);
            } else if constexpr (kInt4) {
              a = bytes_bf16((k ? w[2 * h] << 4 : w[2 * h]) & 0xf0f0f0f0u);
              b = bytes_bf16((k ? w[2 * h + 1] << 4 : w[2 * h + 1]) & 0xf0f0f0f0u);
            } else {
              a = bytes_bf16(w[2 * h]);
              b = bytes_bf16(w[2 * h + 1]);
            }
            put(lds_v[buf], kInt4 ? 2 * r + k : r, 2 * c + h, u32x4{a[0], a[1], b[0], b[1]});
          }
      }
    }
    if (kQuant && p.smode == 1 && wave < 2 && lane < kT) {
      const uint32_t w = ((uint32_t)sc_hi << 16) | (sc_shift == 2 ? sc_lo : 0u);
      (wave == 0 ? lds_ks : lds_vs)[buf][lane] = sc_ok ? __uint_as_float(w) : 0.0f;
    }
  };

  // channels past kD that the last QK MFMA reads are zeros, for good
  if constexpr (kD % 32 != 0) {
    for (int x = tid; x < 2 * kT * 2; x += 256) {
      const int buf = x & 1, r = (x >> 2), c = kD / 8 + ((x >> 1) & 1);
      put(lds_k[buf], r, c, u32x4{0u, 0u, 0u, 0u});
    }
  }
  if (kQuant && p.smode != 1) {
    for (int x = tid; x < kT; x += 256)
      lds_ks[0][x] = lds_ks[1][x] = lds_vs[0][x] = lds_vs[1][x] = 1.0f;
  }
  if (tiles > 0) {
    refill();
    issue(0);
  }

  // ---- the wavefront's columns: c = token s * g + head hc
  u32x4 qhi[kC][kQM], qlo[kQLo ? kC : 1][kQLo ? kQM : 1];
  float sscale[kC], mrun[kC], lpart[kC];
  int32_t klo[kC];
  uint32_t kspan[kC];         // keys klo .. klo + kspan of the column
  bool qvalid[kC];
  int32_t wklo = INT32_MIN, wkhi = INT32_MAX;  // keys inside every valid column's range
#pragma unroll
  for (int cb = 0; cb < kC; ++cb) {
    const int c = cbg * kCols + (wave * kC + cb) * 16 + col;
    const int tok = c / p.g;
    const int hq = hk * p.g + (c - tok * p.g);
    qvalid[cb] = c < p.ncols && token_valid(p, sq, tok);
    const int64_t qrow = sq.row0 + tok;
    const int32_t pos = (int32_t)(sq.L - sq.nq) + tok;
    klo[cb] = (int32_t)rg.begin;
    int32_t khi = (int32_t)rg.end - 1;
    if (p.window >= 0 && pos - (int32_t)p.window > klo[cb]) klo[cb] = pos - (int32_t)p.window;
    if (pos < khi) khi = pos;
    const uint32_t lo = qvalid[cb] ? ((uint32_t)klo[cb] ^ 0x80000000u) : 0u;
    const uint32_t hi = qvalid[cb] ? ~((uint32_t)khi ^ 0x80000000u) : 0u;
    const int32_t l1 = (int32_t)((uint32_t)__builtin_amdgcn_readfirstlane((int)group_max_u32<16>(lo)) ^ 0x80000000u);
    const int32_t h1 = (int32_t)(~(uint32_t)__builtin_amdgcn_readfirstlane((int)group_max_u32<16>(hi)) ^ 0x80000000u);
    wklo = l1 > wklo ? l1 : wklo;
    wkhi = h1 < wkhi ? h1 : wkhi;
    kspan[cb] = (uint32_t)(khi - klo[cb]);
    if (!qvalid[cb] || khi < klo[cb]) {  // no key: every tile position is out of range
      klo[cb] = INT32_MAX;
      kspan[cb] = 0;
    }
    mrun[cb] = -__builtin_inff();
    lpart[cb] = 0.0f;

    // Q operand: channels 32 m + 8 grp .. + 7; for codes scaled by a power of two into f16, with
    // a lo part when folded with per-channel key scales (see attn_mfma)
    float x[kQM][8];
    float qabs = 0.0f;
    const int64_t qe = i * p.q_sb + qrow * p.q_ss + (int64_t)hq * p.q_sh;
    const int64_t qse = i * p.qs_sb + qrow * p.qs_ss + (int64_t)hq * p.qs_sh;
#pragma unroll
    for (int m = 0; m < kQM; ++m) {
      const int d0 = 32 * m + 8 * grp;
      const bool in = qvalid[cb] && (kD % 32 == 0 || d0 < kD);
      if (p.q_vec) {
        u32x4 w = {0u, 0u, 0u, 0u};
        if (in) w = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.q) + qe + d0);
        if (p.q_dtype == TMO_DTYPE_BF16) unpack(BF16{}, w, x[m]);
        else unpack(F16{}, w, x[m]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[m][e] = in ? load_q(p, qe + d0 + e) : 0.0f;
          if (kQuant && p.qs_mode == 3 && in) x[m][e] *= q_group_scale(p, qse, d0 + e);
        }
      }
      if (kQuant && p.smode == 2) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (in) x[m][e] *= scale_at(p.ks, (int64_t)hk * kD + d0 + e, p.s_bf16);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) qabs = fmaxf(qabs, fabsf(x[m][e]));
    }
    // The column's factor is positive (maxima of the unscaled scores, and masked scores stay -inf
    // under it): its sign goes into q, and so does a factor of zero (a zero softmax scale, the
    // zero scale of an all-zero q row), whose product with -inf would be NaN
    const float q_rs = (kQuant && qvalid[cb] && p.qs_mode) ? q_row_scale(p, qse) : 1.0f;
    float sigma = 1.0f, inv_sigma = 1.0f;
    if constexpr (kQuant) {
      qabs = col_max(qabs);
      // a column's largest |q| in [2^(ex-1), 2^ex); no lower than 2^-100, so that sigma stays finite
      const int ex = qabs > 0.0f ? max(__builtin_amdgcn_frexp_expf(qabs), -100) : 1;
      sigma = __builtin_ldexpf(1.0f, 15 - ex);
      inv_sigma = __builtin_ldexpf(1.0f, ex - 15);
    }
    sscale[cb] = p.scale_log2 * inv_sigma * q_rs;
    if (sscale[cb] < 0.0f) {
      sscale[cb] = -sscale[cb];
      sigma = -sigma;
    }
    if (sscale[cb] == 0.0f) {
      sscale[cb] = 1.0f;
      sigma = 0.0f;
    }
#pragma unroll
    for (int m = 0; m < kQM; ++m)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float a = x[m][2 * k] * sigma, b = x[m][2 * k + 1] * sigma;
        if constexpr (kF16K) {
          const h2 h = {(_Float16)a, (_Float16)b};
          qhi[cb][m][k] = __builtin_bit_cast(uint32_t, h);
          if constexpr (kQLo) {
            const h2 l = {(_Float16)(a - (float)h[0]), (_Float16)(b - (float)h[1])};
            qlo[cb][m][k] = __builtin_bit_cast(uint32_t, l);
          }
        } else {
          qhi[cb][m][k] = (uint32_t)bf16_bits_rne(a) | ((uint32_t)bf16_bits_rne(b) << 16);
        }
      }
    // wait for the column's q here: left pending into the loop, the waits at the first uses there
    // would also wait for a tile's rows
#pragma unroll
    for (int m = 0; m < kQM; ++m) {
      asm volatile("" : "+v"(qhi[cb][m]));
      if constexpr (kQLo) asm volatile("" : "+v"(qlo[cb][m]));
    }
    asm volatile("" : "+v"(sscale[cb]));
  }

  f32x4 acc[kC][kVB];
#pragma unroll
  for (int cb = 0; cb < kC; ++cb)
#pragma unroll
    for (int b = 0; b < kVB; ++b) acc[cb][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // LDS offsets of the operand reads: K chunk 4 m + grp of row `col`; V rows 4 grp + col / 4,
  // 8-byte piece col & 3 of the 16-channel block
  constexpr int kKM = G::kX >> 2, kVM = G::kX >> 1;  // operand indices inside the XORed span
  const int ka = col * kPitch + ((grp ^ (col & G::kX)) << 4);
  const int vrow = 4 * grp + (col >> 2);
  const int va = vrow * kPitch + ((((col >> 1) & 1) ^ (vrow & G::kX)) << 4) + (col & 1) * 8;

  auto compute = [&](int buf, int32_t t0, uint32_t missing) {
    f32x4 s[kC][kTT];
    const char* kb = lds_k[buf];
    u32x4 ak[2][kQM];  // K operands of two 16-key tiles: the next one's reads go out first
    auto read_k = [&](int t, u32x4 (&a)[kQM]) {
#pragma unroll
      for (int m = 0; m < kQM; ++m)
        a[m] = *reinterpret_cast<const u32x4*>(kb + (ka ^ ((m & kKM) << 6)) + m / (kKM + 1) * (64 * (kKM + 1)) + t * 16 * kPitch);
    };
    read_k(0, ak[0]);
    f32x4 sc[kTT];  // the tile's key scales, then its value scales (tokens 16 t + 4 grp ..)
    auto read_scales = [&](const float* from) {
      if constexpr (kQuant) {
#pragma unroll
        for (int t = 0; t < kTT; ++t) sc[t] = *reinterpret_cast<const f32x4*>(&from[16 * t + 4 * grp]);
      }
    };
    read_scales(lds_ks[buf]);
#pragma unroll
    for (int t = 0; t < kTT; ++t) {
      if (t + 1 < kTT) read_k(t + 1, ak[(t + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the MFMAs
#pragma unroll
      for (int cb = 0; cb < kC; ++cb) s[cb][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int m = 0; m < kQM; ++m) {
#pragma unroll
        for (int cb = 0; cb < kC; ++cb) {
          s[cb][t] = mfma32<kF16K>(ak[t & 1][m], qhi[cb][m], s[cb][t]);
          if constexpr (kQLo) s[cb][t] = mfma32<kF16K>(ak[t & 1][m], qlo[cb][m], s[cb][t]);
        }
      }
    }
    if constexpr (kQuant) {
#pragma unroll
      for (int cb = 0; cb < kC; ++cb)
#pragma unroll
        for (int t = 0; t < kTT; ++t) s[cb][t] *= sc[t];
      read_scales(lds_vs[buf]);
    }
    u32x4 phi[kC][kTT / 2], plo[kC][kTT / 2];
    // wave-uniform: some key of the tile is outside some column's range, or has no page
    const bool edge = t0 < wklo || t0 + kT - 1 > wkhi || missing != 0;
#pragma unroll
    for (int cb = 0; cb < kC; ++cb) {
      __builtin_amdgcn_sched_barrier(0);  // one column block's softmax at a time: registers
      if (edge) {
        keep_branch();
#pragma unroll
        for (int t = 0; t < kTT; ++t) {
          // a missing page's keys: moved past every range
          const uint32_t far = missing >> t & 1 ? 0x80000000u : 0u;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t j = (uint32_t)(t0 + 16 * t + 4 * grp + e - klo[cb]) | far;
            s[cb][t][e] = j > kspan[cb] ? -__builtin_inff() : s[cb][t][e];
          }
        }
      }
      const float cs = sscale[cb];  // scores are in units of the column's factor
      float tmax = s[cb][0][0];
#pragma unroll
      for (int t = 0; t < kTT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) tmax = fmaxf(tmax, s[cb][t][e]);
      tmax = col_max_swap(tmax) * cs;
      // the lazily moved maximum of attn_mfma
      const bool was_empty = mrun[cb] == -__builtin_inff();
      const bool raise = tmax > mrun[cb] + kLazy || (was_empty && tmax != -__builtin_inff());
      const float mnew = raise ? tmax : mrun[cb];
      const float mref = mnew == -__builtin_inff() ? 0.0f : mnew;  // no key yet: every p is 0
      const float corr = raise ? __builtin_amdgcn_exp2f(mrun[cb] - mnew) : 1.0f;
      mrun[cb] = mnew;
      float psum = 0.0f;
#pragma unroll
      for (int t = 0; t < kTT; ++t) {
        float pe[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pe[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[cb][t][e], cs, -mref));
          psum += pe[e];
        }
        if constexpr (kQuant) {
#pragma unroll
          for (int e = 0; e < 4; ++e) pe[e] *= sc[t][e];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint32_t hi, lo;
          split2<kF16V>(pe[2 * h], pe[2 * h + 1], hi, lo);
          phi[cb][t >> 1][2 * (t & 1) + h] = hi;
          plo[cb][t >> 1][2 * (t & 1) + h] = lo;
        }
      }
      lpart[cb] = lpart[cb] * corr + psum;
      asm volatile("" : "+v"(lpart[cb]));  // here, not after the MFMAs with every p kept for it
      if (__ballot(corr != 1.0f && !was_empty)) {
#pragma unroll
        for (int b = 0; b < kVB; ++b) acc[cb][b] *= corr;
      }
    }
    const char* vb = lds_v[buf];
    // V operands of kBS channel blocks and 32 keys per step, the next step's read ahead.  The
    // step's MFMAs go round its kBS * kC accumulators, hi parts first, so none waits for the one
    // before it.
    constexpr int kBS = kVB % 2 ? 1 : 2, kSteps = kVB / kBS * (kTT / 2);
    u32x4 av[2][kBS];
    auto read_v = [&](int step, u32x4 (&a)[kBS]) {
      const int g = step % (kTT / 2), b0 = step / (kTT / 2) * kBS;
#pragma unroll
      for (int k = 0; k < kBS; ++k) {
        const int b = b0 + k;
        const char* vp = vb + (va ^ ((b & kVM) << 5)) + b / (kVM + 1) * (32 * (kVM + 1)) + g * 32 * kPitch;
        typedef __attribute__((address_space(3))) s16x4* lptr;
        const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lptr)vp);
        const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lptr)(vp + 16 * kPitch));
        a[k] = __builtin_bit_cast(u32x4, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    __builtin_amdgcn_sched_barrier(0);
    read_v(0, av[0]);
#pragma unroll
    for (int step = 0; step < kSteps; ++step) {
      if (step + 1 < kSteps) read_v(step + 1, av[(step + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const int g = step % (kTT / 2), b0 = step / (kTT / 2) * kBS;
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int k = 0; k < kBS; ++k)
#pragma unroll
          for (int cb = 0; cb < kC; ++cb)
            acc[cb][b0 + k] = mfma32<kF16V>(av[step & 1][k], part ? plo[cb][g] : phi[cb][g], acc[cb][b0 + k]);
    }
  };

  uint32_t cleared = 0;  // this wavefront cleared a value that is no number
  auto check = [&](int buf) {
    uint32_t none = 0;
    int first = tid;
    asm volatile("" : "+v"(first));  // addresses are made here: kept over the loop, they cost registers
    if constexpr (!kQuant || kKind == 3) {
#pragma unroll 1
      for (int u = first; u < kT * (kD / 8); u += 256) {
        const int r = u / (kD / 8), c = u - r * (kD / 8);
        u32x4* at = reinterpret_cast<u32x4*>(lds_v[buf] + r * kPitch + ((c ^ (r & G::kX)) << 4));
        u32x4 w = *at;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          uint32_t x = w[k];
          none |= clear_non_numbers<kF16V>(x);
          w[k] = x;
        }
        *at = w;
      }
    }
    if (kQuant && p.smode == 1 && first < kT && !(fabsf(lds_vs[buf][first]) < __builtin_inff())) {
      lds_vs[buf][first] = 0.0f;
      none = 1;
    }
    cleared |= __ballot(none != 0) ? 1u : 0u;
    __syncthreads();
  };

  // Tile n is computed from buffer n & 1 while tile n + 1 is in flight; it is then written to the
  // other buffer (free since the barrier that ended tile n - 1), tile n + 2's loads go out and a
  // barrier ends the step.
  if (tiles > 0) {
    stage(0);
    uint32_t missing = bad_next;
    issue(1);
    __syncthreads();
    for (int32_t n = 0; n < tiles; ++n) {
      if (n < rag_lo || n >= rag_hi) {
        keep_branch();
        check(n & 1);
      }
      compute(n & 1, kbeg + n * kT, missing);
      stage((n + 1) & 1);
      missing = bad_next;
      issue(n + 2);
      __syncthreads();
    }
  }

  // The cleared values reach the columns that see them
  if (rag_lo > 0 || rag_hi < tiles) {
    uint32_t* any = reinterpret_cast<uint32_t*>(&lds_k[0][0]);  // free since the last barrier
    if (lane == 0) any[wave] = cleared;
    __syncthreads();
    if (any[0] | any[1] | any[2] | any[3]) {
      for (int32_t j = kbeg; j < kend; ++j) {
        const int32_t tile = (j - kbeg) / kT;
        if (tile >= rag_lo && tile < rag_hi) continue;
        const int32_t pg = page_index(j), off = j - pg * p.BS, blk = bt_row[pg];
        if (blk < 0 || blk >= p.NB) continue;
        const int64_t row = ((int64_t)blk * p.Hkv + hk) * p.BS + off;
        const char* src = static_cast<const char*>(p.vc) + (kInt4 ? row >> 1 : row) * G::kVRow;
        const float scale = kQuant && p.smode == 1 ? scale_at(p.vs, blk * p.vs_sb + hk * p.vs_sh + off, p.s_bf16) : 1.0f;
#pragma unroll
        for (int b = 0; b < kVB; ++b) {
          const int d = 16 * b + 4 * grp;
          const u32x2 w = kQuant ? u32x2{*reinterpret_cast<const uint32_t*>(src + d), 0u}
                                 : *reinterpret_cast<const u32x2*>(src + 2 * d);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v;
            if constexpr (kKind == 1) v = bf16_value((uint16_t)(w[e >> 1] >> (16 * (e & 1))));
            else if constexpr (kKind == 2) v = f16_bits_to_f32(w[e >> 1] >> (16 * (e & 1)) & 0xffffu);
            else if constexpr (kKind == 3) v = fp8_value(w[0], e);
            else if constexpr (kInt4) v = (float)((int8_t)(w[0] >> (8 * e) << (j & 1 ? 4 : 0)) >> 4);
            else v = (float)(int8_t)(w[0] >> (8 * e));
            v *= scale;
            const bool number = fabsf(v) < __builtin_inff();
#pragma unroll
            for (int cb = 0; cb < kC; ++cb)
              if (!number && (uint32_t)(j - klo[cb]) <= kspan[cb]) acc[cb][b][e] += v;
          }
        }
      }
    }
  }

  // ---- output: lane (col, grp) holds channels 16 b + 4 grp + e of its columns
#pragma unroll
  for (int cb = 0; cb < kC; ++cb) {
    const float lsum = col_sum(lpart[cb]);
    if (!qvalid[cb]) continue;
    const int c = cbg * kCols + (wave * kC + cb) * 16 + col;
    const int tok = c / p.g;
    const int hq = hk * p.g + (c - tok * p.g);
    const int64_t qrow = sq.row0 + tok;
    float lse_v;
    const float inv = (direct ? finish(p, hq, mrun[cb], lsum, &lse_v) : (lsum > 0.0f ? 1.0f / lsum : 0.0f)) *
                      (kInt4 ? 0.0625f : 1.0f);
    float* ws_row = p.ws + ((((i * p.Hkv + hk) * p.splits + split) * p.ncols + c) * (int64_t)(kD + 2));
    const int64_t orow = i * p.o_sb + qrow * p.o_ss + (int64_t)hq * p.o_sh;
    if (!direct && grp == 0) {
      ws_row[0] = mrun[cb];
      ws_row[1] = lsum;
    }
#pragma unroll
    for (int b = 0; b < kVB; ++b) {
      const int d = 16 * b + 4 * grp;
      f32x4 o = acc[cb][b] * inv;
      if (kQuant && p.smode == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= scale_at(p.vs, (int64_t)hk * kD + d + e, p.s_bf16);
      }
      if (direct) {
        store_out4(p, orow + d, o);
      } else {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        f32x2* w = reinterpret_cast<f32x2*>(ws_row + 2 + d);  // rows are 8-byte aligned
        w[0] = f32x2{o[0], o[1]};
        w[1] = f32x2{o[2], o[3]};
      }
    }
    if (direct && grp == 0 && p.lse)
      p.lse[i * p.lse_sb + qrow * p.lse_ss + (int64_t)hq * p.lse_sh] = lse_v;
  }
}

template <int kD, int kKind, bool kQLo>
int launch_q(const AttnParams& p, hipStream_t st) {
  constexpr int kCols = 64 * Geo<kD, kKind, kQLo>::kC;
  const dim3 grid((unsigned)(p.Hkv * p.splits * ((p.ncols + kCols - 1) / kCols)), (unsigned)p.B);
  if constexpr (kD % 64 == 0) {
    if (p.few) return launch_kernel(attn_chunk<kD, kKind, kQLo, true>, grid, dim3(256), st, p);
  }
  return launch_kernel(attn_chunk<kD, kKind, kQLo, false>, grid, dim3(256), st, p);
}

template <int kD, int kKind>
int launch_d(const AttnParams& p, bool qlo, hipStream_t st) {
  if constexpr (chunk_quant(kKind)) {
    if (qlo) return launch_q<kD, kKind, true>(p, st);
  }
  return launch_q<kD, kKind, false>(p, st);
}

template <int kKind>
int launch(const AttnParams& p, bool qlo, hipStream_t st) {
  switch (p.D) {
    case 64: return launch_d<64, kKind>(p, qlo, st);
    case 80:
      if constexpr (kKind != 4) return launch_d<80, kKind>(p, qlo, st);
      return TMO_ERR_INVALID_ARGUMENT;
    case 96: return launch_d<96, kKind>(p, qlo, st);
    case 128: return launch_d<128, kKind>(p, qlo, st);
    default: return launch_d<256, kKind>(p, qlo, st);
  }
}

}  // namespace

int launch_attn_chunk(const AttnParams& p, bool qlo, hipStream_t st) {
  switch (p.c_dtype) {
    case TMO_DTYPE_I8: return launch<0>(p, qlo, st);
    case TMO_DTYPE_BF16: return launch<1>(p, false, st);
    case TMO_DTYPE_F16: return launch<2>(p, false, st);
    case TMO_DTYPE_F8E4M3: return launch<3>(p, qlo, st);
    default: return launch<4>(p, qlo, st);
  }
}

}  // namespace tmo
