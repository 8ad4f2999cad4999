// Shared by the attention kernels (decode_attn.hip, attn_mfma.h, attn_latent.hip, attn_chunk.hip):
// the launch parameters, the sequence and key-range rules, the softmax's last step, and the MFMA
// operand conversions.
#pragma once

#include "attn_rules.h"
#include "tmo_device.h"

namespace tmo {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazy = 8.0f;  // log2 headroom of the lazily moved softmax maximum
constexpr float kLn2 = 0.6931471805599453f;

// Query rows: token s of sequence i is at element i * q_sb + (row0_i + s) * q_ss + hq * q_sh,
// row0_i = cu[i] with cu_seq_q (q_sb 0 then) and 0 without; out and lse alike.
struct AttnParams {
  const void* q;
  int64_t q_sb, q_ss, q_sh;      // strides (elements); last dim contiguous
  const int32_t* cu;             // cu_seq_q [B + 1], or null: S tokens per sequence
  int32_t S;                     // tokens per sequence (at most, with cu)
  int32_t ncols;                 // S * g query columns per (sequence, KV head)
  int32_t ncb;                   // column blocks of 16
  int64_t total_q;               // q rows with cu: rows outside [0, total_q) are skipped
  const float* sink;             // [Hq] natural-log logits, or null
  const void* kc;
  const void* vc;                // caches [NB, Hkv, BS, k_row / v_row] contiguous
  int64_t k_row, v_row;          // cache row lengths (elements)
  const void* ks;                // scales: fp32, or bf16 when s_bf16
  const void* vs;
  int32_t s_bf16;
  int32_t smode;                 // 0 plain caches, 1 per token, 2 per channel, 3 per group
  int64_t ks_sb, ks_sh, vs_sb, vs_sh;  // per-token scale strides (page, head)
  const int32_t* bt;
  int64_t max_blocks;
  const int32_t* lens;
  const float* alibi;            // [B, Hq] or null
  int64_t window;                // < 0: unlimited
  float scale_log2;              // softmax_scale * log2(e)
  void* out;
  int64_t o_sb, o_ss, o_sh;
  float* lse;                    // null when not requested
  int64_t lse_sb, lse_ss, lse_sh;
  int32_t B, Hq, Hkv, g, D, Dv, BS;  // D: query / key head size, Dv: value head size
  int32_t bs_shift;              // log2(BS) when BS is a power of two, else -1
  int64_t NB;
  int32_t q_dtype;               // TMO_DTYPE_*: F32 / F16 / BF16, or I8 / F8E4M3 codes (qs)
  int32_t o_dtype;               // output TMO_DTYPE_* (q's for unquantised q)
  const void* qs;                // q scales of I8 / F8E4M3 q: fp32, or bf16 when qs_bf16
  int32_t qs_mode;               // 0 none, 1 per tensor, 2 per (token, head), 3 per channel group
  int32_t qs_bf16;
  int64_t qs_sb, qs_ss, qs_sh;   // q scale strides (sequence, token, head), as q's
  int32_t qs_group;              // mode 3: channels per scale (head_size / scale_num)
  int64_t bt_heads;              // block-table rows per sequence: 0 ([B, MB]), Hkv or Hq
  int32_t o_vec;                 // 2-byte output rows 8-byte aligned: vector stores
  int32_t q_vec;                 // q rows 16-byte aligned 2-byte values: vector q loads
  int32_t c_dtype;               // cache TMO_DTYPE_*
  int32_t v_ch;                  // int4 caches: V pairs channels (else the rows of a page)
  const void* mask;              // [B, S, mask_len] logit terms of the last keys, or null
  int32_t mask_dtype;            // F32 / F16 / BF16
  int32_t mask_len;
  int64_t m_sb, m_ss;            // mask strides (sequence, token); last dim contiguous
  int32_t splits;
  int32_t packed;                // 1-D grid, live workgroups first (work_of)
  int32_t lone;                  // a sequence's only live split writes the output itself
  int32_t few;                   // many columns: splits that leave a CU at most one workgroup, or 0: splits as announced
  int64_t split_tokens;          // multiple of 64 (latent caches: 32)
  float* ws;                     // [B, Hkv, splits, ncols, Dv + 2] when splits > 1
};

// ------------------------------------------------------------------------------ small helpers

// One load from each 64-byte line of the launch parameters, together: the compiler loads them block
// by block, and each first touch of a line is a round trip.
__device__ __forceinline__ void touch_params() {
  typedef const __attribute__((address_space(4))) uint32_t* Arg;
  const Arg a = (Arg)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int kLines = (sizeof(AttnParams) + 63) / 64;
  static_assert(kLines == 8, "one load per line");
  asm volatile("" ::"s"(a[0]), "s"(a[16]), "s"(a[32]), "s"(a[48]), "s"(a[64]), "s"(a[80]), "s"(a[96]), "s"(a[112]));
}

__device__ __forceinline__ uint16_t bf16_bits_rne(float x) {
  return __builtin_bit_cast(uint16_t, (__bf16)x);
}
__device__ __forceinline__ float bf16_value(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Query element e as stored: a float, or an int8 / float8_e4m3fn code (its scale applies
// separately: q_scale_of below).
__device__ __forceinline__ float load_q(const AttnParams& p, int64_t e) {
  switch (p.q_dtype) {
    case TMO_DTYPE_BF16: return load1(BF16{}, p.q, e);
    case TMO_DTYPE_F16: return load1(F16{}, p.q, e);
    case TMO_DTYPE_I8: return (float)static_cast<const int8_t*>(p.q)[e];
    case TMO_DTYPE_F8E4M3: return fp8_value(static_cast<const uint8_t*>(p.q)[e], 0);
    default: return load1(F32{}, p.q, e);
  }
}

// Scale of quantised q: the whole row's (per tensor, per token and head) -- `base` the row's
// scale element i * qs_sb + row * qs_ss + hq * qs_sh -- or, per channel group, channel d's.
__device__ __forceinline__ float q_row_scale(const AttnParams& p, int64_t base) {
  if (p.qs_mode == 1) return scale_at(p.qs, 0, p.qs_bf16);
  if (p.qs_mode == 2) return scale_at(p.qs, base, p.qs_bf16);
  return 1.0f;
}
__device__ __forceinline__ float q_group_scale(const AttnParams& p, int64_t base, int d) {
  return p.qs_mode == 3 ? scale_at(p.qs, base + d / p.qs_group, p.qs_bf16) : 1.0f;
}

// The block-table row of sequence i for query head hq (KV head hk): sparse-KV tables hold one
// per KV head or per query head.
__device__ __forceinline__ const int32_t* bt_row_of(const AttnParams& p, int64_t i, int hq, int hk) {
  const int64_t r = p.bt_heads == 0 ? i : i * p.bt_heads + (p.bt_heads == p.Hq ? hq : hk);
  return p.bt + r * p.max_blocks;
}

__device__ __forceinline__ void store_out(const AttnParams& p, int64_t e, float v) {
  switch (p.o_dtype) {
    case TMO_DTYPE_BF16: store1(BF16{}, p.out, e, v); break;
    case TMO_DTYPE_F16: store1(F16{}, p.out, e, v); break;
    default: store1(F32{}, p.out, e, v); break;
  }
}

// Mask element e (a logit term, natural-log units) as fp32.
__device__ __forceinline__ float mask_value(const AttnParams& p, int64_t e) {
  switch (p.mask_dtype) {
    case TMO_DTYPE_BF16: return load1(BF16{}, p.mask, e);
    case TMO_DTYPE_F16: return load1(F16{}, p.mask, e);
    default: return load1(F32{}, p.mask, e);
  }
}

// Sequence i: its keys L (clamped to its block table), its query tokens nq (the first
// min(nq, S) are computed) and the row of its token 0.
struct Seq {
  int64_t L, nq, row0;
};

__device__ __forceinline__ Seq seq_of(const AttnParams& p, int64_t i) {
  Seq q;
  int64_t L = p.lens[i];
  const int64_t cap = p.max_blocks * (int64_t)p.BS;
  if (L > cap) L = cap;
  if (L < 0) L = 0;
  q.L = L;
  if (p.cu) {
    q.row0 = p.cu[i];
    q.nq = (int64_t)p.cu[i + 1] - q.row0;
  } else {
    q.row0 = 0;
    q.nq = p.S;
  }
  return q;
}

// Lane l: the length of sequence l (batches of up to 64; 0 past them and in larger ones), in one load.
__device__ __forceinline__ int32_t lane_length(const AttnParams& p) {
  const int lane = threadIdx.x & (kWave - 1);
  return p.B <= kWave && lane < p.B ? p.lens[lane] : 0;
}

// The sequence of rank r by context length, longest first (batches of at most 64 sequences; r
// itself in larger ones, which even out by their number).  Workgroups are dispatched in order, so
// a long sequence that comes last would run on alone.  own: lane_length.
__device__ __forceinline__ int64_t seq_by_length(const AttnParams& p, int r, int32_t own) {
  if (p.B < 2 || p.B > kWave) return r;
  const int lane = threadIdx.x & (kWave - 1);
  int rank = 0;
  for (int j = 0; j < p.B; ++j) {
    const int32_t other = __builtin_amdgcn_readlane(own, j);
    rank += other > own || (other == own && j < lane) ? 1 : 0;
  }
  return __builtin_ctzll(__ballot(lane < p.B && rank == r));
}

// Token s of the sequence is computed: within S and nq, and (with cu_seq_q) a row of q.
__device__ __forceinline__ bool token_valid(const AttnParams& p, const Seq& q, int64_t s) {
  return s < p.S && s < q.nq && (!p.cu || (q.row0 + s >= 0 && q.row0 + s < p.total_q));
}

// Key range of the sequence (token 0's window start to L) and of split s within it.
struct Range {
  int64_t begin, end;
};

__device__ __forceinline__ Range token_range(const AttnParams& p, const Seq& q, int s, int64_t per) {
  Range r;
  const int64_t L = q.L;
  int64_t j0 = 0;
  if (p.window >= 0 && L - q.nq - p.window > 0) j0 = L - q.nq - p.window;
  r.begin = j0 + (int64_t)s * per;
  r.end = r.begin + per < L ? r.begin + per : L;
  if (s == p.splits - 1) r.end = L;  // the last split takes any tokens past max_context_len
  if (p.splits == 1) r.begin = j0;
  return r;
}
__device__ __forceinline__ Range token_range(const AttnParams& p, const Seq& q, int s) {
  return token_range(p, q, s, p.split_tokens);
}

// The many-column kernel's keys per split with p.few: as many as the split counts for the longest
// context present would give, where the announced maximum (split_tokens) gives more.  own:
// lane_length.
__device__ __forceinline__ int64_t fitted_split(const AttnParams& p, int32_t own) {
  uint32_t most = max(own, 0);
  if (p.B > kWave)
    for (int j = threadIdx.x & (kWave - 1); j < p.B; j += kWave) most = max(most, (uint32_t)max(p.lens[j], 0));
  const uint32_t longest = wave_max_u32_sgpr(most);
  uint32_t n = (longest + 255) / 256;
  if (n > 1) n -= 1 - (n & 1);
  n = max(n, min((longest + 127) / 128, (uint32_t)p.few));
  n = min(n, (uint32_t)p.splits);
  const uint32_t per = n <= 1 ? longest : (longest + n - 1) / n;
  const int64_t fit = ((int64_t)per + 63) / 64 * 64;
  return fit > 0 && fit < p.split_tokens ? fit : p.split_tokens;
}

// Splits of the sequence that hold keys, `per` each: a prefix of the launch's (the others write
// nothing).
__device__ __forceinline__ int live_splits(const AttnParams& p, const Seq& q, int64_t per) {
  if (p.splits <= 1 || per <= 0) return p.splits;
  const int64_t left = q.L - token_range(p, q, 0, per).begin;
  if (left <= 0) return 0;
  if (left <= per) return 1;
  const uint32_t n = ((uint32_t)left + (uint32_t)per - 1) / (uint32_t)per;  // per < left < 2^31
  return n < (uint32_t)p.splits ? (int)n : p.splits;
}

// A workgroup's work: split `split` of column-block group cb of KV head hk of sequence i.
struct Work {
  Seq sq;
  int64_t i;
  int hk, cb, split;
};

// The workgroup's work, or false when it has none.  On the 3-D grid (column block and split, KV
// head, sequence) the splits past a short sequence's keys leave at once, but the dispatcher has
// dealt the workgroups to the CUs by then: some get several live ones and others none.  The packed
// grid counts the live workgroups of every sequence (one wavefront scan over at most 64 lengths)
// and numbers them first, so the live ones are spread evenly.  Ragged contexts of 512 keys to the
// maximum, 3-D -> packed: 4 sequences to 8192 keys (32 / 8 heads x 128, int8) 31.8 -> 26.9 us,
// 32 to 4096 (bf16) 81.0 -> 77.3 us, 32 to 8192 on latent rows with 64 heads 108.6 -> 93.7 us;
// 64 sequences, whose workgroups run in many rounds, 467.3 -> 465.4 us.  kPacked is p.packed: a
// choice inside attn_mfma cost the calls of one split, a few hundred keys long, 0.2 to 0.4 us (4
// sequences of up to 250 int8 keys, head size 128: 13.2 us, 12.9 with an instance of each).
template <bool kPacked>
__device__ __forceinline__ bool work_of(const AttnParams& p, int ncb, Work& w) {
  if constexpr (!kPacked) {
    w.i = blockIdx.z;
    w.hk = blockIdx.y;
    w.cb = (int)(blockIdx.x / (unsigned)p.splits);
    w.split = (int)blockIdx.x - w.cb * p.splits;
    w.sq = seq_of(p, w.i);
    return true;
  }
  // lane s: sequence s (at most 64)
  const int lane = threadIdx.x & (kWave - 1);
  const Seq own = seq_of(p, lane < p.B ? lane : 0);
  const int64_t begin = token_range(p, own, 0).begin;
  uint32_t live = begin < own.L ? ((uint32_t)(own.L - begin) + (uint32_t)p.split_tokens - 1) /
                                      (uint32_t)p.split_tokens
                                : 0;
  if (live > (uint32_t)p.splits) live = p.splits;
  const uint32_t n = lane < p.B ? live * (uint32_t)(ncb * p.Hkv) : 0;
  const uint32_t incl = wave_incl_sum_u32(n);
  const uint64_t hit = __ballot(incl > blockIdx.x);
  if (!hit) return false;
  const int s = __builtin_ctzll(hit);
  const uint32_t rem = blockIdx.x - (uint32_t)__builtin_amdgcn_readlane((int)(incl - n), s);
  const uint32_t lv = (uint32_t)__builtin_amdgcn_readlane((int)live, s);
  const uint32_t unit = __builtin_amdgcn_readfirstlane(rem / lv);
  w.i = s;
  // Consecutive workgroups go round the 8 XCDs.  Where the live splits divide that round, the last
  // and shorter ones would all come to the same XCDs: every second four units count backwards (64
  // sequences of up to 1000 int8 keys, 4 tokens: 43.5 -> 40.3 us).
  const uint32_t nth = rem - unit * lv;
  w.split = (int)(unit & 4 ? lv - 1 - nth : nth);
  w.hk = (int)(__builtin_amdgcn_readfirstlane(unit / (uint32_t)ncb));
  w.cb = (int)(unit - (uint32_t)w.hk * (uint32_t)ncb);
  w.sq.L = __builtin_amdgcn_readlane((int)own.L, s);
  w.sq.row0 = __builtin_amdgcn_readlane((int)own.row0, s);
  w.sq.nq = p.S;
  if (p.cu) w.sq.nq = (int64_t)__builtin_amdgcn_readlane((int)(own.row0 + own.nq), s) - w.sq.row0;
  return true;
}

// Grid of the kernels that call work_of with ncb column-block groups.
inline dim3 attn_grid(const AttnParams& p, int ncb) {
  if (p.packed) return dim3((unsigned)((int64_t)p.splits * ncb * p.Hkv * p.B));
  return dim3((unsigned)(p.splits * ncb), (unsigned)p.Hkv, (unsigned)p.B);
}

// Final normalisation with the sink: m, l the column's maximum (base 2) and sum over its keys
// (l = 0: none).  Returns the factor of the unnormalised accumulators and writes the lse.
__device__ __forceinline__ float finish(const AttnParams& p, int hq, float m, float l, float* lse) {
  float inv = l > 0.0f ? 1.0f / l : 0.0f;
  float lg = l > 0.0f ? m + log2f(l) : -__builtin_inff();
  if (p.sink) {
    const float sk = p.sink[hq] * kLog2e;
    if (l > 0.0f) {
      const float mm = fmaxf(m, sk);
      const float lt = l * __builtin_amdgcn_exp2f(m - mm) + __builtin_amdgcn_exp2f(sk - mm);
      inv = __builtin_amdgcn_exp2f(m - mm) / lt;
      lg = mm + log2f(lt);
    } else {
      lg = sk;
    }
  }
  *lse = lg * kLn2;
  return inv;
}

// Max / sum over the four lane groups (lanes l, l ^ 16, l ^ 32, l ^ 48) of a column.
__device__ __forceinline__ float col_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, kWave));
  return fmaxf(v, __shfl_xor(v, 32, kWave));
}
__device__ __forceinline__ float col_sum(float v) {
  v += __shfl_xor(v, 16, kWave);
  return v + __shfl_xor(v, 32, kWave);
}

// The 16-bit values of dword w that are no number (all exponent bits set) cleared; nonzero where
// there was one.
template <bool kF16>
__device__ __forceinline__ uint32_t clear_non_numbers(uint32_t& w) {
  // the magnitude's carry into the sign's place
  const uint32_t hit = ((w & 0x7fff7fffu) + (kF16 ? 0x04000400u : 0x00800080u)) & 0x80008000u;
  w &= ~((hit >> 15) * 0xffffu);
  return hit;
}

// ------------------------------------------------------------------------------ MFMA kernel

template <bool kF16>
struct Mfma;
template <>
struct Mfma<false> {  // bf16 operands
  typedef bf16x4 V4;
  static __device__ __forceinline__ f32x4 run(V4 a, V4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ short bits(float x) { return (short)bf16_bits_rne(x); }
  static __device__ __forceinline__ float value(short b) { return bf16_value((uint16_t)b); }
};
template <>
struct Mfma<true> {  // f16 operands
  typedef f16x4 V4;
  static __device__ __forceinline__ f32x4 run(V4 a, V4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// D = A B + C over 32 channels, bf16 or f16 operands.
template <bool kF16>
__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (kF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a),
                                                 __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// Four int8 codes (one dword) -> four f16 operands holding 1152 + code exactly: with
// u = code + 128 (the byte with its top bit flipped), the f16 pattern 0x6400 | u is 1024 + u
// (ulp 1 in [1024, 2048)), so two byte permutes build the four values.  The QK product then
// carries 1152 * sum(q), which is subtracted per query column.
constexpr float kCodeBias = 1152.0f;
__device__ __forceinline__ f16x4 codes_f16(uint32_t w) {
  const uint32_t u = w ^ 0x80808080u;
  u32x2 h;
  h[0] = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);  // [u0, 0x64, u1, 0x64]
  h[1] = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);  // [u2, 0x64, u3, 0x64]
  return __builtin_bit_cast(f16x4, h);
}

// Four float8_e4m3fn codes (one dword) -> four f16 operands holding their values exactly:
// v_cvt_pk_f32_fp8 decodes two codes to fp32, v_cvt_pkrtz_f16_f32 packs two fp32 into f16
// (every e4m3fn value -- at most 4 significant bits, 2^-9 .. 448 -- is an f16 value, so the
// conversion's rounding never acts).
__device__ __forceinline__ f16x4 fp8_f16(uint32_t w) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
  const f2 b = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
  u32x2 h;
  h[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a[0], a[1]));
  h[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(b[0], b[1]));
  return __builtin_bit_cast(f16x4, h);
}

// Eight int4 codes (one dword of a K row: byte b holds channels 2b (high nibble) and 2b + 1
// (low nibble)) -> the f16 operands of channels 4h + {0, 2, 1, 3}, h = `half` (bytes 2h and
// 2h + 1), as 2 + u / 8 with u = code + 8 (the nibble with its top bit flipped): the f16
// pattern 0x4000 | u << 6 has exponent 1 and u in the top four mantissa bits, so the value
// 3 + code / 8 is exact.  Each f16 pair is one byte permute (the two high or two low nibbles
// into the pair's low bytes) and one shift-or.  The QK product then carries 3 * sum(q) and a
// factor 1/8; the channel order within the operand is matched by q's.
__device__ __forceinline__ f16x4 int4_f16(uint32_t w, int half) {
  const uint32_t x = w ^ 0x88888888u;
  const uint32_t hi = x & 0xf0f0f0f0u, lo = x & 0x0f0f0f0fu;
  const uint32_t sel = half ? 0x0c030c02u : 0x0c010c00u;  // [byte 2h, 0, byte 2h + 1, 0]
  u32x2 h;
  h[0] = (__builtin_amdgcn_perm(hi, hi, sel) << 2) | 0x40004000u;  // channels 4h, 4h + 2
  h[1] = (__builtin_amdgcn_perm(lo, lo, sel) << 6) | 0x40004000u;  // channels 4h + 1, 4h + 3
  return __builtin_bit_cast(f16x4, h);
}
constexpr float kInt4Bias = 3.0f;
// Channel of operand element e of QK MFMA m within the lane's run: int4 operands hold
// channels 4m + {0, 2, 1, 3}
__host__ __device__ constexpr int qk_channel(bool int4, int m, int e) {
  return 4 * m + (int4 ? (((e & 1) << 1) | (e >> 1)) : e);
}

// Two fp32 values as a packed 16-bit pair of the operand type, and the remainders as another.
template <bool kF16>
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  if constexpr (kF16) {
    const _Float16 ha = (_Float16)a, hb = (_Float16)b;
    const _Float16 la = (_Float16)(a - (float)ha), lb = (_Float16)(b - (float)hb);
    hi = (uint32_t)__builtin_bit_cast(uint16_t, ha) | ((uint32_t)__builtin_bit_cast(uint16_t, hb) << 16);
    lo = (uint32_t)__builtin_bit_cast(uint16_t, la) | ((uint32_t)__builtin_bit_cast(uint16_t, lb) << 16);
  } else {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 v = {a, b};
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2));
    const f2 r = {a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u)};
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf2));
  }
}

// Output elements e .. e + 3 (one 8-byte store where the rows allow it).
__device__ __forceinline__ void store_out4(const AttnParams& p, int64_t e, f32x4 v) {
  if (p.o_vec) {
    u32x2 w;
    if (p.o_dtype == TMO_DTYPE_BF16) {
      w[0] = pack2(BF16{}, v[0], v[1]);
      w[1] = pack2(BF16{}, v[2], v[3]);
    } else {
      w[0] = pack2(F16{}, v[0], v[1]);
      w[1] = pack2(F16{}, v[2], v[3]);
    }
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.out) + e) = w;
    return;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) store_out(p, e + k, v[k]);
}

// The MFMA kernel over each kind of cache (attn_mfma_*.hip): p.splits partials per column when > 1;
// qlo: q needs a lo operand.
int launch_attn_int8(const AttnParams& p, bool qlo, hipStream_t st);
int launch_attn_fp8(const AttnParams& p, bool qlo, hipStream_t st);
int launch_attn_int4(const AttnParams& p, bool qlo, hipStream_t st);
int launch_attn_plain(const AttnParams& p, hipStream_t st);
// The latent-cache kernel (attn_latent.hip): p.splits partials per column when > 1, as
// attn_mfma leaves them.
int launch_attn_latent(const AttnParams& p, hipStream_t st);
// The many-column kernel (attn_chunk.hip), likewise; qlo: q needs a lo operand.
int launch_attn_chunk(const AttnParams& p, bool qlo, hipStream_t st);

}  // namespace tmo
