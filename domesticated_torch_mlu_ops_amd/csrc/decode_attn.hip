// single_query_cached_kv_attn for gfx950: the query tokens of each sequence against its paged
// KV cache (reference _ops.py:777-900; header include/torch_mlu_ops.h:107-130).
//
//   s_j = softmax_scale * q . k_j (+ alibi_slope * (j - P)),
//   out = sum_j e^(s_j) v_j / (sum_j e^(s_j) (+ e^sink)),  lse = log of that denominator,
//
// for query token s of a sequence with nq tokens and L keys at position P = L - nq + s (one
// token: P = L - 1), over keys j in [max(0, P - window_left), P]; key j at row j % BS of page
// block_tables[i, j / BS] (pages outside [0, NB) are masked): k_j its first D channels, v_j
// the first Dv of the V cache's row, or of the K row when both live in one cache; query head
// hq reads KV head hq / (Hq / Hkv).  Caches are int8 codes, float8_e4m3fn values or int4 pairs
// (K pairing channels, V pairing the rows of a page or channels) with fp32 or bf16 scales (k =
// code * scale) per token [NB, Hkv, BS] (strided in the first two dims), per channel [Hkv, D],
// or per group (K [NB, Hkv, BS, D / 32], V [NB, Hkv, BS / 32, Dv]), or of q's dtype.  A mask
// adds its terms to the logits of each sequence's last mask_len keys.
//
// MFMA kernels: attn_mfma.h (K and V head sizes and cache rows all 64 / 128 / 256, block_size a
// multiple of 16, per-token or per-channel scales), attn_latent.hip (K rows of 576 channels whose
// first 512 are the value row) and attn_chunk.hip (many query columns per KV head, head sizes 80
// and 96).  With more than one split per (sequence, KV head) their partials (max, sum, normalised
// row) go to a caller-provided workspace and attn_combine merges them.  A generic kernel (one
// wavefront per (query token, query head), VALU) serves every other shape, dtype and scale layout.
#include "attn_common.h"

namespace tmo {
namespace {

// Merge the splits of one (query token, query head): one wavefront per row (kWhole) or per row and
// 64 channels (blockIdx.y).  Lane s holds split s's (max, sum) and turns them into the split's weight sum_s *
// 2^(max_s - max), once; the output channels then read each split's row once, weighted through a
// lane broadcast.
template <int kBatch, bool kWhole>
__global__ __launch_bounds__(256) void attn_combine(AttnParams p) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;  // (i * S + s) * Hq + hq
  if (row >= (int64_t)p.B * p.S * p.Hq) return;
  int d = kWhole ? lane : blockIdx.y * kWave + lane;
  int dc = d < p.Dv ? d : p.Dv - 1;
  const int64_t it = row / p.Hq;
  const int hq = (int)(row - it * p.Hq);
  const int64_t i = it / p.S;
  const int tok = (int)(it - i * p.S);
  const Seq sq = seq_of(p, i);
  if (!token_valid(p, sq, tok)) return;
  const int hk = hq / p.g;
  const int c = tok * p.g + (hq - hk * p.g);
  const int64_t stride = (int64_t)p.ncols * (p.Dv + 2);
  const float* base = p.ws + ((i * p.Hkv + hk) * p.splits * (int64_t)p.ncols + c) * (p.Dv + 2);
  // splits past the sequence's keys wrote nothing (the main kernel returned early)
  const int live = live_splits(p, sq, p.few ? fitted_split(p, lane_length(p)) : p.split_tokens);
  if (p.lone && live == 1) return;
  // Every load is unconditional (split and channel indices clamped into this column's rows of
  // the workspace; an empty split's row is read and given weight 0), so the loads of a batch
  // issue together.  Under the per-split weight test each row load waited for the previous
  // one: up to 2 x live round trips per wavefront.
  const int last = live > 0 ? live - 1 : 0;
  const int64_t qrow = sq.row0 + tok;
  const int64_t orow = i * p.o_sb + qrow * p.o_ss + (int64_t)hq * p.o_sh;
  if (live <= kWave) {  // wave-uniform; every launch of the torch op (at most 63 splits)
    // lane s holds split s's (max, sum), loaded once; the values in batches of kBatch splits.
    // The first two batches' values do not wait for the weights, or for each other: a row's time
    // is its chain of round trips.  32 latent sequences of 512..8192 rows (up to 21 splits): 46.7
    // -> 45.9 us a call, 8 bf16 ones of 128..4096 keys 33.6 -> 33.4, with 89 registers for 32.
    const int sc = lane < live ? lane : last;
    const float m_raw = base[sc * stride], l_raw = base[sc * stride + 1];
    float v[kBatch], v2[kBatch];
    auto load = [&](int k0, float (&x)[kBatch]) {
#pragma unroll
      for (int k = 0; k < kBatch; ++k) x[k] = base[(k0 + k < live ? k0 + k : last) * stride + 2 + dc];
    };
    load(0, v);
    if (live > kBatch) load(kBatch, v2);
    const float m = lane < live ? m_raw : -__builtin_inff();
    float mx = m;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    const float wgt = m != -__builtin_inff() ? l_raw * __builtin_amdgcn_exp2f(m - mx) : 0.0f;
    float lt = wgt;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) lt += __shfl_xor(lt, o, kWave);
    float lse_v;
    const float inv = finish(p, hq, mx, lt, &lse_v);
    auto add = [&](int k0, const float (&x)[kBatch], float& o) {
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const float wk = __shfl(wgt, k0 + k < live ? k0 + k : 0, kWave);
        if (k0 + k < live && wk != 0.0f) o += x[k] * wk;
      }
    };
    for (;;) {
      float o = 0.0f;
      add(0, v, o);
      if (live > kBatch) add(kBatch, v2, o);
      for (int k0 = 2 * kBatch; k0 < live; k0 += kBatch) {
        load(k0, v);
        add(k0, v, o);
      }
      if (d < p.Dv) store_out(p, orow + d, o * inv);
      if (d == 0 && p.lse) p.lse[i * p.lse_sb + qrow * p.lse_ss + (int64_t)hq * p.lse_sh] = lse_v;
      if (!kWhole) return;
      d += kWave;
      if (d - lane >= p.Dv) return;
      dc = d < p.Dv ? d : p.Dv - 1;
      load(0, v);
      if (live > kBatch) load(kBatch, v2);
    }
  }
  float mx = -__builtin_inff();
  for (int s0 = 0; s0 < live; s0 += kWave) {
    const int s = s0 + lane;
    const float m = base[(s < live ? s : last) * stride];
    mx = fmaxf(mx, s < live ? m : -__builtin_inff());
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
  float lt = 0.0f;
  for (int s0 = 0; s0 < live; s0 += kWave) {
    const int s = s0 + lane;
    const int sc = s < live ? s : last;
    const float m = s < live ? base[sc * stride] : -__builtin_inff();
    const float l = base[sc * stride + 1];
    lt += m != -__builtin_inff() ? l * __builtin_amdgcn_exp2f(m - mx) : 0.0f;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) lt += __shfl_xor(lt, o, kWave);
  float lse_v;
  const float inv = finish(p, hq, mx, lt, &lse_v);
  float o = 0.0f;
  for (int s0 = 0; s0 < live; s0 += kWave) {
    const int sl = s0 + lane;
    const int sc = sl < live ? sl : last;
    const float m = sl < live ? base[sc * stride] : -__builtin_inff();
    const float wgt = m != -__builtin_inff() ? base[sc * stride + 1] * __builtin_amdgcn_exp2f(m - mx) : 0.0f;
    const int n = live - s0 < kWave ? live - s0 : kWave;
    for (int k0 = 0; k0 < n; k0 += kBatch) {
      float v[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const int s = s0 + (k0 + k < n ? k0 + k : n - 1);
        v[k] = base[s * stride + 2 + dc];
      }
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const float wk = __shfl(wgt, k0 + k < n ? k0 + k : 0, kWave);
        if (k0 + k < n && wk != 0.0f) o += v[k] * wk;
      }
    }
  }
  if (d < p.Dv) store_out(p, orow + d, o * inv);
  if (d == 0 && p.lse) p.lse[i * p.lse_sb + qrow * p.lse_ss + (int64_t)hq * p.lse_sh] = lse_v;
}

// ------------------------------------------------------------------------------ generic kernel

__device__ __forceinline__ float plain_value(const void* base, int64_t e, int cache_dtype) {
  switch (cache_dtype) {
    case TMO_DTYPE_BF16: return load1(BF16{}, base, e);
    case TMO_DTYPE_F16: return load1(F16{}, base, e);
    default: return load1(F32{}, base, e);
  }
}

// Code e of a quantised cache as fp32: an int8 code, or a float8_e4m3fn value.
__device__ __forceinline__ float code_value(const void* base, int64_t e, int cache_dtype) {
  if (cache_dtype == TMO_DTYPE_I8) return (float)static_cast<const int8_t*>(base)[e];
  return fp8_value(static_cast<const uint8_t*>(base)[e], 0);
}

// Signed 4-bit code `odd` of byte e of an int4-pair cache: the even element of a pair in the
// high nibble, the odd one in the low nibble, sign-extended.
__device__ __forceinline__ float nibble_value(const void* base, int64_t e, int odd) {
  const int32_t b = static_cast<const int8_t*>(base)[e];
  return (float)(odd ? (int32_t)((uint32_t)b << 28) >> 28 : b >> 4);
}

__device__ __forceinline__ bool quant_cache(int cache_dtype) {
  return cache_dtype == TMO_DTYPE_I8 || cache_dtype == TMO_DTYPE_F8E4M3 ||
         cache_dtype == TMO_DTYPE_I4;
}

// Key channel d of row `row` of page blk, KV head hk.
__device__ __forceinline__ float key_value(const AttnParams& p, int64_t blk, int hk, int64_t row,
                                           int d, int cache_dtype) {
  const int64_t r = (blk * p.Hkv + hk) * p.BS + row;
  if (!quant_cache(cache_dtype)) return plain_value(p.kc, r * p.k_row + d, cache_dtype);
  // int4: K pairs adjacent channels, k_row bytes per row
  const float code = cache_dtype == TMO_DTYPE_I4 ? nibble_value(p.kc, r * p.k_row + (d >> 1), d & 1)
                                                 : code_value(p.kc, r * p.k_row + d, cache_dtype);
  switch (p.smode) {
    case 1: return code * scale_at(p.ks, blk * p.ks_sb + hk * p.ks_sh + row, p.s_bf16);
    case 2: return code * scale_at(p.ks, (int64_t)hk * p.D + d, p.s_bf16);
    default: return code * scale_at(p.ks, r * (p.D >> 5) + (d >> 5), p.s_bf16);
  }
}

// Value channel d: per-group V scales hold one number per 32 rows of a page and channel.
__device__ __forceinline__ float value_value(const AttnParams& p, int64_t blk, int hk, int64_t row,
                                             int d, int cache_dtype) {
  const int64_t r = (blk * p.Hkv + hk) * p.BS + row;
  if (!quant_cache(cache_dtype)) return plain_value(p.vc, r * p.v_row + d, cache_dtype);
  float code;
  if (cache_dtype != TMO_DTYPE_I4)
    code = code_value(p.vc, r * p.v_row + d, cache_dtype);
  else if (p.v_ch)  // int4, V pairing channels: as K
    code = nibble_value(p.vc, r * p.v_row + (d >> 1), d & 1);
  else  // int4, V pairing the rows of a page: [NB, Hkv, BS / 2, v_row]
    code = nibble_value(p.vc, ((blk * p.Hkv + hk) * (p.BS >> 1) + (row >> 1)) * p.v_row + d,
                        (int)(row & 1));
  switch (p.smode) {
    case 1: return code * scale_at(p.vs, blk * p.vs_sb + hk * p.vs_sh + row, p.s_bf16);
    case 2: return code * scale_at(p.vs, (int64_t)hk * p.Dv + d, p.s_bf16);
    default:
      return code * scale_at(p.vs, ((blk * p.Hkv + hk) * (p.BS >> 5) + (row >> 5)) * p.Dv + d,
                             p.s_bf16);
  }
}

// One wavefront per (query token, query head): 64 keys at a time, one per lane (a lane
// computes its key's full dot product), then every lane accumulates its channels over the 64
// keys.  Value head sizes up to 512 (8 accumulators per lane); any key head size.
__global__ __launch_bounds__(256) void attn_generic(AttnParams p) {
  const int cache_dtype = p.c_dtype;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;  // (i * S + s) * Hq + hq
  if (row >= (int64_t)p.B * p.S * p.Hq) return;
  const int64_t it = row / p.Hq;
  const int hq = (int)(row - it * p.Hq);
  const int64_t i = it / p.S;
  const int64_t tok = it - i * p.S;
  const Seq sq = seq_of(p, i);
  if (!token_valid(p, sq, tok)) return;
  const int hk = hq / p.g;
  // keys [jb, je) of the token at position P
  const int64_t P = sq.L - sq.nq + tok;
  const int64_t je = P + 1 < sq.L ? P + 1 : sq.L;
  const int64_t jb = p.window >= 0 && P - p.window > 0 ? P - p.window : 0;
  const float alibi = p.alibi ? p.alibi[i * p.Hq + hq] * kLog2e : 0.0f;
  float mrun = -__builtin_inff(), l = 0.0f;
  float acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = 0.0f;
  const int64_t qrow = sq.row0 + tok;
  const int64_t qe = i * p.q_sb + qrow * p.q_ss + (int64_t)hq * p.q_sh;
  const int64_t qse = i * p.qs_sb + qrow * p.qs_ss + (int64_t)hq * p.qs_sh;  // quantised q
  const float q_rs = p.qs_mode ? q_row_scale(p, qse) : 1.0f;
  const int32_t* btr = bt_row_of(p, i, hq, hk);
  for (int64_t j0 = jb; j0 < je; j0 += kWave) {
    const int64_t j = j0 + lane;
    float s = -__builtin_inff();
    int blk = -1, r = 0;
    if (j < je) {
      blk = btr[j / p.BS];
      r = (int)(j % p.BS);
      if (blk >= 0 && blk < p.NB) {
        float dot = 0.0f;
        for (int d = 0; d < p.D; ++d)
          dot += load_q(p, qe + d) * q_group_scale(p, qse, d) *
                 key_value(p, blk, hk, r, d, cache_dtype);
        s = dot * q_rs * p.scale_log2;
        if (p.alibi) s += alibi * (float)(j - P);
        if (p.mask && j >= sq.L - p.mask_len)
          s += mask_value(p, i * p.m_sb + tok * p.m_ss + (j - (sq.L - p.mask_len))) * kLog2e;
      } else {
        blk = -1;
      }
    }
    float tmax = s;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) tmax = fmaxf(tmax, __shfl_xor(tmax, o, kWave));
    const float mnew = fmaxf(mrun, tmax);
    if (mnew == -__builtin_inff()) continue;
    const float corr = __builtin_amdgcn_exp2f(mrun - mnew);
    mrun = mnew;
    const float pj = __builtin_amdgcn_exp2f(s - mnew);
    float ps = pj;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) ps += __shfl_xor(ps, o, kWave);
    l = l * corr + ps;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] *= corr;
    for (int t = 0; t < kWave; ++t) {
      const float pt = __shfl(pj, t, kWave);
      const int bt_ = __shfl(blk, t, kWave);
      const int rt = __shfl(r, t, kWave);
      if (pt == 0.0f || bt_ < 0) continue;  // the same in every lane
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int d = lane + u * kWave;
        if (d < p.Dv) acc[u] += pt * value_value(p, bt_, hk, rt, d, cache_dtype);
      }
    }
  }
  float lse_v;
  const float inv = finish(p, hq, mrun, l, &lse_v);
  const int64_t orow = i * p.o_sb + qrow * p.o_ss + (int64_t)hq * p.o_sh;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int d = lane + u * kWave;
    if (d < p.Dv) store_out(p, orow + d, p.sink ? acc[u] * inv : (l > 0.0f ? acc[u] / l : 0.0f));
  }
  if (lane == 0 && p.lse) p.lse[i * p.lse_sb + qrow * p.lse_ss + (int64_t)hq * p.lse_sh] = lse_v;
}

// ------------------------------------------------------------------------------ launch

// A row is one wavefront's where the rows alone give each CU 16 wavefronts: 5120 rows of 128
// channels, 3 splits: 7.9 us shared by two, 7.1 alone; 3200 rows, 7 splits, a call of attention
// 77.0 and 78.5 us.
template <int kBatch>
int launch_combine(const AttnParams& p, hipStream_t st) {
  const int64_t rows = (int64_t)p.B * p.S * p.Hq;
  const unsigned blocks = (unsigned)((rows + 3) / 4), chunks = (unsigned)((p.Dv + kWave - 1) / kWave);
  if (rows >= (chunks > 1 ? 4096 : 16384) && p.splits <= kWave)
    return launch_kernel(attn_combine<4, true>, dim3(blocks), dim3(256), st, p);
  return launch_kernel(attn_combine<kBatch, false>, dim3(blocks, chunks), dim3(256), st, p);
}

// Short batches for few splits: a batch issues all its loads, whatever the splits (100 sequences of
// up to 1000 int8 keys, 8 KV heads, 3 splits: a call 50.5 us in batches of 16, 47.5 in 4).
int launch_combine(const AttnParams& p, hipStream_t st) {
  return p.splits <= 4 ? launch_combine<4>(p, st) : p.splits <= 8 ? launch_combine<8>(p, st) : launch_combine<16>(p, st);
}

}  // namespace
}  // namespace tmo

using namespace tmo;

extern "C" int64_t tmo_hip_cached_kv_attn_workspace_bytes(int64_t batch, int64_t num_kv_heads,
                                                          int64_t num_q_heads,
                                                          int64_t head_size_v, int64_t seq_q,
                                                          int64_t splits) {
  if (batch <= 0 || num_kv_heads <= 0 || num_q_heads <= 0 || head_size_v <= 0 || seq_q <= 0 ||
      splits <= 1)
    return 0;
  return batch * num_kv_heads * splits * seq_q * (num_q_heads / num_kv_heads) *
         (head_size_v + 2) * (int64_t)sizeof(float);
}

extern "C" int64_t tmo_hip_attn_workspace_bytes(int64_t batch, int64_t num_kv_heads,
                                                int64_t num_q_heads, int64_t head_size,
                                                int64_t max_context_len, int64_t splits) {
  (void)max_context_len;
  return tmo_hip_cached_kv_attn_workspace_bytes(batch, num_kv_heads, num_q_heads, head_size, 1,
                                                splits);
}

extern "C" int tmo_hip_cached_kv_attn(
    const void* q, int64_t q_stride_batch, int64_t q_stride_token, int64_t q_stride_head,
    const void* q_scale, int q_scale_mode, int q_scale_dtype, int64_t q_scale_stride_batch,
    int64_t q_scale_stride_token, int64_t q_scale_stride_head, int64_t q_scale_groups,
    const int32_t* cu_seq_q, int64_t seq_q, int64_t total_q, const void* k_cache,
    const void* v_cache, int64_t k_cache_dim, int64_t v_cache_dim, const void* k_scale,
    const void* v_scale, int scale_mode, int scale_dtype, int64_t k_scale_stride_block,
    int64_t k_scale_stride_head, int64_t v_scale_stride_block, int64_t v_scale_stride_head,
    const int32_t* block_tables, int64_t max_blocks, int64_t block_table_heads,
    const int32_t* context_lens, const float* alibi_slopes, const float* sink, const void* mask,
    int mask_dtype,
    int64_t mask_len, int64_t mask_stride_batch, int64_t mask_stride_token, void* out,
    int64_t out_stride_batch, int64_t out_stride_token, int64_t out_stride_head, float* lse,
    int64_t lse_stride_batch, int64_t lse_stride_token, int64_t lse_stride_head, int64_t batch,
    int64_t num_q_heads, int64_t num_kv_heads, int64_t head_size, int64_t head_size_v,
    int64_t num_blocks, int64_t block_size, int64_t max_context_len, int64_t window_left,
    float softmax_scale, int q_dtype, int cache_dtype, int v_pair_channels, int out_dtype,
    int64_t splits, void* workspace, int64_t workspace_bytes, void* stream) {
  // q: floats (the output of q's dtype), or int8 / float8_e4m3fn codes with q_scale (the
  // output of out_dtype) over quantised caches
  const bool qquant = q_dtype == TMO_DTYPE_I8 || q_dtype == TMO_DTYPE_F8E4M3;
  if (q_dtype != TMO_DTYPE_BF16 && q_dtype != TMO_DTYPE_F16 && q_dtype != TMO_DTYPE_F32 && !qquant)
    return TMO_ERR_UNSUPPORTED_DTYPE;
  if (out_dtype != TMO_DTYPE_BF16 && out_dtype != TMO_DTYPE_F16 && out_dtype != TMO_DTYPE_F32)
    return TMO_ERR_UNSUPPORTED_DTYPE;
  if (!qquant && out_dtype != q_dtype) return TMO_ERR_UNSUPPORTED_DTYPE;
  if (qquant) {
    if (q_scale_mode < 1 || q_scale_mode > 3) return TMO_ERR_UNSUPPORTED_MODE;
    if (q_scale_dtype != TMO_DTYPE_F32 && q_scale_dtype != TMO_DTYPE_BF16)
      return TMO_ERR_UNSUPPORTED_DTYPE;
    if (!q_scale || q_scale_stride_batch < 0 || q_scale_stride_token < 0 ||
        q_scale_stride_head < 0 ||
        (q_scale_mode == 3 && (q_scale_groups <= 0 || head_size % q_scale_groups != 0)))
      return TMO_ERR_INVALID_ARGUMENT;
  }
  if (block_table_heads != 0 && block_table_heads != num_kv_heads &&
      block_table_heads != num_q_heads)
    return TMO_ERR_INVALID_ARGUMENT;
  // quantised caches: int8 codes, float8_e4m3fn values or int4 pairs, times fp32 or bf16 scales
  const bool int4 = cache_dtype == TMO_DTYPE_I4;
  const bool quant = cache_dtype == TMO_DTYPE_I8 || cache_dtype == TMO_DTYPE_F8E4M3 || int4;
  if (!quant && cache_dtype != q_dtype) return TMO_ERR_UNSUPPORTED_DTYPE;  // quantised q: quantised caches
  if (mask && mask_dtype != TMO_DTYPE_F32 && mask_dtype != TMO_DTYPE_F16 &&
      mask_dtype != TMO_DTYPE_BF16)
    return TMO_ERR_UNSUPPORTED_DTYPE;
  if (mask && (mask_len <= 0 || mask_len > 0x7fffffffLL || mask_stride_batch < 0 ||
               mask_stride_token < 0))
    return TMO_ERR_INVALID_ARGUMENT;
  if (quant && scale_dtype != TMO_DTYPE_F32 && scale_dtype != TMO_DTYPE_BF16)
    return TMO_ERR_UNSUPPORTED_DTYPE;
  if (quant && (scale_mode < 1 || scale_mode > 3)) return TMO_ERR_UNSUPPORTED_MODE;
  // An empty cache (num_blocks 0: every block-table entry is outside it, so every key is
  // masked) may come with null cache and per-token scale pointers; nothing reads them.
  // Likewise an empty block table (max_blocks 0 caps every context at 0 keys).
  if (!q || !context_lens || !out) return TMO_ERR_INVALID_ARGUMENT;
  if ((num_blocks > 0 && !k_cache) || (max_blocks > 0 && !block_tables))
    return TMO_ERR_INVALID_ARGUMENT;
  if (quant && (!k_scale || !v_scale) && (num_blocks > 0 || scale_mode != 1))
    return TMO_ERR_INVALID_ARGUMENT;
  // v_cache null: the values are the first head_size_v channels of the K cache's rows (not
  // for int4 pairs, whose K and V caches pair different axes: null only with an empty cache)
  const bool v_null = !v_cache;
  if (!v_cache) {
    if (int4 && num_blocks > 0) return TMO_ERR_INVALID_ARGUMENT;
    v_cache = k_cache;
    v_cache_dim = k_cache_dim;
  }
  // max_context_len <= 0: "an uncertain maximum value of context_lens" (reference _ops.py,
  // single_query_cached_kv_attn's max_context_len); it only sizes the splits, so a negative
  // value is taken as 0 (the last split always runs to the sequence's own length)
  if (max_context_len < 0) max_context_len = 0;
  if (batch < 0 || num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads != 0 ||
      head_size <= 0 || head_size > 4096 || head_size_v <= 0 || head_size_v > 512 ||
      num_blocks < 0 ||
      block_size <= 0 || max_blocks < 0 || splits < 1 || seq_q < 0 || q_stride_batch < 0 ||
      q_stride_token < 0 || q_stride_head < 0 || out_stride_batch < 0 || out_stride_token < 0 ||
      out_stride_head < 0 || (cu_seq_q && total_q < 0))
    return TMO_ERR_INVALID_ARGUMENT;
  if (quant && scale_mode == 1 &&
      (k_scale_stride_block < 0 || k_scale_stride_head < 0 || v_scale_stride_block < 0 ||
       v_scale_stride_head < 0))
    return TMO_ERR_INVALID_ARGUMENT;
  if (quant && scale_mode == 3 && (head_size % 32 != 0 || block_size % 32 != 0))
    return TMO_ERR_INVALID_ARGUMENT;
  // cache rows: elements, or bytes of int4 pairs (K: head_size / 2 channel pairs; V: pairs of
  // rows -- [num_blocks, Hkv, block_size / 2, v_cache_dim], block_size even -- or of channels)
  if (!int4 ? (k_cache_dim < head_size || v_cache_dim < head_size_v)
            : (2 * k_cache_dim < head_size ||
               (!v_null && (v_pair_channels ? 2 * v_cache_dim < head_size_v
                                            : (v_cache_dim < head_size_v || block_size % 2 != 0)))))
    return TMO_ERR_INVALID_ARGUMENT;
  const int64_t g = num_q_heads / num_kv_heads;
  if (batch > 65535 || num_kv_heads > 65535 || splits > 65535 || num_q_heads > 0x7fffffffLL ||
      seq_q > 0x7fffffffLL / num_q_heads)
    return TMO_ERR_INVALID_ARGUMENT;
  const int64_t ncb = (seq_q * g + 15) / 16;
  if (splits * ncb > 0x7fffffffLL || (batch * seq_q * num_q_heads + 3) / 4 > 0x7fffffffLL)
    return TMO_ERR_INVALID_ARGUMENT;
  if (splits > 1 && (!workspace ||
                     workspace_bytes < tmo_hip_cached_kv_attn_workspace_bytes(
                                           batch, num_kv_heads, num_q_heads, head_size_v, seq_q,
                                           splits)))
    return TMO_ERR_INVALID_ARGUMENT;
  if (batch == 0 || seq_q == 0) return TMO_OK;

  AttnParams p{};
  p.q = q;
  p.q_sb = cu_seq_q ? 0 : q_stride_batch;
  p.q_ss = q_stride_token;
  p.q_sh = q_stride_head;
  p.cu = cu_seq_q;
  p.S = (int32_t)seq_q;
  p.ncols = (int32_t)(seq_q * g);
  p.ncb = (int32_t)ncb;
  p.total_q = cu_seq_q ? total_q : batch * seq_q;
  p.sink = sink;
  p.kc = k_cache;
  p.vc = v_cache;
  p.k_row = k_cache_dim;
  p.v_row = v_cache_dim;
  p.ks = k_scale;
  p.vs = v_scale;
  p.smode = quant ? scale_mode : 0;
  p.s_bf16 = quant && scale_dtype == TMO_DTYPE_BF16;
  p.ks_sb = k_scale_stride_block;
  p.ks_sh = k_scale_stride_head;
  p.vs_sb = v_scale_stride_block;
  p.vs_sh = v_scale_stride_head;
  p.bt = block_tables;
  p.max_blocks = max_blocks;
  p.lens = context_lens;
  p.alibi = alibi_slopes;
  p.window = window_left < 0x7fffffffLL ? window_left : -1;  // positions are 32-bit
  p.scale_log2 = softmax_scale * kLog2e;
  p.out = out;
  p.o_sb = cu_seq_q ? 0 : out_stride_batch;
  p.o_ss = out_stride_token;
  p.o_sh = out_stride_head;
  p.lse = lse;
  p.lse_sb = cu_seq_q ? 0 : lse_stride_batch;
  p.lse_ss = lse_stride_token;
  p.lse_sh = lse_stride_head;
  p.B = (int32_t)batch;
  p.Hq = (int32_t)num_q_heads;
  p.Hkv = (int32_t)num_kv_heads;
  p.g = (int32_t)g;
  p.D = (int32_t)head_size;
  p.Dv = (int32_t)head_size_v;
  p.BS = (int32_t)block_size;
  p.bs_shift = ilog2_if_pow2(block_size);
  p.NB = num_blocks;
  p.q_dtype = q_dtype;
  p.o_dtype = out_dtype;
  p.qs = qquant ? q_scale : nullptr;
  p.qs_mode = qquant ? q_scale_mode : 0;
  p.qs_bf16 = qquant && q_scale_dtype == TMO_DTYPE_BF16;
  p.qs_sb = cu_seq_q ? 0 : q_scale_stride_batch;
  p.qs_ss = q_scale_stride_token;
  p.qs_sh = q_scale_stride_head;
  p.qs_group = qquant && q_scale_mode == 3 ? (int32_t)(head_size / q_scale_groups) : 1;
  p.bt_heads = block_table_heads;
  p.q_vec = (q_dtype == TMO_DTYPE_BF16 || q_dtype == TMO_DTYPE_F16) &&
            reinterpret_cast<uintptr_t>(q) % 16 == 0 &&
            p.q_sb % 8 == 0 && q_stride_token % 8 == 0 && q_stride_head % 8 == 0 &&
            (!quant || scale_mode != 2 || reinterpret_cast<uintptr_t>(k_scale) % 16 == 0);
  p.o_vec = out_dtype != TMO_DTYPE_F32 && reinterpret_cast<uintptr_t>(out) % 8 == 0 &&
            p.o_sb % 4 == 0 && out_stride_token % 4 == 0 && out_stride_head % 4 == 0;
  p.ws = static_cast<float*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);

  // MFMA path eligibility: one head size for K and V that is also both caches' row length,
  // page rows in whole 16-token tiles, 16-byte aligned rows and scale vectors (per-token scale
  // offsets of a page and head in multiples of four), q's dtype representable by the operands
  // (quantised caches: f16 with a lo part when needed), per-token or per-channel scales.
  auto al = [](const void* x, int a) { return reinterpret_cast<uintptr_t>(x) % a == 0; };
  // The MFMA kernel always issues its tile loads (a wave with no valid page yet reads page 0,
  // see attn_mfma), so an empty cache takes attn_generic, whose loads are all under the page
  // check: every output row is then 0 and its lse -inf (nothing to attend to).
  // int4 pages: K rows of head_size / 2 bytes, V pairing rows (pair rows of head_size bytes)
  const bool whole = head_size == 64 || head_size == 128 || head_size == 256;
  const bool part = (head_size == 80 && !int4) || head_size == 96;  // attn_chunk only
  bool mfma = num_blocks > 0 && (whole || part) && head_size_v == head_size &&
              k_cache_dim == (int4 ? head_size / 2 : head_size) && v_cache_dim == head_size &&
              !(int4 && v_pair_channels) && block_size % 16 == 0 && al(k_cache, 16) &&
              al(v_cache, 16) && q_dtype != TMO_DTYPE_F32 &&
              (block_table_heads != num_q_heads || num_q_heads == num_kv_heads);
  if (quant)
    mfma = mfma && scale_mode != 3 &&
           (scale_mode != 1 ||
            (al(k_scale, p.s_bf16 ? 8 : 16) && al(v_scale, p.s_bf16 ? 8 : 16) &&
             k_scale_stride_block % 4 == 0 &&
             k_scale_stride_head % 4 == 0 && v_scale_stride_block % 4 == 0 &&
             v_scale_stride_head % 4 == 0));
  p.c_dtype = cache_dtype;
  p.v_ch = int4 && v_pair_channels;
  p.mask = mask;
  p.mask_dtype = mask_dtype;
  p.mask_len = (int32_t)mask_len;
  p.m_sb = mask_stride_batch;
  p.m_ss = mask_stride_token;
  // Latent caches: values and keys in one cache of 576 channels, 512 of them values
  const bool latent = !quant && v_null && num_blocks > 0 && head_size == 576 &&
                      head_size_v == 512 && k_cache_dim == 576 && block_size % 8 == 0 && p.q_vec &&
                      al(k_cache, 16) &&
                      (block_table_heads != num_q_heads || num_q_heads == num_kv_heads);
  // Many query columns (attn_many_columns) and head sizes 80 and 96 take attn_chunk, but for fp32
  // outputs of the latter, where the VALU kernel's fp32 probabilities show: 16 sequences of
  // 512..8192 int8 keys, 32 heads x 96, one token each, 12486 us there, 104 here.
  // It indexes cache rows and scales with 32 bits and has no mask or ALiBi terms.
  auto scale_span = [&](int64_t sb, int64_t sh) {
    return num_blocks * sb + num_kv_heads * sh + block_size;
  };
  const bool chunk = mfma && (whole || out_dtype != TMO_DTYPE_F32) && !mask && !alibi_slopes &&
                     attn_many_columns(quant, int4, head_size, p.ncols, num_kv_heads, batch,
                                       max_context_len, max_blocks * block_size, splits) &&
                     num_kv_heads * splits * ((p.ncols + 63) / 64) <= 0x7fffffffLL &&
                     num_blocks * num_kv_heads * block_size <= 0x7fffffffLL &&
                     (!quant || scale_mode != 1 ||
                      (scale_span(k_scale_stride_block, k_scale_stride_head) <= 0x7fffffffLL &&
                       scale_span(v_scale_stride_block, v_scale_stride_head) <= 0x7fffffffLL));
  if (!(mfma && whole) && !chunk && !latent) {
    p.splits = 1;
    p.split_tokens = 1;
    const int64_t rows = batch * seq_q * num_q_heads;
    return launch_kernel(attn_generic, dim3((unsigned)((rows + 3) / 4)), dim3(256), st, p);
  }
  p.splits = (int32_t)splits;
  // tokens per split: the context divided evenly, rounded up to whole 64-token steps (four
  // wavefronts x 16-token tiles)
  int64_t per = (max_context_len + splits - 1) / splits;
  per = latent ? (per + 31) / 32 * 32 : (per + 63) / 64 * 64;
  p.split_tokens = per > 0 ? per : 64;
  // Packed numbering for up to 64 sequences, one lane each; one sequence has nothing to even out
  p.packed = p.splits > 1 && batch > 1 && batch <= kWave && p.split_tokens < (1LL << 31) &&
             (int64_t)p.splits * p.ncb * num_kv_heads * batch < (1LL << 24);
  if (latent) {
    const int rc = launch_attn_latent(p, st);
    return rc != TMO_OK || p.splits == 1 ? rc : launch_combine(p, st);
  }
  // quantised caches: bf16 and f16 q, and int8 / float8_e4m3fn q codes, are exact f16 operands
  // after the power-of-two scaling; q folded with per-channel key scales or group-wise q
  // scales needs the lo operand
  const bool qlo = scale_mode == 2 || p.qs_mode == 3;
  if (chunk) {
    p.lone = 1;
    p.packed = 0;
    // Splits as long as the contexts present need where the announced ones could make the call
    // slower than on attn_mfma: whole head sizes with fewer than 128 workgroups per split (256 for
    // codes of 64).  64 columns of 8 sequences of 2048 int8 keys, head size
    // 128, announced as 32768: 76 us on attn_mfma, 88 with the announced splits, 46 with fitted ones.
    if (whole && p.splits > 1) {
      p.few = (int32_t)(255 / (batch * num_kv_heads * ((p.ncols + 127) / 128)));
      if (p.few == 1 && !(quant && head_size == 64)) p.few = 0;
    }
    const int rc = launch_attn_chunk(p, qlo, st);
    return rc != TMO_OK || p.splits == 1 ? rc : launch_combine(p, st);
  }
  const int rc = cache_dtype == TMO_DTYPE_I8 ? launch_attn_int8(p, qlo, st)
                 : cache_dtype == TMO_DTYPE_F8E4M3 ? launch_attn_fp8(p, qlo, st)
                 : int4 ? launch_attn_int4(p, qlo, st) : launch_attn_plain(p, st);
  return rc != TMO_OK || p.splits == 1 ? rc : launch_combine(p, st);
}

extern "C" int tmo_hip_single_query_cached_kv_attn(
    const void* q, int64_t q_stride_seq, int64_t q_stride_head, const void* k_cache,
    const void* v_cache, const float* k_scale, const float* v_scale, int scale_mode,
    const int32_t* block_tables, int64_t max_blocks, const int32_t* context_lens,
    const float* alibi_slopes, void* out, int64_t out_stride_seq, int64_t out_stride_head,
    float* lse, int64_t lse_stride_seq, int64_t lse_stride_head, int64_t batch,
    int64_t num_q_heads, int64_t num_kv_heads, int64_t head_size, int64_t num_blocks,
    int64_t block_size, int64_t max_context_len, int64_t window_left, float softmax_scale,
    int q_dtype, int cache_dtype, int64_t splits, void* workspace, int64_t workspace_bytes,
    void* stream) {
  if ((cache_dtype == TMO_DTYPE_I8 || cache_dtype == TMO_DTYPE_F8E4M3) && scale_mode == 3)
    return TMO_ERR_UNSUPPORTED_MODE;
  if (!v_cache && num_blocks > 0) return TMO_ERR_INVALID_ARGUMENT;
  if (head_size > 512) return TMO_ERR_INVALID_ARGUMENT;
  // contiguous per-token scales [num_blocks, Hkv, block_size]
  const int64_t sb = num_kv_heads * block_size, sh = block_size;
  if (cache_dtype == TMO_DTYPE_I4) return TMO_ERR_UNSUPPORTED_DTYPE;
  if (q_dtype == TMO_DTYPE_I8 || q_dtype == TMO_DTYPE_F8E4M3) return TMO_ERR_UNSUPPORTED_DTYPE;
  return tmo_hip_cached_kv_attn(
      q, q_stride_seq, 0, q_stride_head, nullptr, 0, TMO_DTYPE_F32, 0, 0, 0, 0, nullptr, 1, 0,
      k_cache, v_cache, head_size, head_size, k_scale, v_scale, scale_mode, TMO_DTYPE_F32, sb,
      sh, sb, sh, block_tables, max_blocks, 0, context_lens, alibi_slopes, nullptr, nullptr, 0,
      0, 0, 0, out, out_stride_seq, 0, out_stride_head, lse, lse_stride_seq, 0,
      lse_stride_head, batch, num_q_heads, num_kv_heads, head_size, head_size, num_blocks,
      block_size, max_context_len, window_left, softmax_scale, q_dtype, cache_dtype, 0, q_dtype,
      splits, workspace, workspace_bytes, stream);
}
