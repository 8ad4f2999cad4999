// Attention over a latent cache: one cache whose rows of 576 bf16 / f16 channels are the keys and
// whose first 512 channels are the values (single_query_cached_kv_attn with v_cache None,
// reference _ops.py:828-831), for gfx950.
//
// What bounds it: each row is read once from HBM and used by every query head of its KV head, so
// with 16..64 query columns the arithmetic (34..136 flops per byte) hides behind the stream.  The
// kernel's job is to keep the stream deep and to touch each byte once on its way from HBM:
//   * A workgroup owns one (sequence, KV head, split) and 16 * kCB query columns.  Its 4 * kCB
//     wavefronts load tiles of 32 * kCB rows straight into one of two LDS buffers
//     (global_load_lds_dwordx4) while the other is computed, and both products read the tile
//     from there.  Staged through registers instead, one tile ahead took 36 of them per lane (48
//     against 45 us below) and two ahead spilled.
//   * LDS rows are stored as they are, the 16-byte chunk index XORed with the row's low three
//     bits: the 16 rows of a K operand read (ds_read_b128) and the four rows of a V operand
//     read then fall on different banks although the row pitch is a multiple of 128 bytes.
//   * S^T = K Q^T with v_mfma_f32_16x16x32, Q in registers.  The four wavefronts of a column
//     block share the product: one 16-row tile and (with 32-row tiles) one half of the channels
//     each, the results exchanged through LDS; the softmax of the whole tile is then every
//     wavefront's own.  (Every wavefront computing all of S^T needs no exchange and one barrier
//     less, but reads the tile four times from LDS.)
//   * O^T = V^T P^T: each wavefront owns a quarter of the 512 value channels (32 accumulator
//     registers).  ds_read_b64_tr_b16 transposes V on the way out of LDS.  S^T's result layout
//     (lane group c holds tokens 4c .. 4c + 3) is P^T's operand layout for tiles 2g and 2g + 1
//     side by side; V^T takes the same token order.
//   * p enters as hi + lo operands of 16 significant bits, as in attn_mfma.
// 32 sequences of 512..8192 rows, 16 heads, bf16 (157 MB): 34.3 ms on the VALU kernel that served
// this form before, 45 us here (3.5 TB/s), of which 7.5 are the merging of the splits.  One
// workgroup alone takes 1.33 us per 32-row tile; two per CU cover each other's latencies, and
// what is left is their uneven share of ragged contexts.
#include "attn_common.h"

namespace tmo {
namespace {

constexpr int kLatD = 576;                // key channels = row length
constexpr int kLatDv = 512;               // value channels
constexpr int kLatRow = kLatD * 2;        // bytes
constexpr int kLatQK = kLatD / 32;        // MFMAs per 16-token tile
constexpr int kLatVB = kLatDv / 16 / 4;   // 16-channel value blocks per wavefront

__device__ __align__(16) const uint32_t kLatZeros[4] = {};

// 16 bytes per lane from global memory into LDS at byte m0 + 16 * lane of the workgroup's
// allocation.  The caller waits for them (vmcnt) before the barrier that publishes them.  Not
// the builtin: the compiler cannot tell the buffer being filled from the one being read and waits
// for the loads before every LDS read, which ends the overlap.  There is no output register;
// waits that the compiler counts for its own loads only come out longer.  One wait state lies
// between the write of m0 and its use by an LDS load.
__device__ __forceinline__ void load_lds16(const char* base, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(__builtin_amdgcn_readfirstlane((int)dst)), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void load_lds16(const char* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(__builtin_amdgcn_readfirstlane((int)dst)), "v"(src) : "memory", "m0");
}

template <bool kF16, int kCB, bool kMask>
__global__ __launch_bounds__(256 * kCB, 2) void attn_latent(AttnParams p) {
  constexpr int kT = 32 * kCB;        // tokens per LDS tile
  constexpr int kST = 2 * kCB;        // 16-token score tiles per LDS tile
  constexpr int kSplitM = kCB == 1 ? 2 : 1;  // wavefronts that share a score tile's channels
  constexpr int kQM = kLatQK / kSplitM;      // MFMAs of a wavefront's score tile
  constexpr int kLoads = 8 * kLatRow / (kWave * 16);  // 16-byte loads per lane and tile
  __shared__ __align__(128) char lds[2][kT * kLatRow];
  __shared__ __align__(16) float lds_bias[2][kT];  // 0, or -inf for a row that holds no key
  __shared__ f32x4 lds_s[4 * kCB][kWave];          // each wavefront's score tile

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane & 15, grp = lane >> 4;
  const int chq = wave & 3;           // quarter of the value channels, and:
  const int st_tile = chq % kST, st_half = chq / kST;  // score tile, part of its channels
  Work wk;
  if (p.packed) {
    if (!work_of<true>(p, (p.ncb + kCB - 1) / kCB, wk)) return;
  } else {
    work_of<false>(p, (p.ncb + kCB - 1) / kCB, wk);
  }
  const int64_t i = wk.i;
  const int hk = wk.hk, split = wk.split;
  const int cbg = wk.cb;  // group of kCB column blocks
  const Seq sq = wk.sq;
  const Range rg = token_range(p, sq, split);
  if (p.splits > 1 && rg.begin >= rg.end) return;  // an empty split writes no partial
  const int c = (cbg * kCB + (wave >> 2)) * 16 + col;
  const int tok = c / p.g;
  const int hq = hk * p.g + (c - tok * p.g);
  const bool qvalid = c < p.ncols && token_valid(p, sq, tok);
  const int64_t qrow = sq.row0 + tok;

  // keys of this lane's column: [klo, khi] (empty for padding)
  const int32_t pos = (int32_t)(sq.L - sq.nq) + tok;
  int32_t klo = (int32_t)rg.begin, khi = (int32_t)rg.end - 1;
  if (p.window >= 0 && pos - (int32_t)p.window > klo) klo = pos - (int32_t)p.window;
  if (pos < khi) khi = pos;
  if (!qvalid) khi = klo - 1;
  // [wklo, wkhi]: keys inside every valid column's range (no per-key test there)
  int32_t wklo, wkhi;
  {
    const uint32_t lo = qvalid ? ((uint32_t)klo ^ 0x80000000u) : 0u;
    const uint32_t hi = qvalid ? ~((uint32_t)khi ^ 0x80000000u) : 0u;
    wklo = (int32_t)((uint32_t)__builtin_amdgcn_readfirstlane((int)group_max_u32<16>(lo)) ^
                     0x80000000u);
    wkhi = (int32_t)(~(uint32_t)__builtin_amdgcn_readfirstlane((int)group_max_u32<16>(hi)) ^
                     0x80000000u);
  }
  // the workgroup's keys: from its first token's window start to its last token's position
  int64_t bbeg = rg.begin, bend = rg.end;
  {
    const int64_t ntok = sq.nq < p.S ? sq.nq : p.S;
    const int64_t s_first = (int64_t)cbg * (16 * kCB) / p.g;
    int64_t s_last = ((int64_t)cbg * (16 * kCB) + 16 * kCB - 1) / p.g;
    if (s_last > ntok - 1) s_last = ntok - 1;
    const int64_t p_first = sq.L - sq.nq + s_first, p_last = sq.L - sq.nq + s_last;
    if (p.window >= 0 && p_first - p.window > bbeg) bbeg = p_first - p.window;
    if (p_last + 1 < bend) bend = p_last + 1;
    if (s_last < s_first || bend <= bbeg) bbeg = bend = 0;
  }
  // tiles start on a 16-row boundary of the sequence (the rows before bbeg are masked): the
  // eight rows that a wavefront loads lie in one page
  const int32_t kbeg = (int32_t)bbeg & ~15, kend = (int32_t)bend;
  // ---- staging: wavefront w brings rows 8 w .. + 7 of each tile straight into LDS
  // (global_load_lds: no registers, LDS written in lane order).  Load j of lane l fills the
  // 16-byte slot 64 j + l of the group's 72 x 8: row (64 j + l) / 72, whose slot s holds chunk
  // s ^ row.
  const int32_t* bt_row = p.bt + (p.bt_heads ? i * p.bt_heads + hk : i) * p.max_blocks;
  auto page_index = [&](int32_t t) -> int32_t { return p.bs_shift >= 0 ? t >> p.bs_shift : t / p.BS; };
  const uint32_t lds_base =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)&lds[0][0];
  uint32_t src_off[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int slot = 64 * j + lane, row = slot / 72;
    src_off[j] = row * kLatRow + (((slot - row * 72) ^ row) << 4);
  }
  // Lane l holds the block of the wavefront's rows in tile win + l (64 tiles per refill)
  int32_t win = 0, lane_blk = -1;
  auto refill = [&]() {
    const int32_t t = kbeg + (win + lane) * kT + 8 * wave;
    lane_blk = t < kend ? bt_row[page_index(t)] : -1;
  };
  auto load_tile = [&](int32_t tile, int buf) {
    if (tile >= win + kWave) {
      win += kWave;
      refill();
    }
    const int32_t blk = __builtin_amdgcn_readlane(lane_blk, tile - win);
    const int32_t t = kbeg + tile * kT + 8 * wave;  // the group's first row
    const bool ok = t < kend && blk >= 0 && blk < p.NB;
    const int64_t row = ((int64_t)blk * p.Hkv + hk) * p.BS + (t - page_index(t) * p.BS);
    const char* src = static_cast<const char*>(p.kc) + row * kLatRow;
    const uint32_t dst = lds_base + (uint32_t)((buf * kT + wave * 8) * kLatRow);
    if (ok && t + 8 <= kend) {
#pragma unroll
      for (int j = 0; j < kLoads; ++j) load_lds16(src, src_off[j], dst + j * 1024);
    } else {
      // rows that hold no key (past the range, or on a missing page) are zeros
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int r = (64 * j + lane) / 72;
        load_lds16(ok && t + r < kend ? src + src_off[j] : reinterpret_cast<const char*>(kLatZeros),
                   dst + j * 1024);
      }
    }
    if (lane < 8) lds_bias[buf][8 * wave + lane] = ok && t + lane < kend ? 0.0f : -__builtin_inff();
  };
  const int32_t tiles = (kend - kbeg + kT - 1) / kT;
  if (tiles > 0) {
    refill();
    load_tile(0, 0);
  }
  // ---- Q operand: channels 32 m + 8 grp .. + 7 of column `col`, this wavefront's m
  u32x4 qf[kQM];
  {
    const u32x4* qp = reinterpret_cast<const u32x4*>(
        static_cast<const uint16_t*>(p.q) + i * p.q_sb + qrow * p.q_ss + (int64_t)hq * p.q_sh + grp * 8);
#pragma unroll
    for (int m = 0; m < kQM; ++m)
      qf[m] = qvalid ? qp[4 * (st_half * kQM + m)] : u32x4{0u, 0u, 0u, 0u};
  }
  // wait for Q here, once: left pending into the loop, the wait at its first use there would
  // also wait for a tile's rows
#pragma unroll
  for (int m = 0; m < kQM; ++m) asm volatile("" : "+v"(qf[m]));
  const float alibi = (p.alibi && qvalid) ? p.alibi[i * p.Hq + hq] * kLog2e : 0.0f;
  const int32_t mask_lo = (int32_t)sq.L - p.mask_len;

  float mrun = -__builtin_inff(), lpart = 0.0f;
  f32x4 acc[kLatVB];
#pragma unroll
  for (int b = 0; b < kLatVB; ++b) acc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // LDS offsets of the operand reads (see the swizzle above)
  // K: channel chunk 4 m + grp of row `col` of the wavefront's score tile
  int ka[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    ka[par] = (st_tile * 16 + col) * kLatRow + ((((4 * (st_half * kQM + par)) + grp) ^ (col & 7)) << 4);
  const int vrow = 4 * grp + (col >> 2);
  const int va = vrow * kLatRow + ((((col >> 1) & 1) ^ (vrow & 7)) << 4) + (col & 1) * 8 + chq * 256;

  auto compute = [&](int buf, int32_t t0) {
    const char* base = lds[buf];
    {
      f32x4 x[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
      for (int m = 0; m < kQM; ++m) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(base + ka[m & 1] + (m >> 1) * 128);
        x[m & 1] = mfma32<kF16>(a, qf[m], x[m & 1]);
      }
      lds_s[wave][lane] = x[0] + x[1];
    }
    __syncthreads();
    f32x4 s[kST];
#pragma unroll
    for (int t = 0; t < kST; ++t) {
      s[t] = lds_s[(wave & ~3) + t][lane];
      if constexpr (kSplitM == 2) s[t] += lds_s[(wave & ~3) + kST + t][lane];
    }
    // V operands of the first half of the wavefront's channel blocks: read ahead of the softmax
    u32x4 vf[kLatVB / 2][kCB];
    auto read_v = [&](int b0) {
#pragma unroll
      for (int b = 0; b < kLatVB / 2; ++b)
#pragma unroll
        for (int g = 0; g < kCB; ++g) {
          const char* vp = base + (va ^ (b << 5)) + (b0 >> 2) * 128 + g * 32 * kLatRow;
          typedef __attribute__((address_space(3))) s16x4* lptr;
          const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lptr)vp);
          const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lptr)(vp + 16 * kLatRow));
          vf[b][g] = __builtin_bit_cast(u32x4, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };
    read_v(0);
    // the largest magnitude of the scores, NaN where one is: two scores per v_maximum3_f32
    float odd = 0.0f;
#pragma unroll
    for (int t = 0; t < kST; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) odd = __builtin_elementwise_maximum(odd, __builtin_fabsf(s[t][e]));
    float tmax = -__builtin_inff();
#pragma unroll
    for (int t = 0; t < kST; ++t) {
      const f32x4 bias = *reinterpret_cast<const f32x4*>(&lds_bias[buf][16 * t + 4 * grp]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[t][e] = s[t][e] * p.scale_log2 + bias[e];
    }
    if (p.alibi) {
      keep_branch();
#pragma unroll
      for (int t = 0; t < kST; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t][e] += alibi * (float)(t0 + 16 * t + 4 * grp + e - pos);
    }
    if (t0 < wklo || t0 + kT - 1 > wkhi) {
      keep_branch();
#pragma unroll
      for (int t = 0; t < kST; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int32_t j = t0 + 16 * t + 4 * grp + e;
          if (j < klo || j > khi) s[t][e] = -__builtin_inff();
        }
    }
    if (kMask && t0 + kT - 1 >= mask_lo) {
      const int ct = c / p.g;
      const int64_t mask_row = i * p.m_sb + (int64_t)(ct < p.S ? ct : p.S - 1) * p.m_ss;
#pragma unroll
      for (int t = 0; t < kST; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int32_t j = t0 + 16 * t + 4 * grp + e;
          // a key that the column does not see stays so, whatever its term
          if (j >= mask_lo && j < (int32_t)sq.L && s[t][e] != -__builtin_inff())
            s[t][e] += mask_value(p, mask_row + (j - mask_lo)) * kLog2e;
        }
    }
#pragma unroll
    for (int t = 0; t < kST; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) tmax = fmaxf(tmax, s[t][e]);
    tmax = col_max(tmax);
    // the lazily moved maximum of attn_mfma
    const bool was_empty = mrun == -__builtin_inff();
    const bool raise = tmax > mrun + kLazy || (was_empty && tmax != -__builtin_inff());
    const float mnew = raise ? tmax : mrun;
    const bool live = mnew != -__builtin_inff();
    const float corr = raise ? __builtin_amdgcn_exp2f(mrun - mnew) : 1.0f;
    mrun = mnew;
    float psum = 0.0f;
    u32x4 phi[kCB], plo[kCB];
#pragma unroll
    for (int t = 0; t < kST; ++t) {
      float pe[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pe[e] = live ? __builtin_amdgcn_exp2f(s[t][e] - mnew) : 0.0f;
        psum += pe[e];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t hi, lo;
        split2<kF16>(pe[2 * h], pe[2 * h + 1], hi, lo);
        phi[t >> 1][2 * (t & 1) + h] = hi;
        plo[t >> 1][2 * (t & 1) + h] = lo;
      }
    }
    lpart = lpart * corr + psum;
    if (__ballot((corr != 1.0f && !was_empty) || !(odd < __builtin_inff()))) {
#pragma unroll
      for (int b = 0; b < kLatVB; ++b) acc[b] *= corr;
      // A row with a channel that is no number has such a score in every column.  Where a column
      // gives it no weight (a masked key, a score of -inf), p = 0 would not remove its values: they
      // become zeros, which change nothing for the columns whose p is NaN.  The wavefront clears
      // its own quarter of the tile (the swizzle stays inside it; another column block's
      // wavefront writes the same zeros) and reads it again.
      if (__ballot(!(odd < __builtin_inff()))) {
        int first = lane;
        asm volatile("" : "+v"(first));  // addresses are made here, not kept over the loop
#pragma unroll 1
        for (int u = first; u < kT * 16; u += kWave) {
          u32x4* at = reinterpret_cast<u32x4*>(lds[buf] + (u >> 4) * kLatRow + (chq * 16 + (u & 15)) * 16);
          u32x4 w = *at;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            uint32_t x = w[k];
            clear_non_numbers<kF16>(x);
            w[k] = x;
          }
          *at = w;
        }
        read_v(0);
      }
    }
    auto pv = [&](int b0) {
#pragma unroll
      for (int b = 0; b < kLatVB / 2; ++b)
#pragma unroll
        for (int g = 0; g < kCB; ++g) {
          acc[b0 + b] = mfma32<kF16>(vf[b][g], phi[g], acc[b0 + b]);
          acc[b0 + b] = mfma32<kF16>(vf[b][g], plo[g], acc[b0 + b]);
        }
    };
    pv(0);
    read_v(kLatVB / 2);
    pv(kLatVB / 2);
  };

  // Tile n + 1 is on its way into the other buffer while tile n is computed.  The barrier that
  // opens a step: every wavefront's rows of tile n have arrived, and tile n - 1's buffer is free.
  for (int32_t n = 0; n < tiles; ++n) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (n + 1 < tiles) load_tile(n + 1, (n + 1) & 1);
    compute(n & 1, kbeg + n * kT);
  }

  // ---- output: lane (col, grp) holds channels 128 chq + 16 b + 4 grp + e of its column
  const float lsum = col_sum(lpart);
  if (!qvalid) return;
  const bool direct = p.splits == 1;
  float lse_v;
  const float inv = direct ? finish(p, hq, mrun, lsum, &lse_v) : (lsum > 0.0f ? 1.0f / lsum : 0.0f);
  const int d0 = chq * 128 + 4 * grp;
  if (!direct) {
    float* ws_row = p.ws + ((((i * p.Hkv + hk) * p.splits + split) * p.ncols + c) * (int64_t)(kLatDv + 2));
    if (chq == 0 && grp == 0) {
      ws_row[0] = mrun;
      ws_row[1] = lsum;
    }
#pragma unroll
    for (int b = 0; b < kLatVB; ++b) {
      typedef float f32x2 __attribute__((ext_vector_type(2)));
      f32x2* w = reinterpret_cast<f32x2*>(ws_row + 2 + d0 + 16 * b);  // rows are 8-byte aligned
      w[0] = f32x2{acc[b][0] * inv, acc[b][1] * inv};
      w[1] = f32x2{acc[b][2] * inv, acc[b][3] * inv};
    }
    return;
  }
  const int64_t orow = i * p.o_sb + qrow * p.o_ss + (int64_t)hq * p.o_sh;
#pragma unroll
  for (int b = 0; b < kLatVB; ++b) store_out4(p, orow + d0 + 16 * b, acc[b] * inv);
  if (chq == 0 && grp == 0 && p.lse)
    p.lse[i * p.lse_sb + qrow * p.lse_ss + (int64_t)hq * p.lse_sh] = lse_v;
}

template <bool kF16, int kCB>
int launch(const AttnParams& p, hipStream_t st) {
  const dim3 grid = attn_grid(p, (p.ncb + kCB - 1) / kCB);
  const dim3 block(256 * kCB);
  return p.mask ? launch_kernel(attn_latent<kF16, kCB, true>, grid, block, st, p)
                : launch_kernel(attn_latent<kF16, kCB, false>, grid, block, st, p);
}

}  // namespace

// One column block takes workgroups of four wavefronts and 32-row tiles (two workgroups per CU),
// more take pairs of blocks, eight wavefronts and 64-row tiles (one workgroup per CU): the same
// 147 KB of LDS and 256 registers per lane either way, and a row read once for 32 columns.
int launch_attn_latent(const AttnParams& p, hipStream_t st) {
  const bool f16 = p.c_dtype == TMO_DTYPE_F16;
  if (p.ncb <= 1) return f16 ? launch<true, 1>(p, st) : launch<false, 1>(p, st);
  return f16 ? launch<true, 2>(p, st) : launch<false, 2>(p, st);
}

}  // namespace tmo
