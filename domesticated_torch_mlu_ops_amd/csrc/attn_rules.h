// Host rules of the decode attention that the op (split counts) and the launcher (kernels) share.
#pragma once

#include <cstdint>

namespace tmo {

// The many-column kernel (attn_chunk, which unpacks a key once for 64 or 128 columns) takes the call,
// attn_mfma (16 columns) otherwise: `cols` query columns per (sequence, KV head) and `splits` of its
// keys.
//
// Head sizes 80 and 96 always: attn_mfma has no instance of them (nor attn_chunk of int4 x 80).
//
// Head sizes 64, 128 and 256 with four column blocks and more (49 columns) and more than five
// million (query column, key) pairs over the KV heads, for the longest context that the call
// announces (unknown: what its block tables can hold).  8 KV heads x 128, int8 pages, contexts of
// 512..8192, attn_mfma against it: 32 columns of 4 / 32 sequences 53 / 160 against 54 / 183 us, 64
// columns 72 / 267 against 55 / 193, 128 columns (32 sequences) 492 against 212, 2048 columns of 8
// sequences 1210 against 437.  Its workgroups walk their keys in one chain where attn_mfma's four
// wavefronts share them, so short or few sequences stay there: 1 / 8 sequences of 512 keys, 64
// columns, 8 KV heads, 18.8 / 19.4 against 26.9 / 27.8 us; 8 of 1024 (4.2 million pairs) 29.8
// against 34.8 us, of 2048 56.3 against 39.3; 288 columns, 2 KV heads, 8 of 1024 (4.7) 30.8 against
// 35.5, of 2048 51.0 against 42.0 us.
//
// For the same reason a single split (an unknown maximum) has to fill the chip with column blocks:
// 8 KV heads, 2048 int8 keys: 64 columns of 8 sequences (256 workgroups of attn_mfma) 45 against 81
// us, 256 of 1 (128) 41 against 78, 256 of 8 (1024) 110 against 81; head size 256 (int4), 64 columns
// of 8 and of 32 sequences 53 and 140 against 99 and 101.
//
// Codes of head size 64 are half the unpacking and MFMAs of 128, which attn_mfma hides better.  Half
// empty workgroups lose: 8 KV heads, 2048 keys, 64 columns of 32 sequences int8 / float8 / int4 79 /
// 78 / 66 against 82 / 83 / 88 us; 96 columns 112 / 109 / 90 against 83 / 83 / 92, 128 columns of 8
// sequences 57 / 55 / 49 against 31 / 31 / 31.  One split needs more column blocks: 256 columns of 8
// sequences (1024 workgroups of attn_mfma), float8, 53 against 60, 96 of 32 (1536) 87 against 62.
inline bool attn_many_columns(bool codes, bool int4, int64_t head_size, int64_t cols, int64_t kv_heads,
                              int64_t batch, int64_t max_context_len, int64_t table_keys,
                              int64_t splits) {
  if (head_size == 80 || head_size == 96) return !(int4 && head_size == 80);
  if (head_size != 64 && head_size != 128 && head_size != 256) return false;
  const int64_t keys = max_context_len > 0 ? max_context_len : table_keys;
  const int64_t blocks = (cols + 15) / 16, all = blocks * kv_heads * batch;
  if (blocks < 4 || (double)cols * (double)kv_heads * (double)batch * (double)keys <= 5e6) return false;
  if (codes && head_size == 64) return blocks >= (int4 ? 7 : 6) && (splits > 1 || all >= 1536);
  return splits > 1 || all >= 1024;
}

}  // namespace tmo
