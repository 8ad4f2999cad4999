// Host rules of the decode attention that the op (split counts) and the launcher (kernels) share.
#pragma once

#include <cstdint>

namespace tmo {

// More than five million (query column, key) pairs over the KV heads of a call, for the longest context
// it announces (unknown: what its block tables can hold).
inline bool attn_large(int64_t cols, int64_t kv_heads, int64_t batch, int64_t max_context_len,
                       int64_t table_keys) {
  const int64_t keys = max_context_len > 0 ? max_context_len : table_keys;
  return (double)cols * (double)kv_heads * (double)batch * (double)keys > 5e6;
}

}  // namespace tmo
