// attn_mfma over bf16 and f16 caches.
#include "attn_mfma.h"

namespace tmo {

int launch_attn_plain(const AttnParams& p, hipStream_t st) {
  return p.c_dtype == TMO_DTYPE_BF16 ? launch_mfma<1>(p, false, st) : launch_mfma<2>(p, false, st);
}

}  // namespace tmo
