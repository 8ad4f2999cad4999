// attn_mfma over int8 caches.
#include "attn_mfma.h"

namespace tmo {

int launch_attn_int8(const AttnParams& p, bool qlo, hipStream_t st) { return launch_mfma<0>(p, qlo, st); }

}  // namespace tmo
