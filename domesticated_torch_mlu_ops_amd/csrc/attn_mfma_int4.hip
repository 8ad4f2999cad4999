// attn_mfma over int4-pair caches.
#include "attn_mfma.h"

namespace tmo {

int launch_attn_int4(const AttnParams& p, bool qlo, hipStream_t st) { return launch_mfma<4>(p, qlo, st); }

}  // namespace tmo
