// attn_mfma over float8_e4m3fn caches.
#include "attn_mfma.h"

namespace tmo {

int launch_attn_fp8(const AttnParams& p, bool qlo, hipStream_t st) { return launch_mfma<3>(p, qlo, st); }

}  // namespace tmo
