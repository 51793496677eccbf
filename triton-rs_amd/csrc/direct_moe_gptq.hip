// Direct kernel instances by expert: GPTQ.
#include "direct_inst.h"

namespace w4a16 {

hipError_t launch_direct_moe_gptq(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    return launch_direct_moe_f<FMT_GPTQ>(p, s, st);
}

}  // namespace w4a16
