// Direct kernel instances: GPTQ (and GPTQ_SYM: no zeros, offset 8), fp16.
#include "direct_inst.h"

namespace w4a16 {

hipError_t launch_direct_gptq(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    return launch_direct_dense<FMT_GPTQ, half_t>(p, s, st);
}

}  // namespace w4a16
