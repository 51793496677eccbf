// Direct kernel instances: AWQ, fp16.
#include "direct_inst.h"

namespace w4a16 {

hipError_t launch_direct_awq(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    return launch_direct_dense<FMT_AWQ, half_t>(p, s, st);
}

}  // namespace w4a16
