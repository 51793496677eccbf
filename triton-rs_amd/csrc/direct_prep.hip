// Direct kernel instances: the prepared layout.
#include "direct_inst.h"

namespace w4a16 {

hipError_t launch_direct_prep(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    return launch_direct_dense<FMT_PREP, half_t>(p, s, st);
}

}  // namespace w4a16
