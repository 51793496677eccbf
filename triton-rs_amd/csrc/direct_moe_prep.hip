// Direct kernel instances by expert: the prepared layout.
#include "direct_inst.h"

namespace w4a16 {

hipError_t launch_direct_moe_prep(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    return launch_direct_moe_f<FMT_PREP>(p, s, st);
}

}  // namespace w4a16
