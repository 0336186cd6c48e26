// kvrt_prefill_wide.hip — prefill instantiations of head_dim 256 and 512, whose
// output accumulators (128 and 256 registers) live in AGPRs.
#include "kvrt_prefill.h"

namespace kvrt {

hipError_t launch_prefill_wide(const PrefillArgs &a, int head_dim, hipStream_t s) {
    const int rw = a.row_waves, ks = a.key_parts;
    if (head_dim == 256) {
        if (rw == 4 && ks == 1) return launch_prefill_shape<256, 4, 1, 2>(a, s);
        if (rw == 2 && ks == 2) return launch_prefill_shape<256, 2, 2, 2>(a, s);
    }
    if (head_dim == 512) {
        if (rw == 4 && ks == 1) return launch_prefill_shape<512, 4, 1, 2>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace kvrt
