// prefill_split.hip -- prefill_kernel with each tile's keys split between two
// waves, for steps whose workgroups would leave the chip idle.
#include "prefill_kernel.hpp"

namespace vmc {

int launch_prefill_split(PrefillParams& prm, bool bf16, int fmt, int src, bool vt, hipStream_t s) {
    return launch_prefill_any<2>(prm, bf16, fmt, src, vt, s);
}

}  // namespace vmc
