#include "kern_mix_launch.hpp"

namespace mifft {

hipError_t launch_mix_f64(int ldm, int stm, int post, const LineArgs& a, const Mix& mx, hipStream_t s) {
    return launch_mix_fmt<FmtF64>(ldm, stm, post, a, mx, s);
}

}  // namespace mifft
