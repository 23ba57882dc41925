#include "mix_conv.hpp"

namespace mifft {

hipError_t launch_mix_conv_df64(bool rader, const ConvArgs& c, hipStream_t s) {
    return launch_mix_conv_fmt<FmtDF64>(rader, c, s);
}

}  // namespace mifft
