// Half-length real lines (mix_real_tile).
#include "mix_kernels.hpp"

namespace mifft {

hipError_t launch_mix_real(bool c2r, const LineArgs& a, const Mix& mx, hipStream_t s) {
    if (mx.nt > 1024 || mx.ns < 2 || !mx.pairs) return hipErrorInvalidValue;
    const void* fn = c2r         ? (const void*)&mix_real_kernel<true, false>
                     : mx.stream ? (const void*)&mix_real_kernel<false, true>
                                 : (const void*)&mix_real_kernel<false, false>;
    const size_t bytes = mix_lds_bytes(P_F32, mx);
    hipError_t e = ensure_lds_attr(fn, bytes);
    if (e != hipSuccess) return e;
    LineArgs ca = a;
    Mix cm = mx;
    void* args[] = {&ca, &cm};
    return hipLaunchKernel(fn, dim3((a.lines + mx.lpw - 1) / mx.lpw), dim3(mx.nt), args, bytes, s);
}

}  // namespace mifft
