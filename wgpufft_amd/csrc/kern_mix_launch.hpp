// Launcher of the runtime-schedule register line kernels of one format; each
// format's kernels compile in a file of their own (kern_mix_*.hip).
#pragma once
#include "mix_kernels.hpp"

namespace mifft {

// f32 kernels need 82 registers (95 with the twiddle on store) whatever the
// launch bound, so one form serves up to 1024 threads; f64 ones take 158 to 166
// where at most 512 threads leave room, and have no non-temporal form above.
template <class Fmt, int LDM, int STM, bool POST>
static const void* mix_fn(const Mix& mx) {
    if constexpr (Fmt::kId == 0)
        return mx.stream ? (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 1024, true>
                         : (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 1024, false>;
    else if (mx.nt > 512)
        return (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 1024, false>;
    else
        return mx.stream ? (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 512, true>
                         : (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 512, false>;
}

template <class Fmt>
static hipError_t launch_mix_fmt(int ldm, int stm, int post, const LineArgs& a, const Mix& mx, hipStream_t s) {
    if (ldm != LD_COMPLEX || stm != ST_COMPLEX || mx.nt > 1024 || mx.ns < 2) return hipErrorInvalidValue;
    const void* fn = post ? mix_fn<Fmt, LD_COMPLEX, ST_COMPLEX, true>(mx)
                          : mix_fn<Fmt, LD_COMPLEX, ST_COMPLEX, false>(mx);
    const size_t bytes = mix_lds_bytes(Fmt::kId == 0 ? P_F32 : P_F64, mx);
    hipError_t e = ensure_lds_attr(fn, bytes);
    if (e != hipSuccess) return e;
    LineArgs ca = a;
    Mix cm = mx;
    void* args[] = {&ca, &cm};
    return hipLaunchKernel(fn, dim3((a.lines + mx.lpw - 1) / mx.lpw), dim3(mx.nt), args, bytes, s);
}

}  // namespace mifft
