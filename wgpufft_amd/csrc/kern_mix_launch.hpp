// Launcher of the runtime-schedule register line kernels of one format; each
// format's kernels compile in a file of their own (kern_mix_*.hip).
#pragma once
#include "mix_kernels.hpp"

namespace mifft {

// f32 kernels need 82 registers whatever the launch bound, so one form serves
// up to 1024 threads; f64 ones take 158 where at most 512 threads leave room.
template <class Fmt, int LDM, int STM, bool POST>
static const void* mix_fn(uint32_t nt) {
    if constexpr (Fmt::kId == 0) return (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 1024>;
    else
        return nt <= 512 ? (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 512>
                         : (const void*)&mix_fft_kernel<Fmt, LDM, STM, POST, 1024>;
}

template <class Fmt>
static hipError_t launch_mix_fmt(int ldm, int stm, int post, const LineArgs& a, const Mix& mx, hipStream_t s) {
    if (ldm != LD_COMPLEX || stm != ST_COMPLEX || mx.nt > 1024 || mx.ns < 2) return hipErrorInvalidValue;
    const void* fn = post ? mix_fn<Fmt, LD_COMPLEX, ST_COMPLEX, true>(mx.nt)
                          : mix_fn<Fmt, LD_COMPLEX, ST_COMPLEX, false>(mx.nt);
    const size_t bytes = mix_lds_bytes(Fmt::kId == 0 ? P_F32 : P_F64, mx);
    hipError_t e = ensure_lds_attr(fn, bytes);
    if (e != hipSuccess) return e;
    LineArgs ca = a;
    Mix cm = mx;
    void* args[] = {&ca, &cm};
    return hipLaunchKernel(fn, dim3((a.lines + mx.lpw - 1) / mx.lpw), dim3(mx.nt), args, bytes, s);
}

}  // namespace mifft
