// Fused Rader and Bluestein line convolutions on the register stages of
// mix_kernels.hpp (the algorithms are in conv_kernels.hpp).
//
// The second transform runs the first one's radices in reverse, so that the
// outputs of the first one's last stage (k = j + i M / R of butterfly j) are
// the inputs of the second one's first stage in the same registers: last
// stage, filter multiply and first stage are one pass over LDS.  A tile of
// S-stage lines crosses LDS 2 S - 2 times (plus Rader's two permutations),
// where the LDS-to-LDS form crosses it 4 S + 4 times and keeps two buffers.
// Bound by those exchanges and the vector units (1009 points: two transforms
// of 1008 points per line).  us per pass, LDS-to-LDS -> this, over one pair of
// arrays: 8192 lines of 1009 points 99 -> 54 (three pairs in turn, beyond the
// last-level cache: 99.7 -> 61.4, 2.2 TB/s), 65536 of 127 100 -> 47, 2^18 of 31
// 125 -> 55, 4096 of 2003 120 -> 60, 1000 of 7561 143 -> 91, f64 4096 of 1009
// 97 -> 59, f64 Bluestein 4096 of 611 103 -> 73.
#pragma once
#include "conv_kernels.hpp"
#include "mix_kernels.hpp"

namespace mifft {

// The reversed schedule's stage 0 follows the last stage `fs` of the first
// transform: X = swap(A F), no exchange between.  keep (Rader): bin 0 of line
// lg to keep[lg].
template <int R, int NB, class T>
__device__ __forceinline__ void mix_turn(const MixConv& mc, const MixStage& fs, const MixStage& rs, const cpx<T>* src,
                                         cpx<T>* dst, const void* tw, const void* filt, cpx<T>* keep) {
    const Mix& mx = mc.f;
    const uint32_t total = mx.lpw * fs.nr;
    for (uint32_t r0 = 0; r0 < total; r0 += blockDim.x * NB) {
        const uint32_t b0 = r0 + threadIdx.x;
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, fs, b < total ? b : total - 1, false);
        }
        mix_take<R, NB, T>(mx, fs, src, tw, at, w);
#pragma unroll
        for (int q = 0; q < NB; q++) {
            if (keep && at[q].j == 0) keep[at[q].lg] = w[q][0];
#pragma unroll
            for (int i = 0; i < R; i++) w[q][i] = swap_ri(cmul(w[q][i], ld_tw<T>(filt, at[q].j + i * fs.nr)));
            Dft<R, T>::run(w[q]);
        }
        if (!mx.pp) __syncthreads();
#pragma unroll
        for (int q = 0; q < NB; q++)
            if (b0 + q * blockDim.x < total) mix_put<R, T>(mx, rs, dst, at[q], w[q]);
    }
}

// Rader's stage 0: a[q] = x[g^q] (zero from p - 1 on) out of the natural-order
// line in LDS.
template <int R, int NB, class T>
__device__ __forceinline__ void mix_rader_in(const ConvArgs& c, const MixStage& st, const cpx<T>* src, cpx<T>* dst,
                                             cpx<T>* x0) {
    const Mix& mx = c.mx.f;
    const uint32_t total = mx.lpw * st.nr, p1 = c.n - 1;
    for (uint32_t r0 = 0; r0 < total; r0 += blockDim.x * NB) {
        const uint32_t b0 = r0 + threadIdx.x;
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, false);
            const cpx<T>* xl = src + at[q].lg * mx.lstr;
            uint32_t e[R];
#pragma unroll
            for (int i = 0; i < R; i++) {
                const uint32_t k = at[q].j + i * st.nr;
                e[i] = gptr<uint32_t>(c.perm_in)[k < p1 ? k : 0];
            }
#pragma unroll
            for (int i = 0; i < R; i++) {
                const cpx<T> v = xl[e[i]];
                w[q][i] = at[q].j + i * st.nr < p1 ? v : mk<T>(T(0), T(0));
            }
            if (at[q].j == 0) x0[at[q].lg] = xl[0];
        }
#pragma unroll
        for (int q = 0; q < NB; q++) Dft<R, T>::run(w[q]);
        if (!mx.pp) __syncthreads();
#pragma unroll
        for (int q = 0; q < NB; q++)
            if (b0 + q * blockDim.x < total) mix_put<R, T>(mx, st, dst, at[q], w[q]);
    }
}

// Rader's last stage: X[g^-u] = x[0] + c[u] into natural order in LDS.
template <int R, int NB, class T>
__device__ __forceinline__ void mix_rader_out(const ConvArgs& c, const MixStage& st, const cpx<T>* src, cpx<T>* dst,
                                              const cpx<T>* x0, const cpx<T>* s0) {
    const Mix& mx = c.mx.r;
    const uint32_t total = mx.lpw * st.nr, p1 = c.n - 1;
    for (uint32_t r0 = 0; r0 < total; r0 += blockDim.x * NB) {
        const uint32_t b0 = r0 + threadIdx.x;
        cpx<T> w[NB][R];
        MixPos at[NB];
        uint32_t e[NB][R];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, false);
#pragma unroll
            for (int i = 0; i < R; i++) {
                const uint32_t u = at[q].j + i * st.nr;
                e[q][i] = gptr<uint32_t>(c.perm_out)[u < p1 ? u : 0];
            }
        }
        mix_take<R, NB, T>(mx, st, src, c.mx.rtw, at, w);
        if (!mx.pp) __syncthreads();
#pragma unroll
        for (int q = 0; q < NB; q++) {
            if (b0 + q * blockDim.x >= total) continue;
            cpx<T>* yl = dst + at[q].lg * mx.lstr;
            const cpx<T> x = x0[at[q].lg];
            if (at[q].j == 0) yl[0] = x + s0[at[q].lg];
#pragma unroll
            for (int i = 0; i < R; i++)
                if (at[q].j + i * st.nr < p1) yl[e[q][i]] = x + swap_ri(w[q][i]);
        }
    }
}

// Bluestein's stage 0: x[q] c[q] from memory, zero from n on.
template <class Fmt, int R, int NB>
__device__ __forceinline__ void mix_chirp_in(const ConvArgs& c, const MixStage& st, cpx<typename Fmt::T>* dst, uint32_t g0) {
    using T = typename Fmt::T;
    const Mix& mx = c.mx.f;
    const LineArgs& a = c.io;
    const uint32_t total = mx.lpw * st.nr, n = c.n;
    for (uint32_t b0 = threadIdx.x; b0 < total; b0 += blockDim.x * NB) {
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, mx.ld_lf);
            const uint32_t g = g0 + at[q].lg;
            const LineBase lb = line_base(a, g < a.lines ? g : a.lines - 1);
#pragma unroll
            for (int i = 0; i < R; i++) {
                const uint32_t k = at[q].j + i * st.nr;
                w[q][i] = load_point_at<Fmt, LD_COMPLEX, false>(a, lb.in + (k < n ? k : n - 1) * (uint32_t)a.in_sn);
            }
#pragma unroll
            for (int i = 0; i < R; i++) {
                const uint32_t k = at[q].j + i * st.nr;
                w[q][i] = k < n ? cmul(w[q][i], ld_tw<T>(c.chirp, k < n ? k : 0)) : mk<T>(T(0), T(0));
            }
        }
#pragma unroll
        for (int q = 0; q < NB; q++) {
            Dft<R, T>::run(w[q]);
            if (b0 + q * blockDim.x < total) mix_put<R, T>(mx, st, dst, at[q], w[q]);
        }
    }
}

// Bluestein's last stage: X[k] = swap(w) c[k] to memory, k < n.
template <class Fmt, int R, int NB>
__device__ __forceinline__ void mix_chirp_out(const ConvArgs& c, const MixStage& st, const cpx<typename Fmt::T>* src,
                                              uint32_t g0) {
    using T = typename Fmt::T;
    const Mix& mx = c.mx.r;
    const LineArgs& a = c.io;
    const uint32_t total = mx.lpw * st.nr, n = c.n;
    for (uint32_t b0 = threadIdx.x; b0 < total; b0 += blockDim.x * NB) {
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, mx.st_lf);
        }
        mix_take<R, NB, T>(mx, st, src, c.mx.rtw, at, w);
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t g = g0 + at[q].lg;
            if (b0 + q * blockDim.x >= total || g >= a.lines) continue;
            const LineBase lb = line_base(a, g);
#pragma unroll
            for (int i = 0; i < R; i++) {
                const uint32_t k = at[q].j + i * st.nr;
                if (k < n)
                    store_point_at<Fmt, ST_COMPLEX, false>(a, lb.out + k * (uint32_t)a.out_sk, lb.j, k, n,
                                                           cmul(swap_ri(w[q][i]), ld_tw<T>(c.chirp, k)));
            }
        }
    }
}

// The middle stages of one of the two transforms; swaps src and dst along.
template <class T>
__device__ __forceinline__ void mix_middle(const Mix& mx, cpx<T>*& src, cpx<T>*& dst, const void* tw) {
#pragma nounroll
    for (uint32_t s = 1; s + 1 < mx.ns; s++) {
        const MixStage st = mx.st[s];
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_mid<R, NB, T>(mx, st, src, dst, tw); break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
        __syncthreads();
        cpx<T>* x = src;
        src = dst;
        dst = x;
    }
}

// Lines [g0, g0 + lpw).
template <class Fmt, bool RADER>
__device__ __forceinline__ void mix_conv_tile(const ConvArgs& c, unsigned char* smem, uint32_t g0) {
    using T = typename Fmt::T;
    const Mix& f = c.mx.f;
    const LineArgs& a = c.io;
    cpx<T>* src = reinterpret_cast<cpx<T>*>(smem);
    cpx<T>* dst = src + f.pp;
    cpx<T>* x0 = src + f.lpw * f.lstr + f.pp;  // lpw entries
    cpx<T>* s0 = x0 + f.lpw;                   // lpw entries
    const uint32_t tpl = slot_tpl(f.lpw), slots = tpl * f.lpw, p = c.n;
    if constexpr (RADER) {
        // the lines in natural order into LDS (coalesced; lines past the end
        // read the last line and are never stored)
        for (uint32_t s = threadIdx.x; s < slots; s += blockDim.x) {
            const LineSlot m = line_slot(s, f.lpw, tpl, f.ld_lf);
            const uint32_t g = g0 + m.l;
            const LineBase b = line_base(a, g < a.lines ? g : a.lines - 1);
            for (uint32_t q0 = m.t; q0 < p; q0 += tpl * kChunk) {
                cpx<T> v[kChunk];
#pragma unroll
                for (uint32_t u = 0; u < kChunk; u++) {
                    const uint32_t q = q0 + u * tpl;
                    v[u] = load_point_at<Fmt, LD_COMPLEX, false>(a, b.in + (q < p ? q : p - 1) * (uint32_t)a.in_sn);
                }
#pragma unroll
                for (uint32_t u = 0; u < kChunk; u++) {
                    const uint32_t q = q0 + u * tpl;
                    if (q < p) src[m.l * f.lstr + q] = v[u];
                }
            }
        }
        __syncthreads();
    }
    {
        const MixStage st = f.st[0];
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB)                                                      \
    case R + 32 * NB:                                                              \
        if constexpr (RADER) mix_rader_in<R, NB, T>(c, st, src, dst, x0);          \
        else mix_chirp_in<Fmt, R, NB>(c, st, src, g0);                             \
        break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
    }
    if constexpr (RADER) {
        cpx<T>* x = src;
        src = dst;
        dst = x;
    }
    __syncthreads();
    mix_middle<T>(f, src, dst, a.tw);
    {
        const MixStage fs = f.st[f.ns - 1], rs = c.mx.r.st[0];
        switch (fs.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_turn<R, NB, T>(c.mx, fs, rs, src, dst, a.tw, c.filt, RADER ? s0 : nullptr); break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
    }
    cpx<T>* x = src;
    src = dst;
    dst = x;
    __syncthreads();
    mix_middle<T>(c.mx.r, src, dst, c.mx.rtw);
    {
        const MixStage st = c.mx.r.st[f.ns - 1];
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB)                                                           \
    case R + 32 * NB:                                                                   \
        if constexpr (RADER) mix_rader_out<R, NB, T>(c, st, src, dst, x0, s0);          \
        else mix_chirp_out<Fmt, R, NB>(c, st, src, g0);                                 \
        break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
    }
    if constexpr (RADER) {
        __syncthreads();
        for (uint32_t s = threadIdx.x; s < slots; s += blockDim.x) {
            const LineSlot m = line_slot(s, f.lpw, tpl, f.st_lf);
            const uint32_t g = g0 + m.l;
            if (g >= a.lines) continue;
            const LineBase b = line_base(a, g);
            for (uint32_t k = m.t; k < p; k += tpl)
                store_point<Fmt, ST_COMPLEX, false>(a, b.out, b.j, k, p, dst[m.l * f.lstr + k]);
        }
    }
}

// f64 tiles of up to 512 threads keep three waves per SIMD (168 registers; 198
// unbounded leave two): 4096 lines of 1009 points 66 -> 58 us, Bluestein 611
// points 74 -> 64.  In f32 a bound below the 111 registers asked for measured
// slower.
template <class Fmt, bool RADER, int NT>
__global__ void __launch_bounds__(NT, Fmt::kId == 0 || NT > 512 ? 4 : 3) mix_conv_kernel(ConvArgs c) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    mix_conv_tile<Fmt, RADER>(c, smem_raw, xcd_remap(blockIdx.x, gridDim.x) * c.mx.f.lpw);
}

// Launcher of one format (each compiles in a file of its own).
template <class Fmt>
static hipError_t launch_mix_conv_fmt(bool rader, const ConvArgs& c, hipStream_t s) {
    const Mix& f = c.mx.f;
    if (!c.mix || f.ns < 2 || f.nt > 1024) return hipErrorInvalidValue;
    const void* fn;
    if constexpr (Fmt::kId == 0)
        fn = rader ? (const void*)&mix_conv_kernel<Fmt, true, 1024> : (const void*)&mix_conv_kernel<Fmt, false, 1024>;
    else if (f.nt <= 512)
        fn = rader ? (const void*)&mix_conv_kernel<Fmt, true, 512> : (const void*)&mix_conv_kernel<Fmt, false, 512>;
    else
        fn = rader ? (const void*)&mix_conv_kernel<Fmt, true, 1024> : (const void*)&mix_conv_kernel<Fmt, false, 1024>;
    const size_t bytes = mix_conv_lds_bytes(Fmt::kId == 0 ? P_F32 : P_F64, c.mx);
    hipError_t e = ensure_lds_attr(fn, bytes);
    if (e != hipSuccess) return e;
    ConvArgs copy = c;
    void* args[] = {&copy};
    return hipLaunchKernel(fn, dim3((c.io.lines + f.lpw - 1) / f.lpw), dim3(f.nt), args, bytes, s);
}

}  // namespace mifft
