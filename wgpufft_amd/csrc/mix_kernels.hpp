// Line FFTs of any {2,3,5,7,11,13}-smooth length with a runtime radix
// schedule whose butterflies stay in registers.
//
// A tile holds `lpw` lines.  Stage 0 loads its butterflies straight from
// memory, the last stage stores straight to memory, and the stages exchange
// through LDS once per stage boundary.  The runtime-schedule engine of
// fft_kernels.hpp (lds_fft_lines) instead copies memory to LDS, runs every
// stage LDS to LDS and copies LDS to memory: 2 S + 2 passes over LDS for S
// stages instead of 2 (S - 1), and two buffers instead of one.
//
// Butterflies are flat over the tile: butterfly b of stage s is butterfly j =
// b mod (n / R_s) of line b / (n / R_s) (lines first where a strided side
// wants adjacent lanes on adjacent lines), so a tile fills its threads
// whatever n / R_s is.  A stage's radix R and unroll NB are compile-time
// constants behind one uniform switch per stage.
//
// What bounds it: memory for short lines (108 points: 5.6 TB/s, the copy rate
// of the card), and for longer ones the exchanges' latency and the vector
// units together (1000 points 3.6-4.5 TB/s; no packed f32).  Against the
// LDS-to-LDS engine, in us: 1000 x 4000 columns and rows (the passes of 10^6
// points x 4) 87 -> 46; 270 x 28822 59 -> 36; one 1000-point line 12.4 -> 7.1
// (call included); 104x140x60 f64 forward and inverse 118 -> 61.
// Loads are plain ones: a butterfly's runs of n / R points share cache lines
// with their neighbours'.
//
// LDS layout between stage s (radix R, previous product L) and the next: output
// m of butterfly j at m * nrp + j, nrp = (n / R) | 1.  Writes are contiguous
// over lanes; output point p = kq L R + m L + k of the Stockham order belongs
// to butterfly j = kq L + k, so the next stage finds its points at one base
// plus a uniform step (two small divisions per butterfly, one add per point,
// where a padded linear order takes three operations per point and side).
// The odd nrp spreads a wave that reads R outputs of neighbouring butterflies
// over the banks.
#pragma once
#include "launch.h"

namespace mifft {

// floor(x / d) for x, d < 2^16 (d = 1 is coded as 0).
__device__ __forceinline__ uint32_t mix_div(uint32_t x, uint32_t mag) { return mag ? __umulhi(x, mag) : x; }

// The compiled (radix, unroll) pairs: NB butterflies of radix R per thread
// and round, up to 16 points (mix_plan.cpp: nb_for).
#define MIFFT_MIX_RADICES(X)                                                                      \
    X(2, 4) X(3, 4) X(4, 1) X(4, 4) X(5, 1) X(5, 3) X(6, 2) X(7, 2) X(8, 1) X(8, 2) X(9, 1)       \
    X(10, 1) X(11, 1) X(12, 1) X(13, 1) X(14, 1) X(15, 1) X(16, 1)

// Line and butterfly of flat index b.
struct MixPos {
    uint32_t lg, j;
};
__device__ __forceinline__ MixPos mix_pos(const Mix& mx, const MixStage& st, uint32_t b, bool lf) {
    MixPos p;
    if (lf) {
        p.j = mix_div(b, mx.dlpw);
        p.lg = b - p.j * mx.lpw;
    } else {
        p.lg = mix_div(b, st.dnr);
        p.j = b - p.lg * st.nr;
    }
    return p;
}

// Reads butterfly p of a stage s >= 1 from LDS, twiddles and transforms it.
// The twiddle loads are issued first: they do not depend on the exchange.
template <int R, int NB, class T>
__device__ __forceinline__ void mix_take(const Mix& mx, const MixStage& st, const cpx<T>* src, const void* tw,
                                         const MixPos (&at)[NB], cpx<T> (&w)[NB][R]) {
    cpx<T> t[NB][R];
    uint32_t adr[NB];
#pragma unroll
    for (int q = 0; q < NB; q++) {
        const uint32_t kq = mix_div(at[q].j, st.dL), k = at[q].j - kq * st.L;
        const uint32_t m = mix_div(k, st.dLp), kk = k - m * st.Lp;
        adr[q] = at[q].lg * mx.lstr + m * st.nrp_prev + kq * st.Lp + kk;
#pragma unroll
        for (int i = 1; i < R; i++) t[q][i] = ld_tw<T>(tw, st.twoff + (i - 1) * st.L + k);
    }
#pragma unroll
    for (int q = 0; q < NB; q++)
#pragma unroll
        for (int i = 0; i < R; i++) w[q][i] = src[adr[q] + i * st.rstep];
#pragma unroll
    for (int q = 0; q < NB; q++) {
#pragma unroll
        for (int i = 1; i < R; i++) w[q][i] = cmul(w[q][i], t[q][i]);
        Dft<R, T>::run(w[q]);
    }
}

// Outputs of a butterfly into LDS.
template <int R, class T>
__device__ __forceinline__ void mix_put(const Mix& mx, const MixStage& st, cpx<T>* dst, MixPos p, const cpx<T> (&w)[R]) {
    const uint32_t a = p.lg * mx.lstr + p.j;
#pragma unroll
    for (int i = 0; i < R; i++) dst[a + i * st.nrp] = w[i];
}

// Stage 0: memory -> LDS.  Lines past the end read the last line and are
// never stored.
template <class Fmt, int LDM, int R, int NB>
__device__ __forceinline__ void mix_first(const LineArgs& a, const Mix& mx, cpx<typename Fmt::T>* dst, uint32_t g0) {
    using T = typename Fmt::T;
    const MixStage& st = mx.st[0];
    const uint32_t total = mx.lpw * st.nr;
    for (uint32_t b0 = threadIdx.x; b0 < total; b0 += blockDim.x * NB) {
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, mx.ld_lf);
            const uint32_t g = g0 + at[q].lg;
            const LineBase lb = line_base(a, g < a.lines ? g : a.lines - 1);
            const uint32_t o0 = lb.in + at[q].j * (uint32_t)a.in_sn, sn = st.nr * (uint32_t)a.in_sn;
#pragma unroll
            for (int i = 0; i < R; i++) w[q][i] = load_point_at<Fmt, LDM, false>(a, o0 + i * sn);
        }
#pragma unroll
        for (int q = 0; q < NB; q++) {
            Dft<R, T>::run(w[q]);
            if (b0 + q * blockDim.x < total) mix_put<R, T>(mx, st, dst, at[q], w[q]);
        }
    }
}

// A middle stage: LDS -> LDS, within one buffer (every butterfly of the tile
// in registers across the barrier; the host sees to one round) or into the
// second one.  Every thread calls it.
template <int R, int NB, class T>
__device__ __forceinline__ void mix_mid(const Mix& mx, const MixStage& st, const cpx<T>* src, cpx<T>* dst, const void* tw) {
    const uint32_t total = mx.lpw * st.nr;
    for (uint32_t r0 = 0; r0 < total; r0 += blockDim.x * NB) {
        const uint32_t b0 = r0 + threadIdx.x;
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, false);
        }
        mix_take<R, NB, T>(mx, st, src, tw, at, w);
        if (!mx.pp) __syncthreads();
#pragma unroll
        for (int q = 0; q < NB; q++)
            if (b0 + q * blockDim.x < total) mix_put<R, T>(mx, st, dst, at[q], w[q]);
    }
}

// The last stage: LDS -> memory, outputs k = j + i n / R.
template <class Fmt, int STM, bool POST, int R, int NB>
__device__ __forceinline__ void mix_last(const LineArgs& a, const Mix& mx, const MixStage& st,
                                         const cpx<typename Fmt::T>* src, uint32_t g0) {
    using T = typename Fmt::T;
    const uint32_t total = mx.lpw * st.nr;
    for (uint32_t b0 = threadIdx.x; b0 < total; b0 += blockDim.x * NB) {
        cpx<T> w[NB][R];
        MixPos at[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t b = b0 + q * blockDim.x;
            at[q] = mix_pos(mx, st, b < total ? b : total - 1, mx.st_lf);
        }
        mix_take<R, NB, T>(mx, st, src, a.tw, at, w);
#pragma unroll
        for (int q = 0; q < NB; q++) {
            const uint32_t g = g0 + at[q].lg;
            if (b0 + q * blockDim.x >= total || g >= a.lines) continue;
            const LineBase lb = line_base(a, g);
            const uint32_t o0 = lb.out + at[q].j * (uint32_t)a.out_sk, sk = st.nr * (uint32_t)a.out_sk;
            PostSeq ps;
            if constexpr (POST) ps.init(a, lb.j, at[q].j, st.nr);
#pragma unroll
            for (int i = 0; i < R; i++) {
                cpx<T> v = w[q][i];
                if constexpr (POST) v = cmul(v, ps.template next<T>());
                store_point_at<Fmt, STM, false>(a, o0 + i * sk, lb.j, at[q].j + i * st.nr, mx.n, v);
            }
        }
    }
}

// Lines [g0, g0 + lpw) of ns >= 2 stages: memory -> stages -> memory.
template <class Fmt, int LDM, int STM, bool POST>
__device__ __forceinline__ void mix_tile(const LineArgs& a, const Mix& mx, unsigned char* smem, uint32_t g0) {
    using T = typename Fmt::T;
    cpx<T>* src = reinterpret_cast<cpx<T>*>(smem);
    cpx<T>* dst = src + mx.pp;
    switch (mx.st[0].code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_first<Fmt, LDM, R, NB>(a, mx, src, g0); break;
        MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
        default: break;
    }
    __syncthreads();
#pragma nounroll
    for (uint32_t s = 1; s + 1 < mx.ns; s++) {
        const MixStage st = mx.st[s];
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_mid<R, NB, T>(mx, st, src, dst, a.tw); break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
        __syncthreads();
        cpx<T>* x = src;
        src = dst;
        dst = x;
    }
    const MixStage st = mx.st[mx.ns - 1];
    switch (st.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_last<Fmt, STM, POST, R, NB>(a, mx, st, src, g0); break;
        MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
        default: break;
    }
}

// NT: the launch bound (the register budget).
template <class Fmt, int LDM, int STM, bool POST, int NT>
__global__ void __launch_bounds__(NT) mix_fft_kernel(LineArgs a, Mix mx) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    mix_tile<Fmt, LDM, STM, POST>(a, mx, smem_raw, xcd_remap(blockIdx.x, gridDim.x) * mx.lpw);
}

}  // namespace mifft
