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
//
// Loads are non-temporal (mx.stream; kernels of their own) where a pass reads 32 MiB or more in runs
// of at least 192 bytes, or strided rows of 128 (64 MiB in and out: 1000
// points 39.4 -> 32.8 us, 1920 36.1 -> 31.4, 60-point rows 31.1 -> 27.6).
// Shorter runs share cache lines with their neighbours' (60 contiguous points
// 36.3 -> 41.5 us with the hint, 32-byte strided rows 45.6 -> 53.2), and
// smaller arrays stay in the last-level cache (3-8 % slower with it).
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
template <class Fmt, int LDM, bool NTL, int R, int NB>
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
            for (int i = 0; i < R; i++) w[q][i] = load_point_at<Fmt, LDM, NTL>(a, o0 + i * sn);
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

// The last stage: LDS -> memory, outputs k = j + i n / R.  SCALE: times a.scale
// (half-length C2R lines were scaled with their bin pairs).
template <class Fmt, int STM, bool POST, int R, int NB, bool SCALE = true>
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
            // (f64: a factor of its own per output, 82.6 -> 87.1 us for five lines of
            // 10^6 points; carried from output to output its error grows, 5.3e-16 ->
            // 6.3e-16 over such a line)
            if constexpr (POST && sizeof(T) == 4) ps.init(a, lb.j, at[q].j, st.nr);
#pragma unroll
            for (int i = 0; i < R; i++) {
                cpx<T> v = w[q][i];
                if constexpr (POST && sizeof(T) == 4) v = cmul(v, ps.template next<T>());
                else if constexpr (POST) v = cmul(v, post_twiddle<T>(a, (uint64_t)lb.j * (at[q].j + i * st.nr)));
                if constexpr (SCALE) store_point_at<Fmt, STM, false>(a, o0 + i * sk, lb.j, at[q].j + i * st.nr, mx.n, v);
                else Fmt::st(a.out, o0 + i * sk, conj_by(v, sign_mask(a.conj_out)));
            }
        }
    }
}

template <class Fmt, int LDM, bool NTL>
__device__ __forceinline__ void mix_load(const LineArgs& a, const Mix& mx, cpx<typename Fmt::T>* dst, uint32_t g0) {
    switch (mx.st[0].code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_first<Fmt, LDM, NTL, R, NB>(a, mx, dst, g0); break;
        MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
        default: break;
    }
}

// Lines [g0, g0 + lpw) of ns >= 2 stages: memory -> stages -> memory.
// NTL: non-temporal loads.
template <class Fmt, int LDM, int STM, bool POST, bool NTL = false>
__device__ __forceinline__ void mix_tile(const LineArgs& a, const Mix& mx, unsigned char* smem, uint32_t g0) {
    using T = typename Fmt::T;
    cpx<T>* src = reinterpret_cast<cpx<T>*>(smem);
    cpx<T>* dst = src + mx.pp;
    mix_load<Fmt, LDM, NTL>(a, mx, src, g0);
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

// ------------------------------------------------ half-length real lines
// A real line of N0 = 2n points read as n complex ones, z[m] = x[2m] + i
// x[2m+1], with Z = DFT_n(z), has the bins (k <= n, W = W_N0^k)
//   X[k] = A + W B,  X[n - k] = conj(A - W B),
//   A = (Z[k] + conj Z[n-k]) / 2,  B = (Z[k] - conj Z[n-k]) / 2i;
// the inverse starts from
//   Z[k] = E + i O,  Z[n-k] = conj E + i conj O,
//   E = X[k] + conj X[n-k],  O = (X[k] - conj X[n-k]) conj W
// (the imaginary parts of bins 0 and n are dropped).  Half the points go
// through the stages, and the pairs k, n - k meet in LDS in natural order,
// joined and scaled (C2R: split and scaled) in 64 bits and rounded once (in 32
// bits 48000 x 400 R2C err 1.06e-7 instead of 9.9e-8, a 1920-point C2R line
// 1.25e-7 instead of 1.08e-7; R2C takes the same time, C2R 3 to 8 % more):
// one exchange more than a complex line of n points, where the full-length
// form runs N0-point lines whose upper half it drops.  48000 x 400 R2C 118 ->
// 44 us (154 MB, 3.5 TB/s; 30 us at the copy rate), 1920x1080x3 R2C + C2R 127
// -> 75 us, 144x120x108 52 -> 44 us.

// A stage from LDS to LDS whose side NAT_IN reads / NAT_OUT writes natural
// point order (stage 0 after, the last stage before the bin pairs); as mix_mid
// otherwise.
template <int R, int NB, bool NAT_IN, class T>
__device__ __forceinline__ void mix_nat(const Mix& mx, const MixStage& st, const cpx<T>* src, cpx<T>* dst, const void* tw) {
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
        if constexpr (NAT_IN) {
#pragma unroll
            for (int q = 0; q < NB; q++)
#pragma unroll
                for (int i = 0; i < R; i++) w[q][i] = src[at[q].lg * mx.lstr + at[q].j + i * st.nr];
#pragma unroll
            for (int q = 0; q < NB; q++) Dft<R, T>::run(w[q]);
        } else {
            mix_take<R, NB, T>(mx, st, src, tw, at, w);
        }
        if (!mx.pp) __syncthreads();
#pragma unroll
        for (int q = 0; q < NB; q++)
            if (b0 + q * blockDim.x < total) {
                if constexpr (NAT_IN) {
                    mix_put<R, T>(mx, st, dst, at[q], w[q]);
                } else {
#pragma unroll
                    for (int i = 0; i < R; i++) dst[at[q].lg * mx.lstr + at[q].j + i * st.nr] = w[q][i];
                }
            }
    }
}

// Bin pairs in flight per thread.
constexpr uint32_t kMixPairs = 4;

// R2C: LDS (natural order) -> packed bins.
template <class T>
__device__ __forceinline__ void mix_pairs_out(const LineArgs& a, const Mix& mx, const cpx<T>* z, uint32_t g0) {
    const uint32_t n = mx.n, total = mx.lpw * mx.pairs;
    const double sc = 0.5 * a.scale;  // the halves of A and B (exact)
    for (uint32_t t0 = threadIdx.x; t0 < total; t0 += blockDim.x) {
        const uint32_t lg = mix_div(t0, mx.dpairs), k = t0 - lg * mx.pairs, g = g0 + lg;
        if (g >= a.lines) return;
        const cpx<double> w = ld_tw<double>(a.half_tw, k);
        const cpx<T>* zl = z + lg * mx.lstr;
        const cpx<T> zp = zl[k], zq = zl[k ? n - k : 0];
        const cpx<double> p = mk<double>(zp.x, zp.y), q = mk<double>(zq.x, zq.y);
        const cpx<double> A = mk<double>(p.x + q.x, p.y - q.y), B = mk<double>(p.y + q.y, q.x - p.x);
        // A +- W B
        const double wbx = fma(w.x, B.x, -(w.y * B.y)), wby = fma(w.x, B.y, w.y * B.x);
        const uint32_t o = line_base(a, g).out;
        FmtF32::st(a.out, o + k, mk<T>((T)((A.x + wbx) * sc), (T)((A.y + wby) * sc)));
        if (2 * k != n) FmtF32::st(a.out, o + n - k, mk<T>((T)((A.x - wbx) * sc), (T)((wby - A.y) * sc)));
    }
}

// C2R: packed bins -> LDS, scaled and conjugated (the inverse is conj DFT conj).
template <class T>
__device__ __forceinline__ void mix_pairs_in(const LineArgs& a, const Mix& mx, cpx<T>* z, uint32_t g0) {
    const uint32_t n = mx.n, total = mx.lpw * mx.pairs;
    const double sc = a.scale;
    for (uint32_t t0 = threadIdx.x; t0 < total; t0 += blockDim.x * kMixPairs) {
        cpx<T> p[kMixPairs], q[kMixPairs];
        cpx<double> w[kMixPairs];
        uint32_t lg[kMixPairs], k[kMixPairs];
#pragma unroll
        for (uint32_t u = 0; u < kMixPairs; u++) {
            const uint32_t t = t0 + u * blockDim.x, tc = t < total ? t : total - 1;
            lg[u] = mix_div(tc, mx.dpairs);
            k[u] = tc - lg[u] * mx.pairs;
            const uint32_t g = g0 + lg[u], o = line_base(a, g < a.lines ? g : a.lines - 1).in;
            p[u] = FmtF32::ld_c(a.in, o + k[u]);
            q[u] = FmtF32::ld_c(a.in, o + n - k[u]);
            w[u] = ld_tw<double>(a.half_tw, k[u]);
        }
#pragma unroll
        for (uint32_t u = 0; u < kMixPairs; u++) {
            if (t0 + u * blockDim.x >= total) break;
            if (k[u] == 0) p[u].y = q[u].y = T(0);
            const cpx<double> P = mk<double>(p[u].x, p[u].y), Q = mk<double>(q[u].x, q[u].y);
            const cpx<double> E = mk<double>(P.x + Q.x, P.y - Q.y), D = mk<double>(P.x - Q.x, P.y + Q.y);
            const double wx = w[u].x, wy = w[u].y;
            const double ox = fma(wx, D.x, wy * D.y), oy = fma(wx, D.y, -(wy * D.x));  // O = D conj W
            // E + i O and conj E + i conj O, conjugated
            cpx<T>* zl = z + lg[u] * mx.lstr;
            zl[k[u]] = mk<T>((T)((E.x - oy) * sc), (T)((-E.y - ox) * sc));
            if (k[u] && 2 * k[u] != n) zl[n - k[u]] = mk<T>((T)((E.x + oy) * sc), (T)((E.y - ox) * sc));
        }
    }
}

// Lines [g0, g0 + lpw) of 2n real points (a's real side in complex elements).
template <bool C2R, bool NTL = false>
__device__ __forceinline__ void mix_real_tile(const LineArgs& a, const Mix& mx, unsigned char* smem, uint32_t g0) {
    using T = float;
    cpx<T>* src = reinterpret_cast<cpx<T>*>(smem);
    cpx<T>* dst = src + mx.pp;
    if constexpr (C2R) {
        mix_pairs_in<T>(a, mx, src, g0);
        __syncthreads();
        const MixStage st = mx.st[0];
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_nat<R, NB, true, T>(mx, st, src, dst, a.tw); break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
        cpx<T>* x = src;
        src = dst;
        dst = x;
    } else {
        mix_load<FmtF32, LD_COMPLEX, NTL>(a, mx, src, g0);
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
    if constexpr (C2R) {
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_last<FmtF32, ST_COMPLEX, false, R, NB, false>(a, mx, st, src, g0); break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
    } else {
        switch (st.code) {
#define MIFFT_MIX_CASE(R, NB) \
    case R + 32 * NB: mix_nat<R, NB, false, T>(mx, st, src, dst, a.tw); break;
            MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
            default: break;
        }
        __syncthreads();
        mix_pairs_out<T>(a, mx, dst, g0);
    }
}

template <bool C2R, bool NTL>
__global__ void __launch_bounds__(1024) mix_real_kernel(LineArgs a, Mix mx) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    mix_real_tile<C2R, NTL>(a, mx, smem_raw, xcd_remap(blockIdx.x, gridDim.x) * mx.lpw);
}

// NT: the launch bound.  Register budgets below what the stages ask for (72 or
// 64 in f32, 128 for 512 threads in f64) spill and measured 5-15 % slower.
template <class Fmt, int LDM, int STM, bool POST, int NT, bool NTL>
__global__ void __launch_bounds__(NT) mix_fft_kernel(LineArgs a, Mix mx) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    mix_tile<Fmt, LDM, STM, POST, NTL>(a, mx, smem_raw, xcd_remap(blockIdx.x, gridDim.x) * mx.lpw);
}

}  // namespace mifft
