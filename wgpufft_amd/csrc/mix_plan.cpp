// Host side of the runtime-schedule register kernels (mix_kernels.hpp): the
// radix schedule of a length and the shape (lines, threads, LDS) of a tile.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>

#include "launch.h"

namespace mifft {

// Arithmetic instructions of a radix-R butterfly (fft_math.hpp: symmetric
// pairs for odd primes, two factors for composites, without a twiddle between
// coprime ones).
static double butterfly_ops(int r) {
    static const double ops[17] = {0, 0, 4, 12, 16, 36, 36, 66, 52, 88, 92, 150, 96, 204, 160, 168, 152};
    return ops[r];
}
// Work of one stage per point: the butterfly, and in the same unit the
// twiddle multiply, one LDS write and read with their addresses and a share
// of the exchange's latency.
static double stage_cost(int r) { return butterfly_ops(r) / r + 14.0; }

static uint32_t mix_mag(uint32_t d) { return d <= 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d); }

// Smallest compiled unroll (MIFFT_MIX_RADICES) that covers `need`
// butterflies of radix r per thread, or the largest.
static uint32_t nb_for(int r, uint32_t need) {
    switch (r) {
        case 2: case 3: return 4;
        case 4: return need <= 1 ? 1 : 4;
        case 5: return need <= 1 ? 1 : 3;
        case 6: case 7: return 2;
        case 8: return need <= 1 ? 1 : 2;
        default: return 1;
    }
}

// Whether stage s of ns writes a second buffer: a stage from LDS to LDS that takes
// more than one round does (the middle ones, and the last (first) one where the
// bin pairs of real lines follow (precede) it).
static bool needs_second(bool real, uint32_t s, uint32_t ns, uint32_t need, uint32_t nb) {
    return (real || (s >= 1 && s + 1 < ns)) && need > nb;
}

static Mix shape(uint64_t n, const std::vector<int>& rad, uint32_t lpw, uint32_t nt, bool ld_lf, bool st_lf,
                 bool real) {
    Mix x;
    std::memset(&x, 0, sizeof(x));
    x.n = (uint32_t)n;
    x.ns = (uint32_t)rad.size();
    x.lpw = lpw;
    x.nt = nt;
    x.ld_lf = ld_lf;
    x.st_lf = st_lf;
    x.dlpw = mix_mag(lpw);
    if (real) {
        x.pairs = x.n / 2 + 1;
        x.dpairs = mix_mag(x.pairs);
    }
    uint32_t L = 1, twoff = 0;
    bool pp = false;
    for (uint32_t s = 0; s < x.ns; s++) {
        MixStage& st = x.st[s];
        const uint32_t R = (uint32_t)rad[s], nr = (uint32_t)n / R;
        const uint32_t need = (lpw * nr + nt - 1) / nt, nb = nb_for((int)R, need);
        st.code = R + 32 * nb;
        st.nr = nr;
        st.nrp = nr | 1u;
        st.L = L;
        st.Lp = s ? L / (uint32_t)rad[s - 1] : 1;
        st.nrp_prev = s ? x.st[s - 1].nrp : 0;
        st.rstep = ((uint32_t)n / (L * R)) * st.Lp;
        st.twoff = twoff;
        st.dnr = mix_mag(nr);
        st.dL = mix_mag(L);
        st.dLp = mix_mag(st.Lp);
        if (s >= 1) twoff += (R - 1) * L;
        if (s + 1 < x.ns) x.lstr = std::max(x.lstr, R * st.nrp);
        pp |= needs_second(real, s, x.ns, need, nb);
        L *= R;
    }
    x.lstr |= 1u;
    x.pp = pp ? lpw * x.lstr : 0;
    return x;
}

size_t mix_lds_bytes(int arith, const Mix& x) {
    if (x.ns <= 1) return 0;
    return (size_t)(x.pp ? 2 : 1) * x.lpw * x.lstr * (arith == P_F32 ? 8 : 16);
}

// Factor of the threads of a workgroup in shape_score: its upper bound too.
static double thread_score(uint32_t nt) { return nt <= 256 ? 1.0 : nt < 512 ? 0.80 : nt == 512 ? 0.78 : 0.68; }

// Factor of the workgroups, at least two per CU where the lines allow it: falls
// with the lines of a workgroup.
static double fill_score(uint64_t lines, uint32_t lpw) {
    const double wgs = std::ceil((double)lines / lpw), want = 2.0 * device_cu_count();
    return wgs < want && lpw > 1 ? 0.3 + 0.7 * wgs / want : 1.0;
}

// What the shapes of one schedule share.
struct Stages {
    uint32_t ns, lstr;
    uint32_t r[kMixStages], nr[kMixStages];
    double w[kMixStages];  // work of a butterfly
    Stages(uint64_t n, const std::vector<int>& rad) : ns((uint32_t)rad.size()), lstr(0) {
        for (uint32_t s = 0; s < ns; s++) {
            r[s] = (uint32_t)rad[s];
            nr[s] = (uint32_t)n / r[s];
            w[s] = butterfly_ops(rad[s]) + 8.0 * rad[s];
            if (s + 1 < ns) lstr = std::max(lstr, r[s] * (nr[s] | 1u));
        }
        lstr |= 1u;
    }
};

// Relative rate of a tile shape, 1 at best; 0 where it does not fit `budget`, or
// needs a second buffer and may not (pp) have one.  Fitted to 8 Mi-point passes of
// 15 lengths from 60 to 7680 points, f32 and f64, contiguous and strided,
// over every thread count: the best contiguous shapes are one to a few lines
// in 64 to 256 threads (1080 points: 1 line, 128 threads 28.5 us; 4 lines,
// 512 threads 33.3 us; 576 threads 45 us), since a barrier then holds up few
// waves; more than 256 threads cost 10 to 30 %, most where they are not a
// multiple of the four SIMDs' waves.
static double shape_score(int arith, const Stages& st, uint32_t lpw, uint32_t nt, uint64_t lines, bool lf, size_t budget,
                          bool pp, bool real) {
    const size_t es = arith == P_F32 ? 8 : 16;
    // share of the launched lanes' butterfly slots that do work
    double useful = 0, slots = 0;
    bool second = false;
    for (uint32_t s = 0; s < st.ns; s++) {
        const uint32_t total = lpw * st.nr[s], need = (total + nt - 1) / nt, nb = nb_for((int)st.r[s], need);
        const uint32_t rounds = (total + nt * nb - 1) / (nt * nb);
        second |= needs_second(real, s, st.ns, need, nb);
        useful += st.w[s] * total;
        slots += st.w[s] * rounds * nb * nt;
    }
    const size_t lds = (size_t)(second ? 2 : 1) * lpw * st.lstr * es;
    if (lds > budget || (second && !pp)) return 0;
    double score = useful / slots;
    score *= thread_score(nt);
    // threads resident on a CU hide the barriers and the memory latency of one
    // another (82 registers in f32, 128 to 158 in f64)
    const double reg_threads = arith == P_F32 ? 1280 : 1024;
    const double wgs_cu = std::floor(std::min((double)kLdsBudget / (double)lds, std::max(1.0, reg_threads / nt)));
    score *= std::sqrt(std::min(1.0, wgs_cu * nt / 1024.0));
    // strided sides: the row segment of a tile; neighbouring tiles run on the
    // same XCD and share what is left of a line through its L2
    if (lf) {
        const size_t seg = lpw * es;
        score *= seg >= 128 ? 1.0 : seg >= 64 ? 0.97 : seg >= 32 ? 0.9 : seg >= 16 ? 0.7 : 0.4;
    }
    return score * fill_score(lines, lpw);
}

static double best_shape(int arith, uint64_t n, const std::vector<int>& rad, uint64_t lines, bool ld_lf, bool st_lf,
                         size_t budget, uint32_t fixed_nt, uint32_t forced_lpw, bool pp, bool real, Mix* out,
                         uint32_t max_lpw = 64) {
    static const uint32_t threads[] = {64, 128, 192, 256, 320, 384, 448, 512, 640, 768, 1024};
    const bool lf = ld_lf || st_lf;
    const Stages st(n, rad);
    double best = -1;
    uint32_t best_lpw = 0, best_nt = 0;
    for (uint32_t nt : threads) {
        if ((fixed_nt && nt != fixed_nt) || thread_score(nt) <= best) continue;
        for (uint32_t lpw = forced_lpw ? forced_lpw : 1; lpw <= (forced_lpw ? forced_lpw : max_lpw);
             lpw = lf && !forced_lpw ? 2 * lpw : lpw + 1) {
            if ((lpw > lines && lpw > 1 && !forced_lpw) || (uint64_t)lpw * n > 0xFFFFu) break;
            // (more than two rounds of 16 points per thread, or under two
            // points: never the best shape)
            if (!fixed_nt && !forced_lpw && lpw > 1 && (uint64_t)lpw * n > 34ull * nt) break;
            if (!fixed_nt && !forced_lpw && nt > 64 && (uint64_t)lpw * n < 2ull * nt) continue;
            if (!forced_lpw && thread_score(nt) * fill_score(lines, lpw) <= best) break;  // nor any wider tile
            const double score = shape_score(arith, st, lpw, nt, lines, lf, budget, pp, real);
            if (score <= 0) break;
            if (score > best + 1e-9) {
                best = score;
                best_lpw = lpw;
                best_nt = nt;
            }
        }
    }
    if (out && best > 0) *out = shape(n, rad, best_lpw, best_nt, ld_lf, st_lf, real);
    return best;
}

static void multisets(uint64_t n, int max_r, double cost, std::vector<int>& cur, double& best,
                      std::vector<std::pair<double, std::vector<int>>>& out) {
    if (n == 1) {
        best = std::min(best, cost);
        out.emplace_back(cost, cur);
        return;
    }
    if (cur.size() >= (size_t)kMixStages) return;
    for (int r = max_r; r >= 2; r--) {
        if (n % (uint64_t)r) continue;
        const double c = cost + stage_cost(r);
        if (c > 1.3 * best) continue;
        cur.push_back(r);
        multisets(n / (uint64_t)r, r, c, cur, best, out);
        cur.pop_back();
    }
}

// The schedule of n: over the radix multisets within 30 % of the cheapest and
// their orders, the least work per point over the rate of its best contiguous
// tile (the fill of the threads decides between, for 1080 points, 15x9x8 at
// 45 us and 12x10x9 at 28 us per 8 Mi points).  The larger radix first where
// nothing else decides (12x9 23.9 us, 9x12 25.7 us).  It depends on
// the length alone: a line's result does not depend on the tile or on the
// number of lines.  (Radices 18 and 20 measured: 270 points 36 -> 33 us, 1000
// points 36 -> 38, 960-point half lines 4 % slower; not used.)
std::vector<int> mix_schedule(uint64_t n) {
    static std::mutex mu;
    static std::map<uint64_t, std::vector<int>> done;  // at most the smooth lengths up to 2^15
    if (n < 2 || n > 0x8000u) return {};
    {
        std::lock_guard<std::mutex> g(mu);
        auto f = done.find(n);
        if (f != done.end()) return f->second;
    }
    // (searched outside the lock: other threads build plans meanwhile, and two
    // that search one length find the same)
    std::vector<std::pair<double, std::vector<int>>> sets;
    std::vector<int> cur, best;
    double least = 1e30;
    multisets(n, 16, 0, cur, least, sets);
    std::stable_sort(sets.begin(), sets.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    double value = 1e30;
    for (auto& s : sets) {
        if (s.first > 1.3 * least || s.first >= value) continue;  // (a rate is at most 1)
        std::vector<int> r = s.second;
        std::sort(r.begin(), r.end());
        // The orders of one set differ in the LDS pitch (every stage but the last)
        // and in which stages must fit one round (every stage but the first and
        // the last): a rate holds for all orders with those two.
        double rate[17][17] = {};
        do {
            double& known = rate[r.front()][r.back()];
            if (!known) {
                known = r.size() < 2 ? 1.0
                                     : best_shape(P_F32, n, r, 1u << 30, false, false, kLdsBudget, 0, 0, false, false,
                                                  nullptr);
                if (known <= 0) known = 1e-3;
            }
            const double v = s.first / known * (r.front() < r.back() ? 1.02 : 1.0) * (r.front() < r[r.size() > 1] ? 1.01 : 1.0);
            if (v < value) {
                value = v;
                best = r;
            }
        } while (std::next_permutation(r.begin(), r.end()));
    }
    std::lock_guard<std::mutex> g(mu);
    done[n] = best;
    return best;
}

bool mix_plan(int arith, uint64_t n, uint64_t lines, bool ld_lf, bool st_lf, size_t budget, uint32_t fixed_nt,
              uint32_t forced_lpw, bool real, Mix* out) {
    const std::vector<int> rad = mix_schedule(n);
    if (rad.size() < 2 || !lines) return false;
    // batched tiles: the launch's LDS is its largest tile's, so half the
    // budget (four workgroups per CU) where the line fits it; a second buffer
    // (several rounds per middle stage) only where nothing else does
    for (int pp = 0; pp < 2; pp++)
        for (size_t b : {fixed_nt ? budget / 2 : budget, budget})
            if (best_shape(arith, n, rad, lines, ld_lf, st_lf, b, fixed_nt, forced_lpw, pp, real, out) > 0) {
                const uint64_t es = arith == P_F32 ? 8 : 16;
                out->stream = lines * n * es >= (32u << 20) && (ld_lf ? out->lpw * es >= 128 : out->st[0].nr * es >= 192);
                return true;
            }
    return false;
}

size_t mix_conv_lds_bytes(int arith, const MixConv& x) {
    // two more elements per line: Rader's x[0] and its sum of inputs
    return mix_lds_bytes(arith, x.f) + 2 * (size_t)x.f.lpw * (arith == P_F32 ? 8 : 16);
}

bool mix_conv_plan(int arith, uint64_t m, uint64_t lines, bool ld_lf, bool st_lf, size_t budget, uint32_t fixed_nt,
                   MixConv* out) {
    const std::vector<int> rad = mix_schedule(m);
    if (rad.size() < 2 || !lines) return false;
    const std::vector<int> rev(rad.rbegin(), rad.rend());
    // Few lines: a tile crosses LDS some ten times, and a wave with many short
    // lines only waits longer at each.  Short of two workgroups per CU a tile
    // takes the lines whose butterflies are one a thread of a wave, not more (300
    // lines of 41 points: 10.1 us at 24 lines, f64 64 lines of 74 points 11.6 at 5
    // and 10.0 at 1).  Batched tiles share the chip with other transforms'.
    const uint64_t fill = lines / (2ull * device_cu_count());
    const uint64_t wave = 64 * (uint64_t)*std::min_element(rad.begin(), rad.end()) / m;
    const uint32_t max_lpw =
        fixed_nt ? 64 : (uint32_t)std::min<uint64_t>(64, std::max<uint64_t>({1, fill, wave}));
    for (int pp = 0; pp < 2; pp++)
        for (size_t b : {fixed_nt ? budget / 2 : budget, budget}) {
            Mix f;
            // (the two extra elements per line fit what a pitch above m leaves)
            if (best_shape(arith, m, rad, lines, ld_lf, st_lf, b - 2048, fixed_nt, 0, pp, true, &f, max_lpw) <= 0) continue;
            Mix r = shape(m, rev, f.lpw, f.nt, ld_lf, st_lf, true);
            if (r.pp && !pp) continue;
            f.lstr = r.lstr = std::max(f.lstr, r.lstr);
            f.pp = r.pp = f.pp || r.pp ? f.lpw * f.lstr : 0;
            out->f = f;
            out->r = r;
            if (mix_conv_lds_bytes(arith, *out) <= budget) return true;
        }
    return false;
}

}  // namespace mifft
