// Checks the tiles and schedules of mix_plan.cpp on the host: every field that
// the register-stage kernels (mix_kernels.hpp, mix_conv.hpp) take for granted.
// Prints one line per violation and a count of what was checked.
#include <complex>
#include <cstdio>
#include <set>

#include "mix_plan.cpp"
#include "mix_kernels.hpp"

namespace mifft {
uint32_t device_cu_count() { return 256; }
}  // namespace mifft
using namespace mifft;

static long g_bad = 0, g_tiles = 0;
#define EXPECT(c, ...)                 \
    do {                               \
        if (!(c) && g_bad++ < 20) {    \
            printf("%s: ", #c);        \
            printf(__VA_ARGS__);       \
            printf("\n");              \
        }                              \
    } while (0)

static bool smooth(uint64_t n) {
    for (uint64_t p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n == 1;
}

static bool compiled(uint32_t code) {
    switch (code) {
#define MIFFT_MIX_CASE(R, NB) case R + 32 * NB:
        MIFFT_MIX_RADICES(MIFFT_MIX_CASE)
#undef MIFFT_MIX_CASE
        return true;
    }
    return false;
}

// One tile.  lds_to_lds: which stages read and write LDS; natural: points that
// some step keeps in natural order (0: none).
static void check_tile(const char* what, const Mix& x, uint64_t n, uint32_t fixed_nt, bool every_stage, uint32_t natural) {
    g_tiles++;
    uint64_t prod = 1;
    EXPECT(x.ns >= 2 && x.ns <= (uint32_t)kMixStages && x.n == n, "%s n=%llu", what, (unsigned long long)n);
    EXPECT(x.nt % 64 == 0 && x.nt >= 64 && x.nt <= 1024 && (!fixed_nt || x.nt == fixed_nt), "%s n=%u nt=%u", what, x.n, x.nt);
    EXPECT((uint64_t)x.lpw * n <= 0xFFFF && (uint64_t)x.lpw * x.pairs <= 0xFFFF, "%s n=%u lpw=%u", what, x.n, x.lpw);
    EXPECT(natural <= x.lstr, "%s n=%u lstr=%u", what, x.n, x.lstr);
    EXPECT(x.pp == 0 || x.pp == x.lpw * x.lstr, "%s n=%u pp=%u", what, x.n, x.pp);
    for (uint32_t s = 0; s < x.ns; s++) {
        const MixStage& st = x.st[s];
        const uint32_t R = st.code & 31u, nb = st.code >> 5;
        EXPECT(compiled(st.code), "%s n=%u stage %u code %u", what, x.n, s, st.code);
        EXPECT(st.L == prod && st.nr * R == n, "%s n=%u stage %u", what, x.n, s);
        prod *= R;
        const bool inside = every_stage || (s > 0 && s + 1 < x.ns);
        EXPECT(x.pp || !inside || x.lpw * st.nr <= x.nt * nb, "%s n=%u lpw=%u nt=%u stage %u: one buffer, several rounds",
               what, x.n, x.lpw, x.nt, s);
        if (s + 1 < x.ns) EXPECT((R - 1) * st.nrp + st.nr <= x.lstr, "%s n=%u stage %u writes past the pitch", what, x.n, s);
        if (!s) continue;
        for (uint32_t j : {0u, st.nr / 2, st.nr - 1}) {
            const uint32_t kq = j / st.L, k = j % st.L, m = k / st.Lp, kk = k % st.Lp;
            const uint32_t a = m * st.nrp_prev + kq * st.Lp + kk + (R - 1) * st.rstep;
            EXPECT(a < x.lstr, "%s n=%u stage %u reads past the pitch", what, x.n, s);
        }
        // the multipliers of the divisions by nr, L and Lp
        for (uint32_t v : {0u, 1u, st.nr - 1, st.nr, x.lpw * st.nr - 1}) {
            const auto div = [](uint32_t a, uint32_t mag) { return mag ? (uint32_t)(((uint64_t)a * mag) >> 32) : a; };
            EXPECT(div(v, st.dnr) == v / st.nr && div(v, st.dL) == v / st.L && div(v, st.dLp) == v / st.Lp &&
                       div(v, x.dlpw) == v / x.lpw,
                   "%s n=%u stage %u divides %u", what, x.n, s, v);
        }
    }
    EXPECT(prod == n, "%s n=%u radices", what, x.n);
}

// A line through the stages at the addresses of the tile's fields.
static double run_line(const Mix& x) {
    using C = std::complex<double>;
    const uint32_t n = x.n;
    auto root = [](double t) { return std::polar(1.0, -2 * M_PI * t); };
    std::vector<C> in(n), out(n), lds(x.lstr);
    for (uint32_t i = 0; i < n; i++) in[i] = C(std::sin(1.0 + i * i % 97), std::cos(3.0 * i));
    for (uint32_t s = 0; s < x.ns; s++) {
        const MixStage& st = x.st[s];
        const uint32_t R = st.code & 31u;
        std::vector<C> next(x.lstr);
        for (uint32_t j = 0; j < st.nr; j++) {
            std::vector<C> w(R);
            const uint32_t kq = j / st.L, k = j % st.L, m = k / st.Lp, kk = k % st.Lp;
            for (uint32_t i = 0; i < R; i++)
                w[i] = s ? lds[m * st.nrp_prev + kq * st.Lp + kk + i * st.rstep] * root((double)k * i / (st.L * R))
                         : in[j + i * st.nr];
            for (uint32_t q = 0; q < R; q++) {
                C v = 0;
                for (uint32_t i = 0; i < R; i++) v += w[i] * root((double)(i * q % R) / R);
                if (s + 1 < x.ns) next[q * st.nrp + j] = v;
                else out[j + q * st.nr] = v;
            }
        }
        lds.swap(next);
    }
    double err = 0;
    for (uint32_t k = 0; k < n; k += n > 1000 ? 37 : 1) {
        C v = 0;
        for (uint32_t i = 0; i < n; i++) v += in[i] * root((double)((uint64_t)i * k % n) / n);
        err = std::max(err, std::abs(v - out[k]));
    }
    return err;
}

// The schedule over every order of every radix set: what mix_schedule finds by
// fewer evaluations.
static std::vector<int> every_order(uint64_t n) {
    std::vector<std::pair<double, std::vector<int>>> sets;
    std::vector<int> cur, best;
    double least = 1e30, value = 1e30;
    multisets(n, 16, 0, cur, least, sets);
    for (auto& s : sets) {
        if (s.first > 1.3 * least) continue;
        std::vector<int> r = s.second;
        std::sort(r.begin(), r.end());
        do {
            double score = r.size() < 2 ? 1.0
                                        : best_shape(P_F32, n, r, 1u << 30, false, false, kLdsBudget, 0, 0, false, false,
                                                     nullptr);
            if (score <= 0) score = 1e-3;
            const double v = s.first / score * (r.front() < r.back() ? 1.02 : 1.0) * (r.front() < r[r.size() > 1] ? 1.01 : 1.0);
            if (v < value) value = v, best = r;
        } while (std::next_permutation(r.begin(), r.end()));
    }
    return best;
}

int main() {
    long schedules = 0, lines_run = 0;
    for (uint64_t n = 2; n <= 0x8000; n++) {
        if (!smooth(n)) continue;
        const std::vector<int> rad = mix_schedule(n);
        schedules++;
        if (n <= 2048 || n % 1000 == 0) EXPECT(rad == every_order(n), "schedule of %llu", (unsigned long long)n);
        for (int arith : {P_F32, P_F64})
            for (uint32_t fixed : {0u, 256u})
                for (uint64_t lines : {1ull, 300ull, 40000ull})
                    for (int lay = 0; lay < 4; lay++) {
                        const bool ld = lay & 1, st = lay & 2;
                        const size_t budget = fixed ? kLdsBudget / 2 : kLdsBudget;
                        Mix x;
                        if (mix_plan(arith, n, lines, ld, st, budget, fixed, 0, false, &x)) {
                            check_tile("line", x, n, fixed, false, 0);
                            EXPECT(mix_lds_bytes(arith, x) <= budget, "line n=%u LDS", x.n);
                            if (arith == P_F32 && lines == 40000 && (n <= 300 || n % 500 == 0)) {
                                lines_run++;
                                const double e = run_line(x);
                                EXPECT(e < 1e-9 * n, "line n=%u lpw=%u: off by %g", x.n, x.lpw, e);
                            }
                        }
                        if (!lay && arith == P_F32 && mix_plan(arith, n, lines, false, false, budget, fixed, 0, true, &x)) {
                            check_tile("real", x, n, fixed, true, (uint32_t)n);
                            EXPECT(x.pairs == n / 2 + 1 && mix_lds_bytes(arith, x) <= budget, "real n=%u", x.n);
                        }
                        MixConv c;
                        // a convolution that the LDS-to-LDS form would fit (two buffers and
                        // two points) has a tile: no longer form of it is kept
                        const size_t es = arith == P_F32 ? 8 : 16;
                        if (n > 16 && (2 * (size_t)lds_line_stride((uint32_t)n) + 2) * es <= budget)
                            EXPECT(mix_conv_plan(arith, n, lines, ld, st, budget, fixed, &c), "conv n=%llu has no tile",
                                   (unsigned long long)n);
                        if (mix_conv_plan(arith, n, lines, ld, st, budget, fixed, &c)) {
                            // (Rader keeps p = n + 1 points in natural order)
                            check_tile("conv", c.f, n, fixed, true, (uint32_t)n + (n % 2 == 0));
                            check_tile("conv back", c.r, n, fixed, true, (uint32_t)n + (n % 2 == 0));
                            EXPECT(c.f.st[c.f.ns - 1].code == c.r.st[0].code, "conv n=%llu turn", (unsigned long long)n);
                            EXPECT(c.f.lpw == c.r.lpw && c.f.nt == c.r.nt && c.f.lstr == c.r.lstr && c.f.pp == c.r.pp,
                                   "conv n=%llu tiles differ", (unsigned long long)n);
                            EXPECT(mix_conv_lds_bytes(arith, c) <= budget, "conv n=%llu LDS", (unsigned long long)n);
                        }
                    }
    }
    printf("checked %ld schedules, %ld tiles, %ld lines\n", schedules, g_tiles, lines_run);
    return g_bad ? 1 : 0;
}
