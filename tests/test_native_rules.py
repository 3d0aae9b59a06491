"""Host side of the kernels' integer and selection arithmetic, in programs compiled against the library's headers."""
import native


def test_digits_of_a_secondary_node(tmp_path):
    """divide_digit, which splits a secondary node's index into its digits with a float quotient: exact for every value
    below 2^32 where those from kFloatDigits on are divided as integers, whatever the last bit of the reciprocal (v_rcp_f32: one ulp)."""
    lines = native.run(tmp_path, r"""
#include "pairs.hpp"
#include <cmath>
#include <cstdio>
#include <random>
int main()
{
    std::mt19937_64 g(1);
    long bad = 0;
    auto check = [&](uint32_t x, uint32_t d) {
        const float inv = 1.0f / (float)d;
        for (float f : {inv, std::nextafterf(inv, 0.0f), std::nextafterf(inv, 1e30f)}) {
            uint32_t r = x;
            const uint32_t q = ccoil::divide_digit(r, d, f, x >= ccoil::kFloatDigits);
            if (q != x / d || r != x % d) ++bad;
        }
    };
    const uint32_t ds[] = {1, 2, 3, 7, 14, 59, 80, 99, 100, 1600, 5900, 8000, 65535, 100000, 4194303, 16777217, 21474836, 2147483647u};
    for (uint32_t d : ds) {
        for (uint32_t x = 0; x < 20000; ++x) check(x, d);
        for (int k = 0; k < 200000; ++k) check((uint32_t)(g() >> (32 + g() % 20)), d);
        for (uint64_t m = d; m < (1ull << 32); m += std::max<uint64_t>(d, ((1ull << 32) - 1) / 5000 / d * d + d))
            for (int e = -1; e <= 1; ++e) check((uint32_t)(m + e), d);
    }
    std::printf("%ld\n", bad);
}
""")
    assert lines == ["0"]


def test_targets_that_the_pair_tuner_times(tmp_path):
    """tune_pairs times the rule's own target, whatever it is, and its neighbours down to 16 reduced-rule (256 planned)
    nodes a lane; a file's entry for the same batch whose target counted planned nodes is not replayed."""
    lines = native.run(tmp_path, r"""
#include "context.hpp"
#include <cstdio>
int main()
{
    ccoil_ctx_s ctx;
    ctx.cu_count = 256;
    for (int32_t precision : {(int32_t)CCOIL_FP64, (int32_t)CCOIL_FP32C})
        for (int64_t target : {16, 64, 128, 256, 2048}) {
            if (precision != CCOIL_FP64 && target < 256) continue;
            ccoil::PairBuild rule;
            rule.sorted.resize(3);
            rule.node_pairs = 1000 * target;
            rule.target = target;
            ctx.tuning["pairs n=3 node_pairs=" + std::to_string(rule.node_pairs) + " what=1 precision=0 cu=256"] = "target=8192";
            int64_t got = 0;
            std::printf("%d %lld:", precision, (long long)target);
            ccoil::tune_pairs(&ctx, rule, 1, precision, [](int64_t c, double &ms) {
                std::printf(" %lld", (long long)c);
                ms = 1.0;
                return (ccoil_status)CCOIL_OK;
            }, got);
            std::printf("\n");
        }
}
""")
    assert lines == ["0 16: 16 32", "0 64: 16 32 64 128", "0 128: 32 64 128 256", "0 256: 64 128 256 512",
                     "0 2048: 512 1024 2048 4096", "1 256: 256 512", "1 2048: 512 1024 2048 4096"]


def test_class_thresholds(tmp_path):
    """Each reduced class starts at or beyond its eta (its ellipse), and at most 1e-4 (2e-4) beyond."""
    lines = native.run(tmp_path, r"""
#include "context.hpp"
#include <cmath>
#include <cstdio>
using namespace ccoil;
// the least float >= 0 whose class, by of(x), is at least cls
template <typename F> float least(F of, int cls)
{
    float lo = 0.0f, hi = 1e4f;
    while (std::nextafterf(lo, hi) < hi) {
        const float m = 0.5f * (lo + hi);
        (of(m) >= cls ? hi : lo) = m;
    }
    return hi;
}
int main()
{
    CoilDev c = {};
    c.red_x = 0.0f;
    c.red_s = 0.0f;
    // class 1 starts where the coil's own rule has converged (red_x)
    for (int k = 2; k <= kRedAng; ++k)
        std::printf("%.9g\n", (double)least([&](float x) { return class_of(c, x, 1.0f, 0.0f) / (kRedThk + 1); }, k) / (std::cosh(kRedFrom[k - 1]) - 1.0));
    for (int t = 2; t <= kRedThk; ++t)
        std::printf("%.9g\n", (double)least([&](float x) { return class_of(c, 0.0f, 1.0f, x) % (kRedThk + 1); }, t) /
                                  (2.0 * std::cosh(std::log(kRedThkC / kRedTol) / (2 * kRedThkN[t - 1]))));
    for (int n = 1; n <= kMaxOrder; ++n) {   // and no coil's own threshold lies below its first class's
        CoilDev d = {};
        d.R = 0.1;
        d.a = 0.1;
        d.n_ang = d.n_thk = n;
        set_rule_limits(d);
        const int k = std::isnan(d.red_x) ? 0 : class_of(d, d.red_x, 1.0f, 0.0f) / (kRedThk + 1);
        if (k > 0 && d.red_x < std::cosh(kRedFrom[k - 1]) - 1.0) std::printf("n_ang %d\n", n);
    }
}
""")
    ratios = [float(v) for v in lines]
    assert len(ratios) == 10 and min(ratios) >= 1.0 and max(ratios[:5]) <= 1.0001 and max(ratios[5:]) <= 1.0002, lines


def test_angular_classes_errors(tmp_path):
    """The reduced angular sums of a ring's A, B and gradient terms, from where class_of takes each class on: within 2e-16 of
    the sum of the terms' magnitudes, the rule's own error, plus the tables' rounding (half an ulp of each weight and of
    each 1 - cos(phi), to the power 5/2: 3.5 x 1.1e-16, as if all had one sign)."""
    lines = native.run(tmp_path, r"""
#include "context.hpp"
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>
using namespace ccoil;
typedef long double ld;
struct Rule { std::vector<ld> s, w; };   // 1 - cos(phi), weights
// the terms of a ring of radius 1 at (r, z): A_phi, B_r, B_z and their derivatives' (integrands.hpp)
void sums(const Rule &q, ld r, ld z, ld *v, ld *m)
{
    std::fill(v, v + 8, 0.0L);
    std::fill(m, m + 8, 0.0L);
    for (size_t i = 0; i < q.s.size(); ++i) {
        const ld s = q.s[i], c = 1 - s, D = (1 - r) * (1 - r) + z * z + 2 * r * s, f = 1 / sqrtl(D), f3 = f / D, f5 = f3 / D;
        const ld nb = 1 - r + r * s, nr = r - 1 + s;
        const ld t[8] = {c * f, z * c * f3, nb * f3, z * nb * f5, z * c * nr * f5, c * f3 - 3 * z * z * c * f5, nb * nr * f5, c * f3};
        for (int k = 0; k < 8; ++k) {
            v[k] += q.w[i] * t[k];
            m[k] += q.w[i] * fabsl(t[k]);
        }
    }
}
int main()
{
    RedTables t;
    reduced_tables(t);
    CoilDev c = {};
    c.red_x = red_limits().x[0];
    for (int k = 0, off = 0; k < kRedAng; off += kRedAngN[k++]) {
        Rule q;
        for (int i = 0; i < kRedAngN[k]; ++i) {
            q.s.push_back(t.omc[off + i]);
            q.w.push_back(t.w[off + i]);
        }
        ld worst = 0;
        int seen = 0;
        for (int e = 0; e <= 120; ++e) {
            const ld eta = (ld)kRedEta[k] * (1 + 0.001L * e), x = coshl(eta) - 1;
            if (class_of(c, (float)x, 1.0f, 0.0f) / (kRedThk + 1) != k + 1) continue;
            ++seen;
            Rule fine;
            const int n = (int)(60 / eta) + 40;   // midpoints, which err like exp(-2 n eta)
            for (int i = 0; i < n; ++i) {
                const ld h = sinl(1.57079632679489661923132169163975L * (i + 0.5L) / n);
                fine.s.push_back(2 * h * h);
                fine.w.push_back(2.0L / n);
            }
            const ld lo = 1 + x - sqrtl((1 + x) * (1 + x) - 1);   // the radii with this eta: lo to 1 / lo
            for (int j = 0; j < 60; ++j) {
                const ld r = powl(lo, cosl(3.14159265358979L * j / 59));
                const ld z = sqrtl(std::max(2 * r * x - (1 - r) * (1 - r), 0.0L));
                ld a[8], am[8], b[8], bm[8];
                sums(q, r, z, a, am);
                sums(fine, r, z, b, bm);
                for (int i = 0; i < 8; ++i)
                    if (bm[i] > 0) worst = std::max(worst, fabsl(a[i] - b[i]) / bm[i]);
            }
        }
        std::printf("%d %d %.3Lg\n", kRedAngN[k], seen, worst);
    }
}
""")
    for line in lines:
        n, seen, err = line.split()
        assert int(seen) > 80 and float(err) <= 2e-16 + 3.5 * 1.11e-16, lines


def test_classes_of_long_thin_coils(tmp_path):
    """rule_class never takes a cheaper rule than the geometry in double gives with the thresholds lowered by class_of's
    float rounding: 3e-7 of the outer radius against a (ellipse), 1e-5 (angular). Points about the winding's end."""
    lines = native.run(tmp_path, r"""
#include "context.hpp"
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
using namespace ccoil;
int main()
{
    std::mt19937_64 g(7);
    std::uniform_real_distribution<double> u(0, 1);
    for (double a : {1e-3, 1e-2, 0.5})
        for (double hb : {0.3, 700.1, 5000.3}) {
            CoilDev c = {};
            c.R = 1.0;
            c.a = a;
            c.b = 2 * hb;
            c.use_fast = 1;
            c.n_ang = 60;
            c.n_thk = 30;
            set_rule_limits(c);
            long bad = 0, reduced = 0;
            for (int i = 0; i < 100000; ++i) {
                const double far = i % 2 ? a : 2.0, z = hb + far * (4 * u(g) - 1), r = std::fabs(1 + 0.5 * a + far * (4 * u(g) - 2));
                const double zd = std::max(std::fabs(z) - hb, 0.0), rho = std::min(std::max(std::hypot(r, zd), 1.0), 1 + a);
                const double num = (rho - r) * (rho - r) + zd * zd, den = 2 * rho * r;
                const double s = (std::hypot(r - 1, zd) + std::hypot(r - 1 - a, zd)) * 2 / a;
                const int got = rule_class(c, z, r);
                const int most = class_of(c, (float)(num * (1 + 1e-5)), (float)den, (float)(s * (1 + 3e-7 * (1 + a) / a)));
                if (got / (kRedThk + 1) > most / (kRedThk + 1) || got % (kRedThk + 1) > most % (kRedThk + 1)) ++bad;
                if (got) ++reduced;
            }
            std::printf("%g %g %ld %d\n", a, hb, bad, reduced > 50000);
        }
}
""")
    assert len(lines) == 9 and all(line.split()[2:] == ["0", "1"] for line in lines), lines
