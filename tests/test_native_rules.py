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
    """Each reduced class starts at or beyond the eta (the ellipse) that its node set is made for, and at most 1e-4 (2e-4) beyond."""
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
        std::printf("%.9g\n", (double)least([&](float x) { return class_of(c, x, 1.0f, 0.0f) / (kRedThk + 1); }, k) / (std::cosh(kRedEta[k - 1]) - 1.0));
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
        if (k > 0 && d.red_x < std::cosh(kRedEta[k - 1]) - 1.0) std::printf("n_ang %d\n", n);
    }
}
""")
    ratios = [float(v) for v in lines]
    assert len(ratios) == 10 and min(ratios) >= 1.0 and max(ratios[:5]) <= 1.0001 and max(ratios[5:]) <= 1.0002, lines
