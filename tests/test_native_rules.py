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
