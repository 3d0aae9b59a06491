// Reduced rules: fewer nodes for a rule's sum where it has converged to rounding (host tables and thresholds).
//
// A coil's field rule is a Gauss-Legendre sum over the angle phi in [0, pi] (n_ang nodes) times one over the thickness
// (n_thk nodes). Away from the winding both integrands are analytic far into the complex plane, the rule's value is
// the integral's to rounding, and so is any other rule's with enough nodes: the angular sum takes 6 to 20 nodes
// where the planned rule has up to 80, the thickness sum 6 to 22. The integrands, and so their conditioning, stay as
// they are. Pairs too close to the winding keep the coil's own rule, whose own error is then part of the result.
//
// Angular. The squared distance from the point (r, z) to the ring element at phi, (rho - r)^2 + z^2 +
// 2 rho r (1 - cos phi), vanishes at phi = +-i eta with cosh(eta) = 1 + ((rho - r)^2 + z^2) / (2 rho r). With
// phi = pi - 2 am(u, k), k' = tanh(eta / 2), the integrand is analytic and 2 K periodic in the strip |Im u| < K'(k)
// for every point whose eta is at least that one, so the N-point midpoint rule in u errs like exp(-2 pi N K' / K): 20
// nodes at eta = 0.1 where Gauss-Legendre takes 80. (k', nodes and weights from the arithmetic-geometric mean and
// Landen's descending transformation, Abramowitz & Stegun 16.4 and 17.6.) Where the singularity is one of the fifth power
// of the distance, the gradient's, that holds a little inside the strip only: in extended precision, over the ring's
// positions at each eta, A and B have errors below 1e-17 of the sum of the node terms' magnitudes at every class's eta, the
// gradient 2.8e-15 at eta = 0.1 (20 nodes), 8.0e-16 at 1.0 (10) and below 2e-16 at the others, falling to 1.9e-16 from
// 0.103 and to 1.1e-16 from 1.01 on, where those two classes begin (kRedFrom). So: at most 2e-16 for A, B and the
// gradient, and less over the sheets, whose ends alone have the ring's terms.
//
// Thickness. The angular sum as a function of the ring radius is singular at rho = r +- i zd (zd: the distance beyond
// the axial span), so n Gauss-Legendre nodes err like C rho_B^(-2n), rho_B the parameter of the Bernstein ellipse
// about [R, R + a] through that point. Measured: C between 3 and 47 for n = 2..30; 200 is used.
//
// The coil's own angular rule counts as converged where 1000 exp(2 eta) rho_B^(-2 n_ang) <= 1e-15 (the constant as in
// the far-field bound, exp(2 eta) for the node terms that cancel far from the coil), its thickness rule where
// 200 rho_B^(-2 n_thk) <= 1e-15.
#include "context.hpp"
#include "multipole.hpp"

#include <algorithm>
#include <array>
#include <cfloat>
#include <cmath>
#include <limits>
#include <complex>

namespace ccoil {

namespace {

// No measure of a point reaches it, also none that overflowed.
constexpr float kNever = std::numeric_limits<float>::quiet_NaN();


typedef long double ld;

const ld kPiL = 3.14159265358979323846264338327950288L;

// sn, cn, dn of u for the complementary modulus kp in (0, 1): Landen's descending transformation.
void jacobi(ld u, ld kp, ld &sn, ld &cn, ld &dn)
{
    ld a[32], c[32], b = kp;
    a[0] = 1.0L;
    c[0] = sqrtl(1.0L - kp * kp);
    int n = 0;
    while (fabsl(c[n]) > 1e-20L && n < 30) {
        a[n + 1] = 0.5L * (a[n] + b);
        c[n + 1] = 0.5L * (a[n] - b);
        b = sqrtl(a[n] * b);
        ++n;
    }
    ld phi = ldexpl(a[n] * u, n);
    for (int i = n; i > 0; --i) phi = 0.5L * (phi + asinl(c[i] / a[i] * sinl(phi)));
    sn = sinl(phi);
    cn = cosl(phi);
    dn = sqrtl(cn * cn + kp * kp * sn * sn);
}

ld complete_k(ld kp)
{
    ld a = 1.0L, b = kp;
    while (fabsl(a - b) > 1e-19L * a) {
        const ld m = 0.5L * (a + b);
        b = sqrtl(a * b);
        a = m;
    }
    return kPiL / (a + b);
}

// ln of the Gauss-Legendre ellipse parameter of the angular singularity at phi = i eta.
double log_ellipse(double eta)
{
    const std::complex<double> xs(-1.0, 2.0 * eta / kPi), sq = std::sqrt(xs * xs - 1.0);
    return std::log(std::max(std::abs(xs + sq), std::abs(xs - sq)));
}

// Least cosh(eta) - 1 at which the n-node angular rule may be replaced (kNever: never).
float ang_threshold(int n)
{
    int first = 0;
    while (first < kRedAng && kRedAngN[first] >= n) ++first;
    if (first == kRedAng) return kNever;
    auto g = [&](double eta) { return std::log(1000.0 / 1e-15) + 2.0 * eta - 2.0 * n * log_ellipse(eta); };
    double lo = kRedFrom[first], hi = 20.0;
    if (g(lo) > 0.0) {
        if (g(hi) > 0.0) return kNever;
        for (int it = 0; it < 60; ++it) {
            const double m = 0.5 * (lo + hi);
            (g(m) > 0.0 ? lo : hi) = m;
        }
        lo = hi;
    }
    return (float)((std::cosh(lo) - 1.0) * (1.0 + 1e-5));
}

// Least ellipse distance sum at which the n-node thickness rule may be replaced (kNever: never).
float thk_threshold(int n)
{
    int first = 0;
    while (first < kRedThk && kRedThkN[first] >= n) ++first;
    if (first == kRedThk) return kNever;
    const double own = std::log(kRedThkC / 1e-15) / (2.0 * n), red = std::log(kRedThkC / kRedTol) / (2.0 * kRedThkN[first]);
    return (float)(2.0 * std::cosh(std::max(own, red)) * (1.0 + 1e-4));
}

struct Thresholds {
    std::array<float, kMaxOrder + 1> ang{}, thk{};
    Thresholds()
    {
        for (int n = 1; n <= kMaxOrder; ++n) {
            ang[(size_t)n] = ang_threshold(n);
            thk[(size_t)n] = thk_threshold(n);
        }
    }
};

}  // namespace

void set_rule_limits(CoilDev &c)
{
    static const Thresholds t;
    // The classes are found in float, to some 1e-7 of the winding's radius and the point's distance from its span: that
    // must not overflow nor underflow when squared, and be small against R (angular) and against a (thickness: 1e-3 of it
    // at the least a, a tenth more of an error that the constant 200 overstates by four). A point's own coordinate z is
    // good to 1e-16 of a coil's half length, and so is the distance: 1e-8 of the least a at the greatest length.
    const bool fits = c.R >= 1e-15 && c.R + c.a <= 1e15 && (!c.use_fast || 0.5 * c.b <= 1e4 * c.R);
    c.red_x = fits ? t.ang[(size_t)c.n_ang] : kNever;
    c.red_s = fits && c.a >= 1e-4 * (c.R + c.a) ? t.thk[(size_t)c.n_thk] : kNever;
    c.r0f = (float)c.R;
    c.r1f = (float)(c.R + c.a);
    c.hb = c.use_fast ? 0.5 * c.b : 0.0;
    c.ia2f = c.red_s < FLT_MAX ? (float)(2.0 / c.a) : 0.0f;
}

int64_t rule_nodes_beyond(const CoilDev &c, double dist)
{
    // every ring element lies within rmax of the centre, so a point at D >= dist is at least gap = D - rmax from it,
    // and r rho <= D (R + a)
    const double gap = dist - c.rmax;
    if (!(gap > 0.0)) return (int64_t)c.n_ang * c.n_thk;
    const RuleSel s = class_rule(c, class_of(c, (float)(gap * gap), (float)(2.0 * dist * (c.R + c.a)),
                                             (float)(2.0 * gap) * c.ia2f));
    return (int64_t)s.na * s.nt;
}

std::vector<double> legendre_rows()
{
    std::vector<double> v(4 * kMpOdd + kMpLegK);
    std::vector<ld> k(kMpLegK + 1, 1.0L);   // the leading coefficient of P_n
    for (int n = 0; n < kMpLegK; ++n) {
        v[(size_t)(4 * kMpOdd + n)] = (double)k[(size_t)n];
        k[(size_t)n + 1] = k[(size_t)n] * (2 * n + 1) / (n + 1);
    }
    for (int i = 0; i < kMpOdd; ++i)
        for (int h = 0; h < 2; ++h) {
            const int n = 2 * i + 3 + h;
            v[(size_t)(4 * i + 2 * h)] = (double)((ld)n * n / (4.0L * n * n - 1.0L));
            v[(size_t)(4 * i + 2 * h + 1)] = (double)((2 * n + 1) * k[(size_t)n]);
        }
    return v;
}

void reduced_tables(RedTables &t)
{
    int e = 0;
    for (int k = 0; k < kRedAng; ++k) {
        const int n = kRedAngN[k];
        const ld kp = tanhl(0.5L * (ld)kRedEta[k]), K = complete_k(kp);
        for (int i = 0; i < n; ++i, ++e) {
            ld sn, cn, dn;
            jacobi(K * (i + 0.5L) / n, kp, sn, cn, dn);
            const ld s = 2.0L * cn * cn, c = 1.0L - s, w = 4.0L * K * dn / (kPiL * n);   // 1 - cos(phi), cos(phi)
            t.w[e] = (double)w;
            t.omc[e] = (double)s;
            t.opc[e] = (double)(2.0L * sn * sn);
            t.wcos[e] = (double)(w * c);
            t.ws[e] = (double)(w * s);
            t.ws2[e] = (double)(w * s * s);
            t.wcs[e] = (double)(w * c * s);
        }
    }
}

}  // namespace ccoil
