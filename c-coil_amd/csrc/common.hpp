// Device-side data layout shared by the field, pair and table kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ccoil {

constexpr int kMaxOrder = 100;                        // Legendre::maxLegendreOrder (LegendreMatrix.h:9)
constexpr int kTableSize = kMaxOrder * (kMaxOrder + 1) / 2;

// Reduced rules: the node sets that replace a rule's Gauss-Legendre angular or thickness sum where that sum has
// converged to rounding (reduced_rules.cpp: the bounds, the tables and what they measured).
//
// Angular class k (1..kRedAng) serves the pairs whose angular integrand is analytic in the strip |Im phi| < eta for an
// eta of at least kRedFrom[k - 1]; its kRedAngN[k - 1] nodes, made for the strip of kRedEta[k - 1], lie in the angular
// double tables at kRedOffset. Class 0 is the coil's own rule.
constexpr int kRedAng = 6;
constexpr int kRedAngN[kRedAng] = {20, 16, 12, 10, 8, 6};
constexpr double kRedEta[kRedAng] = {0.1, 0.3, 0.75, 1.0, 1.8, 3.2};
constexpr double kRedFrom[kRedAng] = {0.103, 0.3, 0.75, 1.01, 1.8, 3.2};
constexpr int kRedNodes = 20 + 16 + 12 + 10 + 8 + 6;
constexpr int kRedOffset = kTableSize;
constexpr int kTableSizeAng = kRedOffset + kRedNodes;   // the w, omc, wcos, opc, ws, ws2 and wcs tables
// Thickness class t (1..kRedThk): the Gauss-Legendre rule of kRedThkN[t - 1] nodes, for points outside the ellipse with
// foci at the winding's inner and outer radius whose parameter is (kRedThkC / kRedTol)^(1 / (2 n)). Class 0 is the
// coil's own rule.
constexpr int kRedThk = 6;
constexpr int kRedThkN[kRedThk] = {22, 17, 13, 10, 8, 6};
constexpr double kRedThkC = 200.0;
constexpr double kRedTol = 3e-16;
// The classes' thresholds, as class_of compares them: the least cosh(eta) - 1 and the least rho_B + 1 / rho_B (the ellipse's
// distance sum over half the thickness), with margins far above the rounding of class_of's float operations.
struct RedLimits {
    float x[kRedAng], s[kRedThk];
};
constexpr double cosh_minus_1(double x)
{
    double t = 1.0, v = 0.0;
    for (int k = 2; k <= 60; k += 2) v += t *= x * x / (k * (k - 1));
    return v;
}
constexpr double natural_log(double y)   // y >= 1
{
    double k = 0.0, v = 0.0;
    for (; y >= 2.0; y *= 0.5) k += 1.0;
    const double u = (y - 1.0) / (y + 1.0);
    double p = 2.0 * u;
    for (int i = 1; i <= 79; i += 2, p *= u * u) v += p / i;
    return 0.69314718055994530942 * k + v;
}
constexpr RedLimits red_limits()
{
    RedLimits l = {};
    for (int i = 0; i < kRedAng; ++i) l.x[i] = (float)(cosh_minus_1(kRedFrom[i]) * 1.00001);
    for (int i = 0; i < kRedThk; ++i)
        l.s[i] = (float)(2.0 * (1.0 + cosh_minus_1(natural_log(kRedThkC / kRedTol) / (2 * kRedThkN[i]))) * 1.0001);
    return l;
}
constexpr int kRuleClasses = (kRedAng + 1) * (kRedThk + 1);   // class = (kRedThk + 1) angular class + thickness class
constexpr double kPi = 3.14159265358979323846;
constexpr double kMuReduced = 1e-7;                    // mu0 / (4 pi), g_MiReduced (CalculateFieldsFast.cxx:10)
constexpr double kGpuAxisRatio = 1e-5;                 // on-axis branch of the GPU gradient (FieldGGroup.cu:134)

__host__ __device__ inline int table_offset(int n) { return n * (n - 1) / 2; }

// One coil as the kernels see it (FP64). Indexed with a wave-uniform coil index, so every field access
// is a scalar (SMEM) load broadcast to the wave.
struct alignas(64) CoilDev {
    double pos[3];
    double T[9];      // local -> global, row-major
    double Tinv[9];   // global -> local
    double R, a, b;   // inner radius, thickness, length (clamped)
    double cf;        // constFactor of generateCoilData (SupportFunctions.cxx:169-172)
    double omega;     // 2 pi f (E = omega * A)
    double current;   // I
    double turns;     // N
    double near_w2;   // squared near-winding shell width
    double sa, ca, sb, cb;   // sin/cos of alpha (y-axis angle) and beta (z-axis angle)
    double om_a[3], om_b[3]; // T^T dT/dalpha and T^T dT/dbeta as axial vectors (Omega v = om x v)
    double cur_used;         // current the constFactor was formed with (1 for a zero-current coil)
    double adj_scale;        // I / cur_used: scales every adjoint term except d/dI
    double ni;               // N I: the coil's total current (J a b)
    double rmax;             // radius of the sphere about the centre that holds the winding, |(R + a, b / 2)|
    double far_d2;           // squared distance beyond which the far-field series replaces the rule (0: never)
    double inv_rmax2;        // 1 / rmax^2
    double hb;               // half the winding's length, 0 where the slow integrands take it for flat
    int32_t use_fast;
    int32_t n_ang, n_thk, n_len;
    int32_t blk_ang, blk_thk, blk_len;
    int32_t near_key; // FP32C near pass: the coil's place in the evaluation order (most nodes first)
    int32_t mp_terms; // highest order of the far-field series a pair of this call can use (0: no series)
    // Reduced rules: the least cosh(eta) - 1 and the least ellipse parameter sum (d1 + d2) / (a / 2) at which the
    // coil's angular and thickness rules may be replaced (NaN: never), and the winding's geometry in float (inner
    // and outer radius, 2 / a).
    float red_x, red_s;
    float r0f, r1f, ia2f;
};

// Gauss-Legendre tables for orders 1..100 at offset table_offset(n), generated in FP64 on the device (w and the double
// angular tables also hold the reduced rules at kRedOffset).
struct Tables {
    const double *x;      // nodes, ascending
    const double *w;      // weights
    const double *cosv;   // cos(pi/2 (1 + x))        (SupportFunctions.cxx:188)
    const double *omc;    // 1 - cos(pi/2 (1 + x)) = 2 sin^2(pi/4 (1 + x))
    const float *xf;
    const float *wf;
    const float *cosf;
    const float *omcf;
    const double *rcos;   // cos(pi (1 + x)): secondary ring nodes of the GPU pair rule (MInductance.cu:34)
    const double *rsin;   // sin(pi (1 + x))
    const double *wcos;   // w cos(pi/2 (1 + x)): the angular weight times the cosine
    const float *wcosf;
    const double *opc;    // 1 + cos(pi/2 (1 + x)) = 2 cos^2(pi/4 (1 + x))
    const float *opcf;
    const double *ws;     // w (1 - cos): the weight times the first and second power of s = 1 - cos
    const double *ws2;    // w (1 - cos)^2
    const double *wcs;    // w cos (1 - cos)
    const float *wcsf;
    const double *leg;    // the far-field series' Legendre coefficients (multipole.hpp)
};

// Quantity bits (mirror of the C ABI enum).
enum : uint32_t { Q_A = 1, Q_B = 2, Q_E = 4, Q_G = 8, Q_GJ = 16 };

// Local cylindrical results of one (coil, point): A_phi, B_rho, B_z and the four gradient terms of
// CalculateFieldsMethods.cxx:53-56 (RPhi, RR, RZ, ZZ).
struct Local {
    double A, Bh, Bz, RP, RR, RZ, ZZ;
};

struct Cart {
    double A[3], E[3], B[3], G[9];
};

__device__ inline void mat_vec(const double *M, const double *v, double *o)
{
    o[0] = M[0] * v[0] + M[1] * v[1] + M[2] * v[2];
    o[1] = M[3] * v[0] + M[4] * v[1] + M[5] * v[2];
    o[2] = M[6] * v[0] + M[7] * v[1] + M[8] * v[2];
}

// 1 / sqrt(x) for a finite positive normal x: v_rsq_f64's estimate (about 2^-23 relative) refined by two Newton steps
// on f(y) = 1 / y^2 - x, y <- y + (y / 2) (1 - x y^2), each of which squares the relative error; within an ulp or two
// of the exact value and a fixed sequence of operations, so the same in every kernel.
__device__ inline double rsqrt_newton(double x)
{
    double y = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const double e = fma(-(x * y), y, 1.0);
        y = fma(0.5 * y, e, y);
    }
    return y;
}

// Point -> coil-local cylindrical (z, r) and the azimuth's cos/sin (cos(atan2(y,x)) = x/r).
// Every operation is rounded on its own (no FMA contraction), so each kernel that classifies a (coil, point) pair
// with is_near gets bitwise the same z and r from the same inputs, whatever the inlining context.
__device__ inline void to_local(const CoilDev &c, double px, double py, double pz, double &z, double &r,
                                double &cph, double &sph)
{
#pragma clang fp contract(off)
    const double d[3] = {px - c.pos[0], py - c.pos[1], pz - c.pos[2]};
    const double *M = c.Tinv;   // written out here rather than through mat_vec, so the pragma covers it
    const double l[3] = {M[0] * d[0] + M[1] * d[1] + M[2] * d[2], M[3] * d[0] + M[4] * d[1] + M[5] * d[2],
                         M[6] * d[0] + M[7] * d[1] + M[8] * d[2]};
    z = l[2];
    const double r2 = l[0] * l[0] + l[1] * l[1];
    if (r2 >= 1e-200) {
        // r and 1 / r from one reciprocal square root (within about an ulp of the correctly rounded values)
        const double ir = rsqrt_newton(r2);
        r = r2 * ir;
        cph = l[0] * ir;
        sph = l[1] * ir;
    } else if (r2 > 0.0) {   // within 1e-100 of the axis: the IEEE operations, clear of the estimates' range limits
        r = sqrt(r2);
        cph = l[0] / r;
        sph = l[1] / r;
    } else {
        r = 0.0;
        cph = 1.0;
        sph = 0.0;
    }
}

// Local cylindrical -> global Cartesian, accumulated into out (CalculateFieldsMethods.cxx:16-19,
// :33-36, :58-83; FieldGGroup.cu:134-174 for the GPU on-axis threshold). With the radial unit vector e = (cph, sph, 0),
// the axis z and E = T e, n = T z, the local gradient is (RR - RP) e e^T + RP (I - z z^T) + RZ (e z^T + z e^T) + ZZ z z^T:
// its product with T needs E, n and one more vector, 31 operations where the two matrix products took 53.
__device__ inline void accumulate_global(const CoilDev &c, const Local &L, double r, double cph, double sph,
                                         uint32_t q, Cart &out)
{
    const double *T = c.T;
    if (q & (Q_A | Q_E)) {
        const double ac = L.A * cph, as = L.A * sph;
        for (int k = 0; k < 3; ++k) {
            const double g = T[3 * k + 1] * ac - T[3 * k] * as;
            if (q & Q_A) out.A[k] += g;
            if (q & Q_E) out.E[k] += c.omega * g;
        }
    }
    if (!(q & (Q_B | Q_G | Q_GJ))) return;
    double E[3];
    for (int k = 0; k < 3; ++k) E[k] = T[3 * k] * cph + T[3 * k + 1] * sph;
    if (q & Q_B)
        for (int k = 0; k < 3; ++k) out.B[k] += L.Bh * E[k] + L.Bz * T[3 * k + 2];
    if (q & (Q_G | Q_GJ)) {
        const bool axis = r <= kGpuAxisRatio * c.R;   // r / R <= 1e-5 without the division: diag(RR, RR, ZZ)
        const double RP = axis ? L.RR : L.RP, RZ = axis ? 0.0 : L.RZ, d = axis ? 0.0 : L.RR - L.RP;
        double w[3], v[3];   // T G = w e^T + RP T (I - z z^T) + v z^T
        for (int k = 0; k < 3; ++k) {
            w[k] = d * E[k] + RZ * T[3 * k + 2];
            v[k] = RZ * E[k] + L.ZZ * T[3 * k + 2];
        }
        if (q & Q_GJ) {
            // (T G) T^T
            for (int i = 0; i < 3; ++i)
                for (int j = 0; j < 3; ++j)
                    out.G[3 * i + j] += w[i] * E[j] + v[i] * T[3 * j + 2] +
                                        RP * (T[3 * i] * T[3 * j] + T[3 * i + 1] * T[3 * j + 1]);
        } else {
            for (int k = 0; k < 3; ++k) {
                out.G[3 * k] += w[k] * cph + RP * T[3 * k];
                out.G[3 * k + 1] += w[k] * sph + RP * T[3 * k + 1];
                out.G[3 * k + 2] += v[k];
            }
        }
    }
}

// Pairs that FP32C evaluates in FP64:
//  - the near-winding shell: distance from (r, z) to the cross-section rectangle [R, R+a] x [-b/2, b/2] below one
//    cross-section width (max(a, b), floored at 1e-3 R for filaments);
//  - with axis (outputs that divide by r: the gradient's hoop term B_rho / r, the pair gradient's A / r), the cone
//    and cylinder around the axis, r < 0.1 sqrt(r^2 + z^2 + R^2): the float angular sums of B_rho and A vanish like
//    r while their rounding does not.
constexpr double kAxisCone2 = 0.01;

// Whether the far-field series replaces the quadrature rule for a point at local (z, r). Rounded operation by
// operation, like to_local, so every kernel that classifies a pair gets the same answer.
__device__ inline bool is_far(const CoilDev &c, double z, double r)
{
#pragma clang fp contract(off)
    return c.far_d2 > 0.0 && r * r + z * z > c.far_d2;
}

__device__ inline bool is_near(const CoilDev &c, double z, double r, bool axis)
{
#pragma clang fp contract(off)
    double dr = fmax(fmax(c.R - r, r - (c.R + c.a)), 0.0);
    double dz = fmax(fabs(z) - 0.5 * c.b, 0.0);
    const double r2 = r * r;
    return dr * dr + dz * dz < c.near_w2 || (axis && r2 < kAxisCone2 * (r2 + z * z + c.R * c.R));
}

// The pairs of the FP32C near pass: near and not far (the far-field series is FP64 and exact on the axis).
__device__ inline bool near_pass_pair(const CoilDev &c, double z, double r, bool axis)
{
    return !is_far(c, z, r) && is_near(c, z, r, axis);
}

// The node sets of one evaluation: offset and count of its angular and thickness rules in the tables.
struct RuleSel {
    int oa, na, ot, nt;
};

__host__ __device__ inline RuleSel full_rule(const CoilDev &c)
{
    return {table_offset(c.n_ang), c.n_ang, table_offset(c.n_thk), c.n_thk};
}

__host__ __device__ inline RuleSel class_rule(const CoilDev &c, int cls)
{
    const int k = cls / (kRedThk + 1), t = cls - k * (kRedThk + 1);
    RuleSel s = full_rule(c);
    int off = kRedOffset;
#pragma unroll
    for (int i = 0; i < kRedAng; ++i) {
        if (k == i + 1) {
            s.oa = off;
            s.na = kRedAngN[i];
        }
        off += kRedAngN[i];
    }
#pragma unroll
    for (int i = 0; i < kRedThk; ++i)
        if (t == i + 1) {
            s.nt = kRedThkN[i];
            s.ot = table_offset(kRedThkN[i]);
        }
    return s;
}

// The class of the cheapest rule whose value at local (z, r) is that of the coil's own rule to rounding
// (reduced_rules.cpp). With zd the point's distance beyond the winding's axial span, the angular integrand of the
// ring at radius rho is analytic for |Im phi| < eta, cosh(eta) = 1 + ((rho - r)^2 + zd^2) / (2 rho r), least at the
// winding's radius nearest to sqrt(r^2 + zd^2); the thickness integrand is analytic outside the point (r, zd) and its
// mirror, whose ellipse about [R, R + a] has the distance sum d1 + d2. zd is formed in double (next to the end of a coil
// thousands of radii long float coordinates are as coarse as its thickness), and every other operation is a float
// operation rounded on its own, so every kernel gives a pair the same class; the thresholds (red_limits) carry margins
// for the rounding.
//
// class_of: the class at num = (rho - r)^2 + zd^2, den = 2 rho r and s = (d1 + d2) / (a / 2), or at bounds of them
// (num / den and s from below).
__host__ __device__ inline int class_of(const CoilDev &c, float num, float den, float s)
{
#pragma clang fp contract(off)
    constexpr RedLimits kLim = red_limits();
    int k = 0, t = 0;
    if (num >= c.red_x * den) {
        k = 1;   // red_x is at least the first class's threshold
#pragma unroll
        for (int i = 1; i < kRedAng; ++i) k += num >= kLim.x[i] * den ? 1 : 0;
    }
    if (s >= c.red_s) {
        t = 1;
#pragma unroll
        for (int i = 1; i < kRedThk; ++i) t += s >= kLim.s[i] ? 1 : 0;
    }
    return (kRedThk + 1) * k + t;
}
__host__ __device__ inline float class_sqrt(float x)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_sqrtf(x);   // within an ulp
#else
    return __builtin_sqrtf(x);
#endif
}
__host__ __device__ inline int rule_class(const CoilDev &c, double z, double r)
{
#pragma clang fp contract(off)
    const float rf = (float)r, zd = fmaxf((float)(fabs(z) - c.hb), 0.0f), zd2 = zd * zd;
    const float rho = fminf(fmaxf(class_sqrt(rf * rf + zd2), c.r0f), c.r1f);
    const float dr = rho - rf, num = dr * dr + zd2, den = 2.0f * rho * rf;
    const float e0 = rf - c.r0f, e1 = rf - c.r1f;
    const float s = (class_sqrt(e0 * e0 + zd2) + class_sqrt(e1 * e1 + zd2)) * c.ia2f;
    return class_of(c, num, den, s);
}

// Largest v over the wave for 0 <= v < 2^BITS (lanes not executing count as 0): its bits from the top, one ballot each.
template <int BITS> __device__ inline int wave_max_bits(int v)
{
    int m = 0;
#pragma unroll
    for (int b = 1 << (BITS - 1); b >= 1; b >>= 1)
        if (__ballot(v >= (m | b))) m |= b;
    return m;
}
// The cheapest rule class that serves every executing lane of the wave (cls: the lane's own).
__device__ inline int wave_rule_class(int cls)
{
    const int k = cls / (kRedThk + 1), t = cls - k * (kRedThk + 1);
    return (7 - wave_max_bits<3>(7 - k)) * (kRedThk + 1) + 7 - wave_max_bits<3>(7 - t);
}
static_assert(kRedAng < 8 && kRedThk < 8, "three bits each");

}  // namespace ccoil
