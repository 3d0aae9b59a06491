// Far field of a coil as an exterior zonal-harmonic (axial multipole) series, in FP64.
//
// Outside the sphere that holds the coil's winding (radius r_max = |(R + a, b/2)| about its centre), the field of an
// axisymmetric azimuthal current is B = -mu0 grad Phi with Phi = sum_l M_l D^-(l+1) P_l(cos theta), D the distance
// from the centre and theta the angle from the axis. On the axis B_z of a loop of current I, radius rho, height z0
// is mu0 I rho^2 / (2 (rho^2 + (z - z0)^2)^(3/2)); expanding it in c / z (c^2 = rho^2 + z0^2) with the Gegenbauer
// generating function and matching mu0 sum_l (l + 1) M_l z^-(l+2) gives, for current spread over rings (rho, z0)
// with weights w_k summing to N I,
//   M_l = sum_k w_k rho_k^2 V_l(rho_k, z0_k) / (2 (l + 1)),   V_l = c^(l-1) P'_l(z0 / c).
// V_l is a polynomial (V_0 = 0, V_1 = 1, V_(l+1) = c^2 V_(l-1) + (2l + 1) U_l with the solid harmonics
// U_l = c^l P_l(z0 / c), U_(l+1) = ((2l + 1) z0 U_l - l c^2 U_(l-1)) / (l + 1)) of degree at most l - 1 in z0.
//
// The rings are the field rule's own: its thickness nodes (the rule's Gauss-Legendre nodes over [R, R + a], so the
// series reproduces the rule's thickness sum exactly, whatever its order), and over the length either the exact
// average (the fast rule integrates the length in closed form; dV_(l+1)/dz0 = (l + 2) V_l, as for all solid harmonics,
// so the average over |z0| <= h is V_(l+1)(h) / ((l + 2) h) for odd l) or the mid-plane alone (the slow rule's flat
// sheet: the limit h = 0). What the series leaves out is then the angular rule's own error
// and the truncation. With s = sin theta, u = 1 / D and q_l = (r_max / D)^(l+1), and the moments normalised as
// m_l = mu0 M_l / r_max^(l+1):
//   A_phi = s sum m_l q_l P'_l / l           B_z  = u sum (l + 1) m_l q_l P_(l+1)
//   B_rho = s u sum m_l q_l P'_(l+1)         B_rho / r = u^2 sum m_l q_l P'_(l+1)
//   dB_z/dz = -u^2 sum (l + 1)(l + 2) m_l q_l P_(l+2)
//   dB_rho/dz = dB_z/drho = -s u^2 sum (l + 1) m_l q_l P'_(l+2)
//   dB_rho/drho = -(B_rho / r + dB_z/dz)      (div B = 0)
// The host sets each coil's distance threshold (CoilDev::far_d2) where a bound on the angular rule's error falls
// below the tolerance of the arithmetic that uses the series.
#pragma once

#include "common.hpp"

namespace ccoil {

//
// The loops hold P_n as the monic polynomial p_n = P_n / k_n, k_n = (2n)! / (2^n n!^2), whose recurrence p_(n+1) =
// c p_n - n^2 / (4n^2 - 1) p_(n-1) has one coefficient, with k_n in the moments and in P'_(n+1) = P'_(n-1) + (2n + 1)
// k_n p_n. The moments of even order are zero, so a term holds one odd order l: q_l steps by (r_max / D)^2, and the
// eight numbers a term takes lie in two rows of 32 bytes, of the coil and of all coils, for two scalar loads a term.
// Bound by FP64 issue (70 % of it) with 15 instructions a term for B and gradient and some 190 around the loop; with 17
// instructions, and loads from seven arrays that the loop waited for five times in two terms, 128 coils x 2^20 points
// took 2.39 ms, this 2.00 in turn on one card, 2.1 to 2.3 on others (loads a term ahead, held there by scheduling
// barriers: the same).
constexpr int kMpTerms = 250;               // highest order l (below 256, the range of wave_max_small)
constexpr int kMpOdd = 128;                 // odd orders l = 2 i + 1 of the tables (a row more than is summed)
// Per coil: rows of m_l, (l + 1) m_l k_(l+1), (l + 1)(l + 2) m_l k_(l+2), (l + 1) m_l; then m_l / l.
constexpr int kMpCoil = 5 * kMpOdd;
// Tables::leg: rows of n^2 / (4n^2 - 1) and (2n + 1) k_n at n = l + 2 and at n = l + 3; then k_n, n < kMpLegK.
constexpr int kMpLegK = 2 * kMpOdd + 2;
static_assert(kMpTerms < 256 && kMpTerms + 2 < 2 * kMpOdd, "series orders and their arrays");
static_assert(4 * kMpOdd + kMpLegK <= kTableSizeAng, "Tables::leg is allocated with the angular tables");
// Every coil's winding is symmetric about its mid-plane (a slow-rule coil is a mid-plane sheet), so its moments of even
// order are zero and have no place in the tables.

// Number of terms for a point at distance D from a coil whose winding lies within r_max: the truncation falls like
// (r_max / D)^L with a constant below 2, so L = ln(2 / tol) / ln(D / r_max), between 4 and kMpTerms; log_tol =
// ln(2 / tol): kMpLogTolFP64 (tol = 1e-15, a hundredth of the FP64 rule's own error against the exact integral) or
// kMpLogTolFP32C (1e-13, far below the float rule's own rounding).
constexpr float kMpLogTolFP64 = 35.2319f;
constexpr float kMpLogTolFP32C = 30.6267f;
__device__ inline int multipole_terms(double D2, double inv_rmax2, float log_tol)
{
    // D^2 / r_max^2 > 1.17^2, a normal number: the bare logarithm (base 2) and reciprocal serve
    const float lg = __builtin_amdgcn_logf((float)(D2 * inv_rmax2));
    const int L = (int)(2.0f / 0.69314718f * log_tol * __builtin_amdgcn_rcpf(lg)) + 2;
    return L < 4 ? 4 : (L > kMpTerms ? kMpTerms : L);
}

// Largest v over the wave for 0 <= v < 256 (every lane active).
__device__ inline int wave_max_small(int v) { return wave_max_bits<8>(v); }

// Smallest v over the lanes with active set, for 0 <= v < 256 (every lane of the wave executing); 255 if none is.
__device__ inline int wave_min_small(int v, bool active)
{
    return 255 - wave_max_small(active ? 255 - v : 0);
}

// The rows of a term: mp, leg at the term's, ma at its m_l / l.
template <bool WA, bool WB>
struct MpTerm {
    double m, zk, zzk, mz, a, b0, k0, b1, k1;
    __device__ inline void load(const double *mp, const double *ma, const double *leg)
    {
        if (WA) a = ma[0];
        if (WB) {
            m = mp[0];
            zk = mp[1];
            zzk = mp[2];
            mz = mp[3];
        }
        b0 = leg[0];
        k0 = leg[1];
        b1 = leg[2];
        k1 = leg[3];
    }
};

// The series' sums at one point: SA = sum m_l q_l P'_l / l, SZ = sum (l + 1) m_l q_l P_(l+1), SB = sum m_l q_l P'_(l+1),
// SZZ = sum (l + 1)(l + 2) m_l q_l P_(l+2), SRZ = sum (l + 1) m_l q_l P'_(l+2); c = cos theta, qr = r_max / D. The loop
// runs L terms (wave-uniform), and terms beyond own add exact zeros, so the value is that of own terms. The first lo
// terms (the least own count among the lanes that call; wave-uniform) need no such test.
struct MpSums { double A, Z, B, ZZ, RZ; };
template <bool WA, bool WB, bool WG>
__device__ inline MpSums multipole_sums(const double *mp, const double *leg, double c, double qr, int L, int lo, int own)
{
    const double c2 = c * c, q2 = qr * qr;
    // p_(l+1), p_(l+2) and P'_l, P'_(l+1), P'_(l+2), from l = 1
    double p1 = c2 - 1.0 / 3.0, p2 = c * (c2 - 0.6);
    double d0 = 1.0, d1 = 3.0 * c, d2 = 1.5 * (5.0 * c2 - 1.0);
    double q = q2;   // q_l
    MpSums S = {0.0, 0.0, 0.0, 0.0, 0.0};
    MpTerm<WA, WB || WG> t0, t1;   // in turn: the term summed and the one loaded meanwhile
    const double *ma = mp + 4 * kMpOdd;
    t0.load(mp, ma, leg);
    auto add = [&](const MpTerm<WA, WB || WG> &t, MpTerm<WA, WB || WG> &next, double ql) {
        mp += 4;
        ma += 1;
        leg += 4;
        next.load(mp, ma, leg);
        if (WA) S.A = fma(t.a * ql, d0, S.A);
        if (WB || WG) {
            S.Z = fma(t.zk * ql, p1, S.Z);
            S.B = fma(t.m * ql, d1, S.B);
        }
        if (WG) {
            S.ZZ = fma(t.zzk * ql, p2, S.ZZ);
            S.RZ = fma(t.mz * ql, d2, S.RZ);
        }
        // p_(l+3), p_(l+4), P'_(l+3), P'_(l+4)
        const double p3 = fma(c, p2, -t.b0 * p1), d3 = fma(t.k0, p2, d1);
        const double p4 = fma(c, p3, -t.b1 * p2), d4 = fma(t.k1, p3, d2);
        d0 = d2;
        p1 = p3;
        p2 = p4;
        d1 = d3;
        d2 = d4;
        q *= q2;
    };
    int l = 1;
    for (; l + 2 <= lo; l += 4) {
        add(t0, t1, q);
        add(t1, t0, q);
    }
    for (; l <= L; l += 4) {
        add(t0, t1, l <= own ? q : 0.0);
        if (l + 2 > L) break;
        add(t1, t0, l + 2 <= own ? q : 0.0);
    }
    return S;
}

// Local (A_phi, B_rho, B_z, B_rho / r, dB_rho/drho, dB_rho/dz, dB_z/dz) of one coil at local (z, r) from its series
// (mp: the coil's kMpCoil doubles, leg: Tables::leg, rmax: the coil's r_max; L, lo, own: multipole_sums).
template <bool WA, bool WB, bool WG>
__device__ inline void eval_multipole(const double *mp, const double *leg, double rmax, double z, double r, int L,
                                      int lo, int own, Local &out)
{
    const double D2 = r * r + z * z;
    const double u = rsqrt_newton(D2);
    const double s = r * u;
    const MpSums S = multipole_sums<WA, WB, WG>(mp, leg, z * u, rmax * u, L, lo, own);
    out.A = s * S.A;
    out.Bz = u * S.Z;
    out.Bh = s * u * S.B;
    out.RP = u * u * S.B;
    out.ZZ = -u * u * S.ZZ;
    out.RZ = -s * u * u * S.RZ;
    out.RR = -(out.RP + out.ZZ);
}

// The pair kernel's view of the series at a secondary node: A_phi (WA), B_rho and B_z (WB), and A_phi / r = u sum
// m_l q_l P'_l / l (also on the axis, where it is the limit), for dA_phi/dr = B_z - A_phi / r.
template <bool WA, bool WB>
__device__ inline void eval_multipole_pair(const double *mp, const double *leg, double rmax, double z, double r, int L,
                                           int lo, int own, Local &out, double &a_over_r)
{
    const double D2 = r * r + z * z;
    const double u = rsqrt_newton(D2);
    const double s = r * u;
    const MpSums S = multipole_sums<WA, WB, false>(mp, leg, z * u, rmax * u, L, lo, own);
    out.A = s * S.A;
    out.Bz = u * S.Z;
    out.Bh = s * u * S.B;
    a_over_r = u * S.A;
}

}  // namespace ccoil
