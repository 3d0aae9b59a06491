// Coaxial (z-axis) mutual inductance, axial force and self-inductance (gfx950).
//
// The length integrals of both coils are analytic in these rules; what remains is a 3-D Gauss-Legendre sum over
// the secondary's radial nodes r, the primary's thickness nodes t and the primary's angular nodes phi:
//   mutual  CalculateMInductanceZAxis.cxx:84-221   sum of w * 2tr cos(phi) * (H1 - H2 + H3 - H4 - E1 + E2 - E3 + E4)
//   force   CalculateForceZAxis.cxx:82-219         sum of w * 2tr cos(phi) * log(G2 G4 / (G1 G3))
//   self    CalculateMInductanceZAxis.cxx:224-317  sum of w * 2tr cos(phi) * (D - E + l H)
// One thread owns one (r, phi) unit and loops over the t nodes; the per-node terms are evaluated exactly as the
// reference writes them, in double with IEEE division and square root and without contraction, so the result
// differs from the reference's CPU sum only by the summation order and the last bit of cos and log.
//
// Mutual and force items of pairs whose windings are clear of each other take reduced rules instead (reduce_item,
// zaxis_api.cpp): the shorter coil's length by Gauss-Legendre nodes, at each of which the longer one is a sheet whose A
// (mutual) or B_rho (force) is summed over 6-20 angular, and mostly 6-22 thickness and radial nodes, by the field
// kernels' cancellation-free node terms with refined reciprocals. The reference's second difference of eight terms
// loses up to the square of distance over length to cancellation; this does not. Bound by FP64 issue either way: an
// item of 80 x 20 x 20 nodes, 9 IEEE square roots, 4 divisions and 4 logarithms each, becomes some 10 x 8 x 8 x 8 of a
// tenth of that (1,500 pairs, M and force: 504 -> 103 us, 40 of them the 72 pairs that keep their rules).
#include "integrands.hpp"
#include "zaxis.hpp"

namespace ccoil {

namespace {

__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// One (radial, length, angular) unit of a reduced item: the sum over its share of the thickness nodes.
template <bool MUTUAL> __device__ inline double reduced_unit(const ZItemDev &it, const Tables &tab, int u)
{
    const int n_phi = it.a_inc * it.l_inc, pl = u % n_phi, rest = u / n_phi, ip = pl % it.a_inc, il = pl / it.a_inc;
    const int ir = rest / it.t_split, ts = rest % it.t_split;
    const int rb = ir / it.r_inc, ri = ir - rb * it.r_inc;
    const double *xr = tab.x + table_offset(it.r_inc), *wr = tab.w + table_offset(it.r_inc);
    const double *xt = tab.x + table_offset(it.t_inc), *wt = tab.w + table_offset(it.t_inc);
    const double *xl = tab.x + table_offset(it.l_inc), *wl = tab.w + table_offset(it.l_inc);
    const double s = tab.omc[it.a_off + ip], wc = tab.wcos[it.a_off + ip];
    const double r = (it.r_inner + it.r_width * (rb + 0.5)) + (it.r_width * 0.5) * xr[ri];
    const double H = fmax(it.hp, it.hs), zc = it.z + fmin(it.hp, it.hs) * xl[il], zm = fabs(zc), z1 = zm + H, z2 = zm - H;
    const double W = it.constant * wr[ri] * wl[il] * wc * 2.0 * r, b = 2.0 * H, tbz = 2.0 * b * zm;
    const bool same = z2 > 0.0;
    SharedSums a = {0, 0, 0, 0, 0, 0};
    for (int tb = 0; tb < it.t_blk; ++tb) {
        const double tpos = it.t_inner + it.t_width * (tb + 0.5);
        for (int ti = ts; ti < it.t_inc; ti += it.t_split) {
            const double t = tpos + (it.t_width * 0.5) * xt[ti];
            shared_node<MUTUAL, !MUTUAL, false, true>(t, r, s, 0.0, 0.0, W * (wt[ti] * t), b, z1, z2, tbz, same, 0.0, a);
        }
    }
    return MUTUAL ? a.A : zc < 0.0 ? -a.Bh : a.Bh;
}

}  // namespace

__global__ __launch_bounds__(kZBlock) void zaxis_kernel(ZParams p)
{
#pragma clang fp contract(off)
    __shared__ double wsum[kZBlock / 64];
    const int64_t wg = blockIdx.x;
    // its item: the last with first_wg <= wg (workgroup-uniform)
    int lo = p.wg_item ? p.wg_item[wg] : 0, hi = p.wg_item ? lo : p.n_items - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.items[mid].first_wg <= wg) lo = mid;
        else hi = mid - 1;
    }
    const ZItemDev &it = p.items[lo];
    const int64_t w = wg - it.first_wg;
    const int mode = w >= it.n_wg ? kZForce : p.mode;
    const int64_t u = (w >= it.n_wg ? w - it.n_wg : w) * kZBlock + threadIdx.x;
    double acc = 0.0;
    if (it.l_inc) {
        if (u < it.units) acc = mode == kZMutual ? reduced_unit<true>(it, p.tab, (int)u)
                                                : reduced_unit<false>(it, p.tab, (int)u);
    } else if (u < it.units) {
        const int n_phi = it.a_blk * it.a_inc;
        const int64_t rest = u / n_phi;
        const int ip = (int)(u % n_phi), ir = (int)(rest / it.t_split), ts = (int)(rest % it.t_split);
        const int ab = ip / it.a_inc, ai = ip - ab * it.a_inc;
        const int rb = ir / it.r_inc, ri = ir - rb * it.r_inc;
        const double *xa = p.tab.x + table_offset(it.a_inc), *wa = p.tab.w + table_offset(it.a_inc);
        const double *xr = p.tab.x + table_offset(it.r_inc), *wr = p.tab.w + table_offset(it.r_inc);
        const double *xt = p.tab.x + table_offset(it.t_inc), *wt = p.tab.w + table_offset(it.t_inc);
        const double cp = cos(it.a_width * (ab + 0.5) + (it.a_width * 0.5) * xa[ai]);
        const double wF = wa[ai];
        const double r = (it.r_inner + it.r_width * (rb + 0.5)) + (it.r_width * 0.5) * xr[ri];
        const double wR = wr[ri];
        const double z[4] = {it.z + it.hs + it.hp, it.z + it.hs - it.hp, it.z - it.hs - it.hp, it.z - it.hs + it.hp};
        const double zsq[4] = {z[0] * z[0], z[1] * z[1], z[2] * z[2], z[3] * z[3]};
        for (int tb = 0; tb < it.t_blk; ++tb) {
            const double tpos = it.t_inner + it.t_width * (tb + 0.5);
            for (int ti = ts; ti < it.t_inc; ti += it.t_split) {
                const double t = tpos + (it.t_width * 0.5) * xt[ti];
                const double tc = it.constant * wR * wt[ti];
                const double A = 2.0 * t * r;
                const double B = t * t + r * r;
                const double C = B - A * cp;
                const double D = sqrt(C);
                double f;
                if (mode == kZMutual) {
                    double E[4], H[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        E[k] = sqrt(C + zsq[k]);
                        const double F = z[k] / D;
                        const double G = sqrt(F * F + 1.0);
                        H[k] = z[k] * log(F + G);
                    }
                    f = H[0] - H[1] + H[2] - H[3] - E[0] + E[1] - E[2] + E[3];
                } else if (mode == kZForce) {
                    double G[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const double E = z[k] / D;
                        G[k] = E + sqrt(E * E + 1.0);
                    }
                    f = log(G[1] * G[3] / (G[0] * G[2]));
                } else {
                    const double len = it.z;
                    const double E = sqrt(C + len * len);
                    const double F = len / D;
                    const double G = sqrt(F * F + 1.0);
                    f = D - E + len * log(F + G);
                }
                acc += tc * wF * A * cp * f;
            }
        }
    }
    // fixed-order workgroup sum: butterfly within each wave, then the waves in index order
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kZBlock / 64; ++w) s += wsum[w];
        p.partial[wg] = s;
    }
}

// One thread per item and quantity: its workgroup partials in workgroup order, then the reference's final factors.
__global__ __launch_bounds__(256) void zaxis_reduce_kernel(ZParams p)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= p.n_items) return;
    const ZItemDev &it = p.items[k];
    const int mode = blockIdx.y ? kZForce : p.mode;
    const double *part = p.partial + it.first_wg + (blockIdx.y ? it.n_wg : 0);
    double s = 0.0;
    for (int64_t w = 0; w < it.n_wg; ++w) s += part[w];
    constexpr double k2Pi = 6.283185307179586476925286766559;
    p.out[it.out + (blockIdx.y ? p.out_stride : 0)] =
        mode == kZMutual ? s * k2Pi / it.div : mode == kZForce ? s * -k2Pi : ((s * k2Pi) * it.mul) / it.div;
}

void launch_zaxis(hipStream_t s, const ZParams &p)
{
    if (p.n_wg <= 0) return;
    hipLaunchKernelGGL(zaxis_kernel, dim3((unsigned)p.n_wg), dim3(kZBlock), 0, s, p);
}

void launch_zaxis_reduce(hipStream_t s, const ZParams &p)
{
    if (p.n_items <= 0) return;
    hipLaunchKernelGGL(zaxis_reduce_kernel, dim3((p.n_items + 255) / 256, p.n_modes), dim3(256), 0, s, p);
}

}  // namespace ccoil
