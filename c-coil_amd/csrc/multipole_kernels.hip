// Far-field moments of the coils and the spatial visit order of the points (gfx950).
//
// multipole_moments_kernel: one workgroup per coil sums the zonal-harmonic moments of the coil's sheets (the field
// rule's thickness nodes, their length in closed form, multipole.hpp) in FP64, with a fixed reduction order.
//
// The visit order: the points' bounding box, a cell of a 2^k x 2^k x 2^k grid for every point (Morton order of the
// cells), a counting sort of the point indices by cell. field_kernel reads its points in that order, so the 64
// points of a wave lie in one or two neighbouring cells and a wave mostly takes one branch (series or rule) per
// coil. Each point's arithmetic does not depend on which wave holds it, so the order within a cell (set by
// atomics) does not change any result.
#include "kernels.hpp"
#include "multipole.hpp"

namespace ccoil {

constexpr int kMomThreads = 128;   // one sheet a thread
constexpr int kMomOrders = 32;     // odd orders summed at a time
constexpr int kMomStride = kMaxOrder + 1;   // odd, so that a column of orders crosses the LDS banks
static_assert(kMaxOrder <= kMomThreads && kMomStride % 2 == 1 && kMpOdd % kMomOrders == 0, "moments block");

// Moments of coil blockIdx.x. Thread j steps the recurrences of the sheet at thickness node j (squared half-length z2,
// c2 = rho^2 + z2, in units of r_max) over 32 odd orders, then four threads an order add the sheets. With U_l, V_l of
// multipole.hpp at height h, E_l = U_l (even l), O_l = U_l / h and G_(l+1) = V_(l+1) / h (odd l) contain no odd power
// of h, so that a flat sheet (h = 0, also a slow-rule coil's) needs no case of its own; the length average of V_l is
// G_(l+1) / (l + 2). Bound by the recurrence's latency, some 25 cycles an order; 63 length nodes for each thickness
// node, summed over the wave at every order, took 90 us for 128 coils and 1.96 ms for 8,192, this 13 and 50 us.
__global__ __launch_bounds__(kMomThreads) void multipole_moments_kernel(const CoilDev *coils, Tables tab, double *mp)
{
    __shared__ double inv[2 * kMpOdd + 2];                // 1 / l
    __shared__ double term[kMomOrders][kMomStride];       // per order and sheet
    __shared__ double part[4][kMomOrders];
    const int ci = blockIdx.x, t = threadIdx.x;
    const CoilDev &c = coils[ci];
    double *out = mp + (size_t)ci * kMpCoil;
    const double *kn = tab.leg + 4 * kMpOdd;
    for (int l = t; l < 2 * kMpOdd + 2; l += kMomThreads) inv[l] = l > 0 ? 1.0 / l : 0.0;
    const int nt = c.n_thk, terms = c.far_d2 > 0.0 ? (c.mp_terms < kMpTerms ? c.mp_terms : kMpTerms) : 0;
    const double scale = 1.0 / c.rmax, h = c.use_fast ? 0.5 * c.b * scale : 0.0, z2 = h * h;
    double c2 = 0.0, w = 0.0;
    if (t < nt) {
        const double *xt = tab.x + table_offset(nt), *wt = tab.w + table_offset(nt);
        const double rho = (c.R + 0.5 * c.a * (1.0 + xt[t])) * scale;
        c2 = rho * rho + z2;
        w = 0.5 * wt[t] * rho * rho;   // its share of the current (the weights sum to 1), times rho^2
    }
    double E = 1.0, O = 1.0, G = 3.0;   // E_(l-1), O_l, G_(l+1) at l = 1
    const double ni = c.ni * (4.0 * kPi * kMuReduced);   // m_l = mu0 N I sum / (2 (l + 1)), mu0 = 4 pi 1e-7
    __syncthreads();
    for (int i0 = 0; i0 < kMpOdd; i0 += kMomOrders) {
        const int l0 = 2 * i0;
        if (l0 >= terms) {   // no series, or none of these orders
            for (int k = t; k < 4 * kMomOrders; k += kMomThreads) out[4 * i0 + k] = 0.0;
            if (t < kMomOrders) out[4 * kMpOdd + i0 + t] = 0.0;
            continue;
        }
        if (t < nt)
#pragma unroll 4
            for (int i = 0; i < kMomOrders; ++i) {
                const int l = l0 + 2 * i + 1;
                const double fl = l;
                term[i][t] = w * G;
                E = ((2.0 * fl + 1.0) * z2 * O - fl * c2 * E) * inv[l + 1];
                O = ((2.0 * fl + 3.0) * E - (fl + 1.0) * c2 * O) * inv[l + 2];
                G = c2 * G + (2.0 * fl + 5.0) * O;
            }
        __syncthreads();
        const int i = t % kMomOrders, q = t / kMomOrders;
        double sum = 0.0;
#pragma unroll 4
        for (int j = q; j < nt; j += 4) sum += term[i][j];
        part[q][i] = sum;
        __syncthreads();
        if (t < kMomOrders) {
            const int l = l0 + 2 * t + 1;
            double m = 0.0;
            if (l <= kMpTerms)
                m = ni * (((part[0][t] + part[1][t]) + (part[2][t] + part[3][t])) * inv[l + 2]) / (2.0 * (l + 1));
            double *row = out + 4 * (i0 + t);
            row[0] = m;
            row[1] = (l + 1) * m * kn[l + 1];
            row[2] = (l + 1.0) * (l + 2.0) * m * kn[l + 2];
            row[3] = (l + 1) * m;
            out[4 * kMpOdd + i0 + t] = m / l;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Visit order.
// ---------------------------------------------------------------------------------------------
constexpr int kBoxBlocks = 512;

__device__ inline void minmax6(double *v, const double *o)
{
    for (int k = 0; k < 3; ++k) {
        v[k] = fmin(v[k], o[k]);
        v[3 + k] = fmax(v[3 + k], o[3 + k]);
    }
}

// Block-wide min/max of 6 values (3 minima, 3 maxima), result in thread 0.
__device__ inline void block_minmax6(double *v)
{
    __shared__ double sh[4][6];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        double o[6];
        for (int k = 0; k < 6; ++k) o[k] = __shfl_xor(v[k], m, 64);
        minmax6(v, o);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0)
        for (int k = 0; k < 6; ++k) sh[wave][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < 4; ++w) minmax6(v, sh[w]);
}

__global__ __launch_bounds__(256) void box_partial_kernel(const double *pts, int64_t n, double *part)
{
    double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const double p[6] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2], pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
        minmax6(v, p);
    }
    block_minmax6(v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; ++k) part[6 * blockIdx.x + k] = v[k];
}

__global__ __launch_bounds__(256) void box_final_kernel(const double *part, int n_part, double *box)
{
    double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int b = threadIdx.x; b < n_part; b += 256) minmax6(v, part + 6 * b);
    block_minmax6(v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; ++k) box[k] = v[k];
}

// Spreads the low 10 bits of x to every third bit.
__device__ inline uint32_t spread3(uint32_t x)
{
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// Cell (Morton code of the 2^bits grid over the box) of every point, and the points per cell.
__global__ __launch_bounds__(256) void cell_count_kernel(const double *pts, int64_t n, const double *box, int bits,
                                                         uint32_t *cell, unsigned long long *count)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int cells = 1 << bits;
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
        const double ext = box[3 + k] - box[k];
        const double f = ext > 0.0 ? (pts[3 * i + k] - box[k]) / ext * cells : 0.0;   // in [0, cells]
        q[k] = f >= 1.0 ? (uint32_t)fmin(f, cells - 1.0) : 0u;   // NaN and non-finite boxes: cell 0
    }
    const uint32_t key = spread3(q[0]) | (spread3(q[1]) << 1) | (spread3(q[2]) << 2);
    cell[i] = key;
    atomicAdd(&count[key], 1ull);
}

// order[cursor[cell]++] = point (cursor: the exclusive prefix sum of the cell counts).
__global__ __launch_bounds__(256) void cell_place_kernel(const uint32_t *cell, int64_t n, unsigned long long *cursor,
                                                         uint32_t *order)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const unsigned long long pos = atomicAdd(&cursor[cell[i]], 1ull);
    if (pos < (unsigned long long)n) order[pos] = (uint32_t)i;
}

void launch_multipole_moments(hipStream_t s, const CoilDev *coils, int n_coils, const Tables &tab, double *mp)
{
    if (n_coils > 0)
        hipLaunchKernelGGL(multipole_moments_kernel, dim3(n_coils), dim3(kMomThreads), 0, s, coils, tab, mp);
}

size_t visit_order_bytes(int64_t cap, int bits, size_t scan_bytes)
{
    const size_t cells = (size_t)1 << (3 * bits);
    return sizeof(double) * (6 * kBoxBlocks + 8) + sizeof(uint32_t) * (size_t)cap + 2 * sizeof(int64_t) * cells +
           scan_bytes + 6 * 256;
}

int64_t *visit_order_counts(void *temp, int64_t cap)
{
    auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
    return (int64_t *)((char *)temp + align(sizeof(double) * 6 * kBoxBlocks) + align(sizeof(double) * 8) +
                       align(sizeof(uint32_t) * (size_t)cap));
}

hipError_t launch_visit_order(hipStream_t s, const double *pts, int64_t n, int bits, void *temp, int64_t cap,
                              size_t scan_bytes, uint32_t *order)
{
    const size_t cells = (size_t)1 << (3 * bits);
    auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
    char *t = (char *)temp;
    double *part = (double *)t;
    t += align(sizeof(double) * 6 * kBoxBlocks);
    double *box = (double *)t;
    t += align(sizeof(double) * 8);
    uint32_t *cell = (uint32_t *)t;
    t += align(sizeof(uint32_t) * (size_t)cap);
    int64_t *count = visit_order_counts(temp, cap);
    t += align(sizeof(int64_t) * cells);
    int64_t *cursor = (int64_t *)t;
    t += align(sizeof(int64_t) * cells);
    void *scan_temp = t;
    const int blocks = (int)((n + 255) / 256 < kBoxBlocks ? (n + 255) / 256 : kBoxBlocks);
    hipLaunchKernelGGL(box_partial_kernel, dim3(blocks), dim3(256), 0, s, pts, n, part);
    hipLaunchKernelGGL(box_final_kernel, dim3(1), dim3(256), 0, s, part, blocks, box);
    const unsigned grid = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(cell_count_kernel, dim3(grid), dim3(256), 0, s, pts, n, box, bits, cell,
                       (unsigned long long *)count);
    size_t tb = scan_bytes;
    hipError_t e = near_scan(s, count, cursor, (int64_t)cells, scan_temp, tb);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(cell_place_kernel, dim3(grid), dim3(256), 0, s, cell, n, (unsigned long long *)cursor, order);
    return hipGetLastError();
}

}  // namespace ccoil
