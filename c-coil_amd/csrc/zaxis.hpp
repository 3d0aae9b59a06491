// Coaxial (z-axis) pair rules and self-inductance on the device: work items, parameters and launchers.
#pragma once

#include "common.hpp"

namespace ccoil {

enum : int32_t { kZMutual = 0, kZForce = 1, kZSelf = 2 };
constexpr int kZBlock = 256;   // threads per workgroup of zaxis_kernel

// Thickness nodes per thread, at most. A full rule's node costs some 1,500 cycles, so that the last workgroups of a
// batch would otherwise run alone through up to 100 of them.
constexpr int kZNodes = 8;

constexpr int64_t kZBatch = 1 << 22;   // workgroups of a launch, of several items at least

// One coaxial pair (its M, its axial force or both) or one coil's self-inductance, by full or reduced rules. Every
// workgroup of a quantity covers kZBlock units; each sums over its share of the primary's thickness nodes.
struct alignas(16) ZItemDev {
    double z;             // the centres' distance (self: the coil's length)
    double hs, hp;        // half-lengths of the secondary and the primary
    double r_inner;       // radial rule: r = r_inner + r_width (block + 0.5) + r_width / 2 x
    double r_width;
    double t_inner;       // primary thickness rule, same form
    double t_width;
    double a_width;       // angular block width pi / blocks
    double constant;      // per-node constant of the reference rule
    double mul, div;      // mutual: sum * 2 pi / div, force: sum * -2 pi, self: sum * 2 pi * mul / div
    int64_t first_wg;     // first workgroup of this item (ascending over items); n_wg of each quantity in turn
    int64_t n_wg, units;  // units: radial nodes x angular nodes x length nodes x t_split
    int32_t r_blk, t_blk, a_blk;
    int32_t out;          // index into ZParams::out, of the first quantity
    int16_t r_inc, t_inc, a_inc;
    int16_t l_inc;        // reduced rules: the length nodes; 0: full rules
    int16_t a_off;        // reduced rules: the angular node set's offset in the tables
    int16_t t_split;      // threads that share a unit's thickness nodes
};

struct ZParams {
    const ZItemDev *items;
    const int32_t *wg_item;   // the item of each workgroup (null for one item beyond kZBatch workgroups)
    int32_t n_items;
    int32_t mode, n_modes;    // the first quantity and their number (kZMutual and kZForce: two)
    int64_t out_stride;       // between the quantities in out
    int64_t n_wg;
    double *partial;      // one per workgroup
    double *out;
    Tables tab;
};

void launch_zaxis(hipStream_t s, const ZParams &p);
void launch_zaxis_reduce(hipStream_t s, const ZParams &p);

}  // namespace ccoil
