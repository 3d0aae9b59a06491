// C ABI: ccoil_pairs_zaxis and ccoil_self_inductance (coaxial rules, include/ccoil_hip.h).
#include "context.hpp"
#include "zaxis.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

using namespace ccoil;

namespace {

constexpr double kMu = 1e-7;   // g_MiReduced (CalculateMInductanceZAxis.cxx:12)

// Distance sum, in units of half the length, from the points (x, y), x in [x0, x1], to the ends of the segment
// [lo, lo + len] of the x axis: the least over them.
double ellipse_sum(double lo, double len, double x0, double x1, double y)
{
    const double mid = lo + 0.5 * len, x = std::fmin(std::fmax(mid, x0), x1);   // the nearest to the middle is the least
    const double d0 = x - lo, d1 = d0 - len;
    return 2.0 * (std::sqrt(d0 * d0 + y * y) + std::sqrt(d1 * d1 + y * y)) / len;
}

// The reduced rules of a pair's M and force sums (na == 0: none); t, r 0: the coil's own nodes.
struct PairRule { int na, a_off, l, t, r; };

// Reduced rules (reduced_rules.cpp) for two coaxial coils clear of each other: R, a, h: the inner radii, thicknesses and
// half-lengths of the primary and the secondary, c the distance of their centres; n_ang, n_thk, n_rad their nodes.
//
// With g the axial and q the radial gap of the windings, the angular integrand at radii t, r is analytic for |Im phi| <
// eta, cosh(eta) = 1 + ((t - r)^2 + g^2) / (2 t r) (the terms singular at t = r alone cancel between the four
// offsets where the coils are axially apart); the thickness and radial integrands are analytic outside the other coil's
// nearest point in the meridian plane, as in the field rules; and the force and inductance of a sheet of half-length H
// at an offset l along the shorter coil (half-length h <= H) outside l = -c +- H +- i D, D >= q the in-plane distance.
// A rule of several blocks converges no later than one block of it. Coils that the angular or the length nodes do not
// serve (72 of a table of 1,500 random pairs) keep their rules.
PairRule pair_rule(double Rp, double ap, double hp, double Rs, double as, double hs, double c, int n_ang, int n_thk, int n_rad)
{
    PairRule rule = {0, 0, 0, 0, 0};
    const double g = std::fmax(0.0, std::fabs(c) - hp - hs);
    const double q = std::fmax(0.0, std::fmax(Rp - (Rs + as), Rs - (Rp + ap)));
    if (!(q + g > 0.0) || !(Rs >= 1e-15 && Rs + as <= 1e15)) return rule;   // (set_rule_limits: the primary's range)
    CoilDev d;
    d.R = Rp;
    d.a = ap;
    d.b = 2.0 * hp;
    d.use_fast = 1;
    d.n_ang = n_ang;
    d.n_thk = n_thk;
    set_rule_limits(d);
    const float num = (float)(q * q + g * g), den = (float)(2.0 * (Rp + ap) * (Rs + as));
    const int cls = class_of(d, num, den, (float)ellipse_sum(Rp, ap, Rs, Rs + as, g));
    const int k = cls / (kRedThk + 1), t = cls % (kRedThk + 1);
    const double H = std::fmax(hp, hs), h = std::fmin(hp, hs), x0 = -c + H, x1 = -c - H;
    d.n_thk = n_rad;
    d.R = Rs;
    d.a = as;
    set_rule_limits(d);
    const int r = class_of(d, num, den, (float)ellipse_sum(Rs, as, Rp, Rp + ap, g)) % (kRedThk + 1);
    d.n_thk = kMaxOrder;
    d.a = d.R;
    set_rule_limits(d);
    const double sl = std::fmin(ellipse_sum(-h, 2.0 * h, x0, x0, q), ellipse_sum(-h, 2.0 * h, x1, x1, q));
    const int l = class_of(d, num, den, (float)sl) % (kRedThk + 1);
    if (k == 0 || l == 0) return rule;
    rule.na = kRedAngN[k - 1];
    rule.a_off = kRedOffset;
    for (int i = 0; i < k - 1; ++i) rule.a_off += kRedAngN[i];
    rule.l = kRedThkN[l - 1];
    rule.t = t ? kRedThkN[t - 1] : 0;
    rule.r = r ? kRedThkN[r - 1] : 0;
    return rule;
}

// Rewrites a pair's item with its reduced rules.
void reduce_item(ZItemDev &it, const PairRule &rule)
{
    it.constant *= kPi * std::fmin(it.hp, it.hs) / it.a_width;
    it.a_blk = 1;
    it.a_inc = (int16_t)rule.na;
    it.a_off = (int16_t)rule.a_off;
    it.l_inc = (int16_t)rule.l;
    if (rule.t) {
        it.constant *= it.t_blk;
        it.t_width *= it.t_blk;
        it.t_blk = 1;
        it.t_inc = (int16_t)rule.t;
    }
    if (rule.r) {
        it.constant *= it.r_blk;
        it.r_width *= it.r_blk;
        it.r_blk = 1;
        it.r_inc = (int16_t)rule.r;
    }
}

// Sets the item's units from its rules. An item that fills the chip several times over by itself needs no sharing of its
// thickness nodes, and so never takes more workgroups than its (radial, angular) nodes.
void set_units(ZItemDev &it)
{
    const int64_t units = (int64_t)it.r_blk * it.r_inc * it.a_blk * it.a_inc * std::max<int>(it.l_inc, 1);
    it.t_split = (int16_t)(units < (int64_t)kZBlock * 16384 ? (it.t_inc + kZNodes - 1) / kZNodes : 1);
    it.units = units * it.t_split;
    it.n_wg = (it.units + kZBlock - 1) / kZBlock;
}

bool valid_rule(int32_t blocks, int32_t inc) { return blocks >= 1 && inc >= 1 && inc <= kMaxOrder; }

// Upload the items, run the node kernel and the ordered reduction for `modes` quantities from `mode` on, copy n_out
// results back. The items go in batches of kZBatch workgroups (one item at least): a launch of 2^32 threads or more runs
// what is left over, without an error, and shared thickness nodes make up to 13 workgroups of one of the planned rule's.
// planned_wg: those of the planned rules, which the documented limit counts.
ccoil_status run_items(ccoil_ctx ctx, std::vector<ZItemDev> &items, int64_t planned_wg, int32_t mode, int32_t modes,
                       size_t n_out, uint32_t flags, double *out_host, double *out_dev, int64_t node_evals,
                       ccoil_report *report)
{
    if (planned_wg > INT32_MAX) return fail(ctx, CCOIL_ERR_ARGUMENT, "coaxial batch needs more than 2^31 - 1 workgroups");
    CC_HIP(ctx, hipSetDevice(ctx->device));
    // each batch: its items, then each workgroup's item
    struct Batch { std::vector<ZItemDev> rows; size_t n_items; int64_t wg; bool mapped; };
    std::vector<Batch> batches;
    size_t max_rows = 0;
    int64_t max_wg = 0;
    for (size_t i = 0; i < items.size();) {
        const size_t i0 = i;
        int64_t wg = 0;
        for (; i < items.size() && (i == i0 || wg + modes * items[i].n_wg <= kZBatch); ++i) {
            items[i].first_wg = wg;
            wg += modes * items[i].n_wg;
        }
        Batch b = {{}, i - i0, wg, wg <= kZBatch};
        if (i0 == 0 && i == items.size()) b.rows.swap(items);
        else b.rows.assign(items.begin() + (std::ptrdiff_t)i0, items.begin() + (std::ptrdiff_t)i);
        if (b.mapped) {
            b.rows.resize(b.n_items + ((size_t)wg * sizeof(int32_t) + sizeof(ZItemDev) - 1) / sizeof(ZItemDev));
            int32_t *wg_item = reinterpret_cast<int32_t *>(b.rows.data() + b.n_items);
            for (size_t k = 0; k < b.n_items; ++k) wg_item = std::fill_n(wg_item, modes * b.rows[k].n_wg, (int32_t)k);
        }
        max_rows = std::max(max_rows, b.rows.size());
        max_wg = std::max(max_wg, wg);
        batches.push_back(std::move(b));
        if (batches.back().n_items == i && items.empty()) break;   // the only batch took them all
    }
    CC_HIP(ctx, ensure(ctx->zitems, sizeof(ZItemDev) * max_rows));
    CC_HIP(ctx, ensure(ctx->zpartial, sizeof(double) * (size_t)max_wg));
    ZParams zp;
    std::memset(&zp, 0, sizeof zp);
    zp.items = (const ZItemDev *)ctx->zitems.p;
    zp.mode = mode;
    zp.n_modes = modes;
    zp.out_stride = modes > 1 ? (int64_t)n_out / modes : 0;
    zp.partial = (double *)ctx->zpartial.p;
    zp.tab = ctx_tables(ctx);
    const bool dev = flags & CCOIL_DEVICE_POINTERS;
    if (dev) {
        zp.out = out_dev;
    } else {
        CC_HIP(ctx, ensure(ctx->zout, sizeof(double) * n_out));
        zp.out = (double *)ctx->zout.p;
    }
    for (size_t k = 0; k < batches.size(); ++k) {   // in stream order, so the next upload waits for the last reduction
        const Batch &b = batches[k];
        CC_HIP(ctx, hipMemcpyAsync(ctx->zitems.p, b.rows.data(), sizeof(ZItemDev) * b.rows.size(), hipMemcpyHostToDevice,
                                   ctx->stream));
        zp.wg_item = b.mapped ? (const int32_t *)(zp.items + b.n_items) : nullptr;
        zp.n_items = (int32_t)b.n_items;
        zp.n_wg = b.wg;
        if (k == 0) CC_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
        launch_zaxis(ctx->stream, zp);
        CC_HIP(ctx, hipGetLastError());
        if (k + 1 == batches.size()) CC_HIP(ctx, hipEventRecord(ctx->evm1, ctx->stream));
        launch_zaxis_reduce(ctx->stream, zp);
        CC_HIP(ctx, hipGetLastError());
    }
    CC_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    if (!dev) CC_HIP(ctx, hipMemcpyAsync(out_host, zp.out, sizeof(double) * n_out, hipMemcpyDeviceToHost, ctx->stream));
    CC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (report) {
        float ms = 0.f, mms = 0.f;
        CC_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        CC_HIP(ctx, hipEventElapsedTime(&mms, ctx->ev0, ctx->evm1));
        report->node_evaluations = node_evals;
        report->kernel_ms = ms;
        report->main_kernel_ms = mms;
        report->block_size = kZBlock;
        report->split = 1;
    }
    return CCOIL_OK;
}

std::string check_coils(const ccoil_coils *c, const char *who)
{
    if (!c) return std::string(who) + " descriptor is NULL";
    if (c->n < 0) return std::string(who) + " count is negative";
    if (c->n == 0) return "";
    if (!c->n_ang || !c->n_thk || !c->R || !c->a || !c->b || !c->J || !c->pos || !c->current || !c->turns)
        return std::string(who) + " descriptor needs n_ang, n_thk, R, a, b, J, pos, current and turns";
    for (int64_t i = 0; i < c->n; ++i) {
        const int32_t ab = c->blocks ? c->blocks[3 * i] : 1, tb = c->blocks ? c->blocks[3 * i + 1] : 1;
        if (!valid_rule(ab, c->n_ang[i]) || !valid_rule(tb, c->n_thk[i]))
            return std::string(who) + " " + std::to_string(i) + ": blocks must be >= 1 and increments in [1, 100]";
        if (!(c->R[i] > 0.0) || !(c->a[i] > 0.0) || !(c->b[i] > 0.0) || !std::isfinite(c->J[i]))
            return std::string(who) + " " + std::to_string(i) + ": R, a, b must be positive and J finite";
    }
    return "";
}

}  // namespace

extern "C" ccoil_status ccoil_pairs_zaxis(ccoil_ctx ctx, const ccoil_coils *prim, const ccoil_coils *sec,
                                          const int64_t *prim_index, const int64_t *sec_index, int64_t n_pairs,
                                          uint32_t what, uint32_t flags, double *M, double *Fz, ccoil_report *report)
{
    if (!ctx) return fail(nullptr, CCOIL_ERR_ARGUMENT, "ccoil_pairs_zaxis: ctx is NULL");
    if (n_pairs < 0) return fail(ctx, CCOIL_ERR_ARGUMENT, "n_pairs is negative");
    if (n_pairs > INT32_MAX / 2) return fail(ctx, CCOIL_ERR_ARGUMENT, "n_pairs exceeds 2^30 - 1");
    if (what == 0 || (what & ~(uint32_t)(CCOIL_PAIR_M | CCOIL_PAIR_FT)))
        return fail(ctx, CCOIL_ERR_ARGUMENT, "coaxial pairs compute CCOIL_PAIR_M and/or CCOIL_PAIR_FT");
    if ((what & CCOIL_PAIR_M) && !M) return fail(ctx, CCOIL_ERR_ARGUMENT, "M requested but M is NULL");
    if ((what & CCOIL_PAIR_FT) && !Fz) return fail(ctx, CCOIL_ERR_ARGUMENT, "force requested but Fz is NULL");
    std::string msg = check_coils(prim, "primary coil");
    if (msg.empty()) msg = check_coils(sec, "secondary coil");
    if (!msg.empty()) return fail(ctx, CCOIL_ERR_ARGUMENT, msg);
    if (report) std::memset(report, 0, sizeof *report);
    if (n_pairs == 0) return CCOIL_OK;
    if (prim->n == 0 || sec->n == 0) return fail(ctx, CCOIL_ERR_ARGUMENT, "pairs given but a coil array is empty");

    std::vector<ZItemDev> items, reduced;   // full rules are launched first: their workgroups run longest
    items.reserve((size_t)n_pairs + 1);
    reduced.reserve((size_t)n_pairs);
    int64_t evals = 0, planned_wg = 0;
    const int modes = (what & CCOIL_PAIR_M ? 1 : 0) + (what & CCOIL_PAIR_FT ? 1 : 0);
    for (int64_t k = 0; k < n_pairs; ++k) {
        const int64_t i = prim_index ? prim_index[k] : k, j = sec_index ? sec_index[k] : k;
        if (i < 0 || i >= prim->n || j < 0 || j >= sec->n)
            return fail(ctx, CCOIL_ERR_ARGUMENT, "pair " + std::to_string(k) + ": coil index out of range");
        ZItemDev it;
        std::memset(&it, 0, sizeof it);
        it.out = (int32_t)k;
        it.a_blk = prim->blocks ? prim->blocks[3 * i] : 1;
        it.t_blk = prim->blocks ? prim->blocks[3 * i + 1] : 1;
        it.r_blk = sec->blocks ? sec->blocks[3 * j + 1] : 1;
        it.a_inc = (int16_t)prim->n_ang[i];
        it.t_inc = (int16_t)prim->n_thk[i];
        it.r_inc = (int16_t)sec->n_thk[j];
        const double t_width = prim->a[i] / it.t_blk, a_width = kPi / it.a_blk, r_width = sec->a[j] / it.r_blk;
        it.t_inner = prim->R[i];
        it.t_width = t_width;
        it.a_width = a_width;
        it.r_inner = sec->R[j];
        it.r_width = r_width;
        it.constant = kMu * prim->J[i] * sec->J[j] * t_width * a_width * r_width * 0.125;
        it.z = sec->pos[3 * j + 2] - prim->pos[3 * i + 2];
        it.hs = sec->b[j] * 0.5;
        it.hp = prim->b[i] * 0.5;
        if (what & CCOIL_PAIR_M) {
            if (prim->current[i] == 0.0 || sec->current[j] == 0.0)
                return fail(ctx, CCOIL_ERR_ARGUMENT, "pair " + std::to_string(k) + ": mutual inductance needs "
                                                     "non-zero currents (M = sum * 2 pi / (I1 I2))");
            it.div = prim->current[i] * sec->current[j];
        }
        planned_wg += modes * (((int64_t)it.r_blk * it.r_inc * it.a_blk * it.a_inc + kZBlock - 1) / kZBlock);
        evals += (int64_t)modes * it.r_blk * it.r_inc * it.a_blk * it.a_inc * it.t_blk * it.t_inc;
        const PairRule rule = pair_rule(it.t_inner, prim->a[i], it.hp, it.r_inner, sec->a[j], it.hs, it.z, it.a_inc,
                                        it.t_inc, it.r_inc);
        const bool reduce = rule.na && it.r_blk <= 1 << 10;   // a reduced item's units are counted in 32 bits
        if (reduce) reduce_item(it, rule);
        set_units(it);
        (reduce ? reduced : items).push_back(it);
    }
    items.insert(items.end(), reduced.begin(), reduced.end());
    const int32_t mode = what & CCOIL_PAIR_M ? kZMutual : kZForce;
    // results: M, then Fz, of what is asked for, staged in one device buffer
    const size_t n_out = (size_t)n_pairs * (size_t)modes;
    const size_t f_at = modes > 1 ? (size_t)n_pairs : 0;
    const bool dev = flags & CCOIL_DEVICE_POINTERS;
    if (dev) {
        // device outputs are written in place: route M and Fz through one staging buffer, then copy on device
        CC_HIP(ctx, ensure(ctx->zout, sizeof(double) * n_out));
        ccoil_status st = run_items(ctx, items, planned_wg, mode, modes, n_out, flags, nullptr, (double *)ctx->zout.p, evals, report);
        if (st != CCOIL_OK) return st;
        const size_t s1 = sizeof(double) * (size_t)n_pairs;
        if (what & CCOIL_PAIR_M) CC_HIP(ctx, hipMemcpyAsync(M, ctx->zout.p, s1, hipMemcpyDeviceToDevice, ctx->stream));
        if (what & CCOIL_PAIR_FT)
            CC_HIP(ctx, hipMemcpyAsync(Fz, (double *)ctx->zout.p + f_at, s1, hipMemcpyDeviceToDevice, ctx->stream));
        CC_HIP(ctx, hipStreamSynchronize(ctx->stream));
        return CCOIL_OK;
    }
    std::vector<double> host(n_out);
    ccoil_status st = run_items(ctx, items, planned_wg, mode, modes, n_out, flags, host.data(), nullptr, evals, report);
    if (st != CCOIL_OK) return st;
    if (what & CCOIL_PAIR_M) std::memcpy(M, host.data(), sizeof(double) * (size_t)n_pairs);
    if (what & CCOIL_PAIR_FT) std::memcpy(Fz, host.data() + f_at, sizeof(double) * (size_t)n_pairs);
    return CCOIL_OK;
}

extern "C" ccoil_status ccoil_self_inductance(ccoil_ctx ctx, const ccoil_coils *coils, const int32_t *radial,
                                              uint32_t flags, double *L, ccoil_report *report)
{
    if (!ctx) return fail(nullptr, CCOIL_ERR_ARGUMENT, "ccoil_self_inductance: ctx is NULL");
    std::string msg = check_coils(coils, "coil");
    if (!msg.empty()) return fail(ctx, CCOIL_ERR_ARGUMENT, msg);
    if (coils->n > INT32_MAX) return fail(ctx, CCOIL_ERR_ARGUMENT, "coil count exceeds 2^31 - 1");
    if (report) std::memset(report, 0, sizeof *report);
    if (coils->n == 0) return CCOIL_OK;
    if (!radial || !L) return fail(ctx, CCOIL_ERR_ARGUMENT, "radial and L must not be NULL");
    std::vector<ZItemDev> items;
    int64_t evals = 0, planned_wg = 0;
    for (int64_t i = 0; i < coils->n; ++i) {
        if (!valid_rule(radial[2 * i], radial[2 * i + 1]))
            return fail(ctx, CCOIL_ERR_ARGUMENT, "coil " + std::to_string(i) + ": radial rule needs blocks >= 1 and "
                                                 "increments in [1, 100]");
        if (coils->current[i] == 0.0)
            return fail(ctx, CCOIL_ERR_ARGUMENT, "coil " + std::to_string(i) + ": self-inductance needs a non-zero "
                                                 "current (L = sum * 2 pi N / (I l))");
        ZItemDev it;
        std::memset(&it, 0, sizeof it);
        it.out = (int32_t)i;
        it.a_blk = coils->blocks ? coils->blocks[3 * i] : 1;
        it.t_blk = coils->blocks ? coils->blocks[3 * i + 1] : 1;
        it.r_blk = radial[2 * i];
        it.a_inc = (int16_t)coils->n_ang[i];
        it.t_inc = (int16_t)coils->n_thk[i];
        it.r_inc = (int16_t)radial[2 * i + 1];
        const double a = coils->a[i], len = coils->b[i];
        const double t_width = a / it.t_blk, a_width = kPi / it.a_blk, r_unit = 1.0 / it.r_blk;
        it.t_inner = coils->R[i];
        it.t_width = t_width;
        it.a_width = a_width;
        it.r_inner = coils->R[i];
        it.r_width = r_unit * a;   // the radial nodes span the thickness; the constant keeps the unit block
        it.constant = kMu * coils->J[i] * t_width * a_width * r_unit * 2 * 0.125;
        it.z = len;
        it.mul = coils->turns[i];
        it.div = coils->current[i] * len;
        planned_wg += ((int64_t)it.r_blk * it.r_inc * it.a_blk * it.a_inc + kZBlock - 1) / kZBlock;
        evals += (int64_t)it.r_blk * it.r_inc * it.a_blk * it.a_inc * it.t_blk * it.t_inc;
        set_units(it);
        items.push_back(it);
    }
    return run_items(ctx, items, planned_wg, kZSelf, 1, (size_t)coils->n, flags, L, L, evals, report);
}
