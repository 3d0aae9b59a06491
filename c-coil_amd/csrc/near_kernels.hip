// Record pass (gfx950): the (coil, point) pairs field_kernel defers. In FP32C those inside a coil's near shell (and,
// for outputs that divide by r, its axis cone) are re-evaluated in FP64; with rule records (the series modes, large
// calls) every pair inside the far-field distance is, by the FP64 or the float rule (its record's kind), on waves
// that share one coil instead of beside the series.
//
// field_kernel skips those pairs and counts them per point; an exclusive scan of the point counts gives each point's
// places; near_count_kernel counts the records of each key (slot and coil, record_slot) and near_key_scan_kernel turns
// those counts into cursors (a counting sort by key) and checks the total against the buffers' capacity;
// near_fill_kernel places one (key, point | place) record per pair at its key's cursor, so that the lanes of a wave
// evaluate the same coil and, in large calls, the same reduced rule (uniform loop bounds and scalar tables);
// near_eval_kernel (in smaller calls near_eval_group_kernel) evaluates a record per lane or group of lanes into its
// place; near_add_kernel adds a point's values to the outputs in coil order. A value depends only on its (coil, point),
// and every sum has a fixed order, so results are bitwise reproducible although the order of the records within a key
// is not. Nothing here is read back by the host before the work is done.
#include <algorithm>
#include <cstddef>

#include "kernels.hpp"
#include "integrands.hpp"

namespace ccoil {

// Whether the points of a wave may be records of the coils c0 .. c0 + 7 (bit j for coil c0 + j < n_coils): false
// only where every point lies beyond the coil's far-field sphere by more than a margin, tested in the global frame
// (the rotation to the coil's frame keeps lengths up to a few ulps, far below the margin). The exact class is
// record_kind's; this lets a wave skip the frame transform of the coils none of its points can be a record of. The
// coils' centres and far_d2 are read through the constant address space: the records do not change during a
// launch, so these are scalar loads at wave-uniform indices although the loops that call this also store to global
// memory (through a generic pointer their loads would be vector loads, each a full memory round trip). The eight
// coils' loads come first, so a wave waits for them once.
__device__ inline uint32_t record_candidates(const CoilDev *coils, int n_coils, int c0, double px, double py,
                                             double pz)
{
    typedef const __attribute__((address_space(4))) double cdouble;
    constexpr int kPos = offsetof(CoilDev, pos) / sizeof(double), kFar = offsetof(CoilDev, far_d2) / sizeof(double);
    double fd[8], cx[8], cy[8], cz[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {   // past the last coil, the last coil again (its bit is cleared below)
        cdouble *f = (cdouble *)(const void *)(coils + min(c0 + j, n_coils - 1));
        fd[j] = f[kFar];
        cx[j] = f[kPos];
        cy[j] = f[kPos + 1];
        cz[j] = f[kPos + 2];
    }
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const double dx = px - cx[j], dy = py - cy[j], dz = pz - cz[j];
        const bool may = !(fd[j] > 0.0) | (dx * dx + dy * dy + dz * dz <= fd[j] * (1.0 + 1e-9));
        m |= (__ballot(may) != 0 && c0 + j < n_coils) ? 1u << j : 0u;
    }
    return m;
}

// Calls with fewer points than kNearSplitPoints split each float record's thickness rows over kRecordSplit lanes.
constexpr int64_t kNearSplitPoints = (int64_t)1 << 17;

// The records of each key (points with near pairs only; the coil loop is wave-uniform, so each key's count in a wave is
// one ballot and one atomic). A block counts its points' keys in LDS where they fit (near_count_keys) and adds them up
// at its end, in some thousand blocks: an atomic on the key per wave made 16,000 on one coil's few keys wait for one
// another (a thin coil of 48 nodes, 2^20 points: counting and placing 542 us; now 270).
constexpr int kCountBlocks = 1024;
__host__ __device__ inline bool near_count_keys(const FieldParams &p) { return p.n_keys <= 10240; }   // 40 KB
__global__ __launch_bounds__(256) void near_count_kernel(FieldParams p)
{
    extern __shared__ uint32_t key_counts[];
    const bool lds = near_count_keys(p);
    if (lds) {
        for (int i = threadIdx.x; i < p.n_keys; i += 256) key_counts[i] = 0u;
        __syncthreads();
    }
    uint32_t *hist = lds ? key_counts : p.near_hist;
    const int lane = threadIdx.x & 63;
    for (int64_t vi = (int64_t)blockIdx.x * 256 + threadIdx.x; vi < p.n_pts; vi += (int64_t)gridDim.x * 256) {
        const int64_t pi = p.order ? (int64_t)p.order[vi] : vi;   // the field kernel's visit order
        if (p.near_counts[pi] == 0) continue;
        const double px = p.pts[3 * pi], py = p.pts[3 * pi + 1], pz = p.pts[3 * pi + 2];
        // coils in ascending order, skipping those no point of the wave can be a record of
        for (int c0 = 0; c0 < p.n_coils; c0 += 8)
            for (uint32_t cand = record_candidates(p.coils, p.n_coils, c0, px, py, pz); cand; cand &= cand - 1) {
                const CoilDev &c = p.coils[c0 + __builtin_ctz(cand)];
                double z, r, cph, sph;
                to_local(c, px, py, pz, z, r, cph, sph);
                const int kind = record_kind(p, c, z, r, p.q & (Q_G | Q_GJ));   // the field kernel's test, bitwise
                const uint32_t key = kind < 0 ? 0u : record_key(p, c, kind, z, r);
                uint64_t todo = __ballot(kind >= 0);
                while (todo) {
                    const uint32_t k = __builtin_amdgcn_readfirstlane(__shfl(key, __builtin_ctzll(todo)));
                    const uint64_t m = __ballot(kind >= 0 && key == k);
                    if (lane == __builtin_ctzll(m)) atomicAdd(&hist[k], (unsigned)__popcll(m));
                    todo &= ~m;
                }
            }
    }
    if (!lds) return;
    __syncthreads();
    for (int i = threadIdx.x; i < p.n_keys; i += 256)
        if (key_counts[i]) atomicAdd(&p.near_hist[i], key_counts[i]);
}

// One workgroup: cursor = exclusive prefix sum of near_hist over the keys, each padded to key_align, and the call's
// total. Four keys per thread and iteration, scanned by waves: a call's few thousand keys (coils x rule classes) take two
// iterations.
constexpr int kKeyScanThreads = 1024;
__global__ __launch_bounds__(kKeyScanThreads) void near_key_scan_kernel(FieldParams p)
{
    __shared__ uint32_t wsum[kKeyScanThreads / 64];
    __shared__ uint32_t n_fp64;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nk = p.n_keys + 1;
    const int k_fp64 = p.n_slots * p.n_coils;   // the kind-0 keys come first, and of those the split ones
    const int k_split = (p.n_slots == kRuleClasses ? kSplitSlots : 1) * p.n_coils;
    const unsigned long long total = (unsigned long long)(p.near_offsets[p.n_pts - 1] + p.near_counts[p.n_pts - 1]);
    const bool overflow = total > (unsigned long long)p.near_cap;
    if (t == 0) n_fp64 = 0u;
    uint32_t carry = 0, fp64 = 0;
    for (int base = 0; base < nk; base += 4 * kKeyScanThreads) {
        const int i0 = base + 4 * t;
        uint32_t v[4], pad[4], own = 0;
        for (int k = 0; k < 4; ++k) {
            v[k] = i0 + k < p.n_keys ? p.near_hist[i0 + k] : 0u;
            pad[k] = (0u - v[k]) & (key_align(p, i0 + k) - 1u);
            own += v[k] + pad[k];
            if (i0 + k < k_fp64) fp64 += v[k];
        }
        uint32_t incl = own;   // inclusive scan of the wave's threads
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t add = __shfl_up(incl, d, 64);
            if (lane >= d) incl += add;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (int w = 0; w < kKeyScanThreads / 64; ++w) {
            if (w < wave) before += wsum[w];
            all += wsum[w];
        }
        uint32_t run = carry + before + incl - own;
        for (int k = 0; k < 4; ++k) {
            if (i0 + k == k_split) p.near_state->split_end = run;
            if (i0 + k == k_fp64) p.near_state->fp64_end = run;
            if (i0 + k < nk) p.near_cursor[i0 + k] = run;
            run += v[k];
            if (!overflow)   // else the arrays may not reach there, and nothing reads them
                for (uint32_t i = 0; i < pad[k]; ++i) p.near_keys[run + i] = kNoKey;
            run += pad[k];
        }
        carry += all;
        __syncthreads();
    }
    if (fp64) atomicAdd(&n_fp64, fp64);
    __syncthreads();
    if (t == 0) {
        p.near_state->total = total;
        p.near_state->overflow = overflow ? 1u : 0u;
        p.near_state->fp64 = n_fp64;
        p.near_state->end = carry;
    }
}

// Coils of a block row of near_fill_kernel: a multiple of record_candidates' eight.
__host__ __device__ inline int fill_coils_per_row(int n_coils, int rows) { return ((n_coils + rows - 1) / rows + 7) / 8 * 8; }

__global__ __launch_bounds__(256) void near_fill_kernel(FieldParams p)
{
    if (p.near_state->overflow) return;
    const int64_t vi = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (vi >= p.n_pts) return;
    const int64_t pi = p.order ? (int64_t)p.order[vi] : vi;
    const int64_t count = p.near_counts[pi];
    if (count == 0) return;
    const uint64_t places = p.near_state->end;
    const double px = p.pts[3 * pi], py = p.pts[3 * pi + 1], pz = p.pts[3 * pi + 2];
    int64_t slot = p.near_offsets[pi];
    const int64_t end = slot + count;
    const uint64_t hi = (uint64_t)pi << 32;
    const int lane = threadIdx.x & 63;
    bool bad = false;
    // coils in ascending order (a point's slots follow its coils), skipping those no point of the wave can be a
    // record of. Block row y takes its share of the coils; the slots before it are counted again, a fifth of the work
    const int per = fill_coils_per_row(p.n_coils, gridDim.y), first = blockIdx.y * per, last = min(first + per, p.n_coils);
    for (int c0 = 0; c0 < first; c0 += 8)
        for (uint32_t cand = record_candidates(p.coils, p.n_coils, c0, px, py, pz); cand; cand &= cand - 1) {
            const CoilDev &c = p.coils[c0 + __builtin_ctz(cand)];
            double z, r, cph, sph;
            to_local(c, px, py, pz, z, r, cph, sph);
            slot += record_kind(p, c, z, r, p.q & (Q_G | Q_GJ)) >= 0 ? 1 : 0;
        }
    for (int c0 = first; c0 < last; c0 += 8) {
        for (uint32_t cand = record_candidates(p.coils, p.n_coils, c0, px, py, pz); cand; cand &= cand - 1) {
            const CoilDev &c = p.coils[c0 + __builtin_ctz(cand)];
            double z, r, cph, sph;
            to_local(c, px, py, pz, z, r, cph, sph);
            const int kind = record_kind(p, c, z, r, p.q & (Q_G | Q_GJ));   // the field kernel's test, bitwise
            // the wave's records of one key take consecutive places from one atomic on the key's cursor; the keys'
            // leading lanes issue theirs together, so a coil costs one round trip
            const uint32_t key = kind < 0 ? 0u : record_key(p, c, kind, z, r);
            uint64_t todo = __ballot(kind >= 0), same = 0;
            while (todo) {
                const uint32_t k = __builtin_amdgcn_readfirstlane(__shfl(key, __builtin_ctzll(todo)));
                const bool mine = kind >= 0 && key == k;
                const uint64_t m = __ballot(mine);
                if (mine) same = m;
                todo &= ~m;
            }
            const int leader = kind < 0 ? lane : __builtin_ctzll(same);
            uint32_t base = 0;
            if (kind >= 0 && lane == leader) base = atomicAdd(&p.near_cursor[key], (unsigned)__popcll(same));
            base = __shfl(base, leader);
            if (kind >= 0) {
                const uint64_t pos = base + (uint64_t)__popcll(same & ((1ull << lane) - 1ull));
                // a pair classified differently from the series or field kernel: report it, write nothing
                if (slot >= end || pos >= places) {
                    bad = true;
                    continue;
                }
                p.near_keys[pos] = key;
                p.near_recs[pos] = hi | (uint64_t)slot;
                ++slot;
            }
        }
    }
    if (bad || (last == p.n_coils && slot != end)) atomicOr(&p.near_state->mismatch, 1u);
}

// Pointers to data that no kernel writes, in the constant address space: what a wave loads through them uniformly is a
// scalar load also where the kernel stores in between.
template <typename T> __device__ inline const T *constant(const T *p)
{
    return (const T *)(const T __attribute__((address_space(4))) *)(uintptr_t)p;
}
__device__ inline Tables constant(const Tables &t)
{
    return {constant(t.x), constant(t.w), constant(t.cosv), constant(t.omc), constant(t.xf), constant(t.wf), constant(t.cosf),
            constant(t.omcf), constant(t.rcos), constant(t.rsin), constant(t.wcos), constant(t.wcosf), constant(t.opc),
            constant(t.opcf), constant(t.ws), constant(t.ws2), constant(t.wcs), constant(t.wcsf), constant(t.leg)};
}

// Sum over the S lanes of a record by a fixed xor butterfly, so every lane of the group holds the same sum.
__device__ inline void reduce_record(Local &L, int S)
{
    for (int m = 1; m < S; m <<= 1) {
        L.A += __shfl_xor(L.A, m, 64);
        L.Bh += __shfl_xor(L.Bh, m, 64);
        L.Bz += __shfl_xor(L.Bz, m, 64);
        L.RP += __shfl_xor(L.RP, m, 64);
        L.RR += __shfl_xor(L.RR, m, 64);
        L.RZ += __shfl_xor(L.RZ, m, 64);
        L.ZZ += __shfl_xor(L.ZZ, m, 64);
    }
}

// Records sorted by rule class and coil. S consecutive lanes of a wave take one record (thickness rows sub, sub + S,
// ...); its value goes to the record's slot. FLOAT: the kind-1 records by the float rule, at 5 waves per SIMD as
// field_kernel's float instances, S = kRecordSplit in calls with few points, where the records are too few to fill the
// chip one lane each; else the kind-0 records by the FP64 rule, S = kRecordSplit for the split ones (record_slot) and 1
// for the others, whose rules have at most a few hundred nodes. S follows from the record and the call's shape alone, so
// a record's value does not depend on its wave.
template <bool WA, bool WB, bool WG, bool FLOAT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(FLOAT ? 5 : WA && (WB || WG) ? 2 : 3)))
void near_eval_kernel(FieldParams p)
{
    if (p.near_state->overflow) return;
    const CoilDev *coils = constant(p.coils);
    const uint32_t *near_coil = constant(p.near_coil);
    const Tables tab = constant(p.tab);
    const int64_t total = (int64_t)p.near_state->total, fp64_end = (int64_t)p.near_state->fp64_end;
    // places [first, first + n_split) hold split records, those from there to hi one a lane; the waves of split records
    // come first, and the last wave of either is part empty
    const int64_t first = FLOAT ? fp64_end : 0, hi = FLOAT ? (int64_t)p.near_state->end : fp64_end;
    const int64_t n_split = FLOAT ? (p.n_pts < kNearSplitPoints ? hi - first : 0) : (int64_t)p.near_state->split_end;
    const int64_t split_waves = (n_split * kRecordSplit + 63) >> 6;
    const int64_t waves = split_waves + ((hi - first - n_split + 63) >> 6);
    const int lane = (int)(threadIdx.x & 63);
    // the bounded grid strides over the waves' worth of records there are; the bounds are wave-uniform
    for (int64_t wave = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6; wave < waves; wave += (int64_t)gridDim.x * 4) {
        const int S = __builtin_amdgcn_readfirstlane(wave < split_waves ? kRecordSplit : 1), sub = lane % S;
        const int64_t e = S > 1 ? first + wave * (64 / kRecordSplit) + lane / kRecordSplit
                                : first + n_split + ((wave - split_waves) << 6) + lane;
        if (e >= (S > 1 ? first + n_split : hi)) continue;
        const uint32_t key = p.near_keys[e];
        if (key == kNoKey) continue;
        const uint64_t rec = p.near_recs[e];
        const int64_t pi = (int64_t)(rec >> 32), slot = (int64_t)(rec & 0xffffffffu);
        // only a near_fill that reported a mismatch leaves records unwritten; never follow one out of bounds
        if (pi >= p.n_pts || slot >= total) continue;
        // A wave holds one key's records or, where keys are not padded, those of several: it takes its keys one at a
        // time (the key of the lowest lane still to do, read into a scalar register), and every lane evaluates that
        // coil at its point, keeping the value only if the key is its own. The control flow stays uniform and the coils
        // and tables are in constant memory to the compiler, so that their loads are scalar, as in field_kernel,
        // whatever the loop stores; a divergent branch would take the same issue time. todo is wave-uniform and loses
        // at least one lane on every pass; a group's lanes share their key, so a group is always active as a whole.
        const double px = p.pts[3 * pi], py = p.pts[3 * pi + 1], pz = p.pts[3 * pi + 2];
        Cart acc;
        for (int j = 0; j < 3; ++j) { acc.A[j] = 0.0; acc.E[j] = 0.0; acc.B[j] = 0.0; }
        for (int j = 0; j < 9; ++j) acc.G[j] = 0.0;
        uint64_t todo = __ballot(1);
        while (todo) {
            const uint32_t k = __builtin_amdgcn_readfirstlane(__shfl(key, __builtin_ctzll(todo)));
            const bool mine = key == k;
            todo &= ~(uint64_t)__ballot(mine);
            // only a reported mismatch can leave a key outside the range's kind
            const uint32_t slot_of = k / (uint32_t)p.n_coils;
            if (k >= (uint32_t)p.n_keys || (slot_of == (uint32_t)p.n_slots) != FLOAT) continue;
            const CoilDev &c = coils[near_coil[k - slot_of * (uint32_t)p.n_coils]];
            double z, r, cph, sph;
            to_local(c, px, py, pz, z, r, cph, sph);
            // FP64 records take their rule classes one at a time too (a slot holds one class, but for the coils of few
            // rows): the rule's node sets stay uniform, hence scalar loads
            const int cls = FLOAT ? 0 : rule_class(c, z, r);
            uint64_t left = __ballot(mine);
            while (left) {
                const int q = FLOAT ? 0 : __builtin_amdgcn_readfirstlane(__shfl(cls, __builtin_ctzll(left)));
                const bool sel = mine && cls == q;
                left &= ~(uint64_t)__ballot(sel);
                Local L;
                if (FLOAT) eval_stable<float, WA, WB, WG>(c, tab, full_rule(c), z, r, sub, S, 0, 1, L);
                else eval_stable<f64s, WA, WB, WG>(c, tab, class_rule(c, q), z, r, sub, S, 0, 1, L);
                reduce_record(L, S);
                if (sel) accumulate_global(c, L, r, cph, sph, p.q, acc);
            }
        }
        if (sub == 0) {
            double *o = p.near_vals + slot * p.near_width;
            if (p.A) { for (int j = 0; j < 3; ++j) o[j] = acc.A[j]; o += 3; }
            if (p.E) { for (int j = 0; j < 3; ++j) o[j] = acc.E[j]; o += 3; }
            if (p.B) { for (int j = 0; j < 3; ++j) o[j] = acc.B[j]; o += 3; }
            if (p.G) for (int j = 0; j < 9; ++j) o[j] = acc.G[j];
        }
    }
}

// The kind-0 records of calls with few of them: a group of consecutive lanes takes a record of its own coil and rule
// class, a whole wave for the first `split` of them (kGroupSplit nodes or more) and kRecordSplit lanes for the others.
// The lanes split the rows in four (two) and the rows' nodes: 80 x 20 nodes take 25 steps of a wave. Coil and tables
// are vector loads; a wave takes as long as its longest record, and the records are sorted by node count.
template <bool WA, bool WB, bool WG>
__global__ __launch_bounds__(256) void near_eval_group_kernel(FieldParams p)
{
    if (p.near_state->overflow) return;
    const int64_t n_split = (int64_t)p.near_state->split_end, fp64 = (int64_t)p.near_state->fp64_end;   // no padding
    const int64_t waves = n_split + (fp64 - n_split + 64 / kRecordSplit - 1) / (64 / kRecordSplit);
    const int lane = (int)(threadIdx.x & 63);
    // a bounded grid strides over the waves' worth of records; the bound is wave-uniform
    for (int64_t wave = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6; wave < waves; wave += (int64_t)gridDim.x * 4) {
        const int group = __builtin_amdgcn_readfirstlane(wave < n_split ? 64 : kRecordSplit);
        const int sub = lane % group;
        const int64_t e = group == 64 ? wave : n_split + (wave - n_split) * (64 / kRecordSplit) + lane / kRecordSplit;
        if (e >= fp64) continue;   // whole groups, in the last wave only
        const uint32_t key = p.near_keys[e];
        const uint64_t rec = p.near_recs[e];
        const int64_t pi = (int64_t)(rec >> 32), slot = (int64_t)(rec & 0xffffffffu);
        // only a near_fill that reported a mismatch leaves records unwritten; never follow one out of bounds
        if (pi >= p.n_pts || slot >= (int64_t)p.near_state->total || key >= (uint32_t)(p.n_slots * p.n_coils)) continue;
        const CoilDev &c = p.coils[p.near_coil[key % (uint32_t)p.n_coils]];
        double z, r, cph, sph;
        to_local(c, p.pts[3 * pi], p.pts[3 * pi + 1], p.pts[3 * pi + 2], z, r, cph, sph);
        const RuleSel rule = class_rule(c, rule_class(c, z, r));
        Local L;
        if (group == 64) {
            // one record: the wave's control flow and loads are uniform
            const int k = __builtin_amdgcn_readfirstlane(key);
            const CoilDev &cu = p.coils[p.near_coil[(uint32_t)k % (uint32_t)p.n_coils]];
            eval_wave<WA, WB, WG>(cu, p.tab, class_rule(cu, __builtin_amdgcn_readfirstlane(rule_class(c, z, r))), z, r, lane,
                                  0, 1, L);
        } else {
            const int sr = rule.nt == 1 ? 1 : 2;
            eval_shared<WA, WB, WG>(c, p.tab, rule, z, r, sub & (sr - 1), sr, sub / sr, kRecordSplit / sr, L);
            reduce_record(L, kRecordSplit);
        }
        if (sub) continue;
        Cart acc;
        for (int j = 0; j < 3; ++j) { acc.A[j] = 0.0; acc.E[j] = 0.0; acc.B[j] = 0.0; }
        for (int j = 0; j < 9; ++j) acc.G[j] = 0.0;
        accumulate_global(c, L, r, cph, sph, p.q, acc);
        double *o = p.near_vals + slot * p.near_width;
        if (p.A) { for (int j = 0; j < 3; ++j) o[j] = acc.A[j]; o += 3; }
        if (p.E) { for (int j = 0; j < 3; ++j) o[j] = acc.E[j]; o += 3; }
        if (p.B) { for (int j = 0; j < 3; ++j) o[j] = acc.B[j]; o += 3; }
        if (p.G) for (int j = 0; j < 9; ++j) o[j] = acc.G[j];
    }
}

// Adds each point's slots to its outputs, in slot order. Points in index order: slots and outputs lie in that order, so
// that a wave reads and writes whole lines (in the visit order each point's took lines of their own: 128 coils x 2^20
// points 0.20 ms, this 0.14; 262,145 points FP32C 45 us, this 28).
__global__ __launch_bounds__(256) void near_add_kernel(FieldParams p)
{
    if (p.near_state->overflow) return;
    const int64_t pi = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (pi >= p.n_pts) return;
    const int64_t count = p.near_counts[pi];
    if (count == 0) return;
    const int64_t e0 = p.near_offsets[pi];
    // the point's outputs are held in registers and each slot added in turn: the same order of additions as a
    // read-modify-write per slot, with one load and one store per output
    double va[3] = {}, ve[3] = {}, vb[3] = {}, vg[9] = {};
    if (p.A) for (int k = 0; k < 3; ++k) va[k] = p.A[3 * pi + k];
    if (p.E) for (int k = 0; k < 3; ++k) ve[k] = p.E[3 * pi + k];
    if (p.B) for (int k = 0; k < 3; ++k) vb[k] = p.B[3 * pi + k];
    if (p.G) for (int k = 0; k < 9; ++k) vg[k] = p.G[9 * pi + k];
    for (int64_t e = e0; e < e0 + count; ++e) {
        const double *o = p.near_vals + e * p.near_width;
        if (p.A) { for (int k = 0; k < 3; ++k) va[k] += o[k]; o += 3; }
        if (p.E) { for (int k = 0; k < 3; ++k) ve[k] += o[k]; o += 3; }
        if (p.B) { for (int k = 0; k < 3; ++k) vb[k] += o[k]; o += 3; }
        if (p.G) for (int k = 0; k < 9; ++k) vg[k] += o[k];
    }
    if (p.A) for (int k = 0; k < 3; ++k) p.A[3 * pi + k] = va[k];
    if (p.E) for (int k = 0; k < 3; ++k) p.E[3 * pi + k] = ve[k];
    if (p.B) for (int k = 0; k < 3; ++k) p.B[3 * pi + k] = vb[k];
    if (p.G) for (int k = 0; k < 9; ++k) p.G[9 * pi + k] = vg[k];
}

// Exclusive prefix sum of the per-point counts in three kernels (tile sums, a one-workgroup scan of the tile sums,
// the tiles' own scans): only kernel launches, so a caller may capture it in a graph, and deterministic.
constexpr int kScanPerThread = 16;
constexpr int kScanTile = 256 * kScanPerThread;

__device__ inline int64_t block_exclusive_scan(int64_t v, int64_t *lds, int64_t &total)
{
    const int t = threadIdx.x;
    lds[t] = v;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
        const int64_t add = t >= d ? lds[t - d] : 0;
        __syncthreads();
        lds[t] += add;
        __syncthreads();
    }
    const int64_t incl = lds[t];
    total = lds[255];
    __syncthreads();
    return incl - v;
}

__global__ __launch_bounds__(256) void scan_tile_sums_kernel(const int64_t *counts, int64_t n, int64_t *sums)
{
    __shared__ int64_t lds[256];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPerThread;
    int64_t v = 0;
    for (int k = 0; k < kScanPerThread; ++k)
        if (base + k < n) v += counts[base + k];
    int64_t total;
    (void)block_exclusive_scan(v, lds, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void scan_sums_kernel(int64_t *sums, int64_t nb)
{
    __shared__ int64_t lds[256];
    int64_t carry = 0;
    for (int64_t base = 0; base < nb; base += 256) {
        const int64_t i = base + threadIdx.x;
        const int64_t v = i < nb ? sums[i] : 0;
        int64_t total;
        const int64_t ex = block_exclusive_scan(v, lds, total);
        if (i < nb) sums[i] = carry + ex;
        carry += total;
    }
}

// sums: the tiles' sums, scanned already or (raw) each tile's block adding those before it.
__global__ __launch_bounds__(256) void scan_tiles_kernel(const int64_t *counts, int64_t n, const int64_t *sums, int raw,
                                                         int64_t *offsets)
{
    __shared__ int64_t lds[256];
    int64_t before = 0;
    if (raw && blockIdx.x > 0) {
        int64_t v = 0;
        for (unsigned i = threadIdx.x; i < blockIdx.x; i += 256) v += sums[i];
        (void)block_exclusive_scan(v, lds, before);
    } else if (!raw) {
        before = sums[blockIdx.x];
    }
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPerThread;
    int64_t v[kScanPerThread], t = 0;
    for (int k = 0; k < kScanPerThread; ++k) {
        v[k] = base + k < n ? counts[base + k] : 0;
        t += v[k];
    }
    int64_t total;
    int64_t run = before + block_exclusive_scan(t, lds, total);
    for (int k = 0; k < kScanPerThread; ++k) {
        if (base + k < n) offsets[base + k] = run;
        run += v[k];
    }
}

hipError_t near_scan(hipStream_t s, const int64_t *counts, int64_t *offsets, int64_t n, void *temp,
                     size_t &temp_bytes)
{
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    if (!temp) {
        temp_bytes = sizeof(int64_t) * (size_t)(nb > 0 ? nb : 1);
        return hipSuccess;
    }
    if (n <= 0) return hipSuccess;
    int64_t *sums = (int64_t *)temp;
    // Up to kScanRaw tiles (eight loads a thread) a tile's block adds the sums before it itself, and one tile needs none:
    // two launches or one in place of three, some 4 us each.
    constexpr int64_t kScanRaw = 2048;
    const int raw = nb <= kScanRaw ? 1 : 0;
    if (nb > 1) hipLaunchKernelGGL(scan_tile_sums_kernel, dim3((unsigned)nb), dim3(256), 0, s, counts, n, sums);
    if (!raw) hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(256), 0, s, sums, nb);
    hipLaunchKernelGGL(scan_tiles_kernel, dim3((unsigned)nb), dim3(256), 0, s, counts, n, (const int64_t *)sums, raw,
                       offsets);
    return hipGetLastError();
}

void launch_near_key_scan(hipStream_t s, const FieldParams &p)
{
    if (p.n_pts <= 0) return;
    hipLaunchKernelGGL(near_key_scan_kernel, dim3(1), dim3(kKeyScanThreads), 0, s, p);
}

void launch_near_count(hipStream_t s, const FieldParams &p)
{
    if (p.n_pts <= 0) return;
    const unsigned blocks = (unsigned)((p.n_pts + 255) / 256);
    if (near_count_keys(p))
        hipLaunchKernelGGL(near_count_kernel, dim3(std::min<unsigned>(blocks, kCountBlocks)), dim3(256),
                           sizeof(uint32_t) * (size_t)p.n_keys, s, p);
    else
        hipLaunchKernelGGL(near_count_kernel, dim3(blocks), dim3(256), 0, s, p);
}

void launch_near_fill(hipStream_t s, const FieldParams &p)
{
    if (p.n_pts <= 0) return;
    // A wave takes its coils in turn, about half a microsecond each, so that few points leave the chip to that chain:
    // rows of at least 8 coils up to eight blocks a CU (128 coils x 16,411 points: 74 us in one row, 34 in eight;
    // 262,145 points, FP32C: 81 in one, 73 in two).
    const int64_t blocks = (p.n_pts + 255) / 256;
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>({8, (p.n_coils + 7) / 8, (2048 + blocks - 1) / blocks}));
    const int per = fill_coils_per_row(p.n_coils, (int)most);
    hipLaunchKernelGGL(near_fill_kernel, dim3((unsigned)blocks, (unsigned)((p.n_coils + per - 1) / per)), dim3(256), 0, s, p);
}

template <bool FLOAT>
static void launch_near_eval_g(hipStream_t s, const FieldParams &p, unsigned blocks)
{
    const bool wa = p.q & (Q_A | Q_E), wb = p.q & Q_B, wg = p.q & (Q_G | Q_GJ);
    const dim3 g(blocks), b(256);
    switch ((wa ? 4 : 0) | (wb ? 2 : 0) | (wg ? 1 : 0)) {
        case 1: hipLaunchKernelGGL((near_eval_kernel<false, false, true, FLOAT>), g, b, 0, s, p); break;
        case 2: hipLaunchKernelGGL((near_eval_kernel<false, true, false, FLOAT>), g, b, 0, s, p); break;
        case 3: hipLaunchKernelGGL((near_eval_kernel<false, true, true, FLOAT>), g, b, 0, s, p); break;
        case 4: hipLaunchKernelGGL((near_eval_kernel<true, false, false, FLOAT>), g, b, 0, s, p); break;
        case 5: hipLaunchKernelGGL((near_eval_kernel<true, false, true, FLOAT>), g, b, 0, s, p); break;
        case 6: hipLaunchKernelGGL((near_eval_kernel<true, true, false, FLOAT>), g, b, 0, s, p); break;
        default: hipLaunchKernelGGL((near_eval_kernel<true, true, true, FLOAT>), g, b, 0, s, p); break;
    }
}

static void launch_near_eval_group(hipStream_t s, const FieldParams &p, unsigned blocks)
{
    const bool wa = p.q & (Q_A | Q_E), wb = p.q & Q_B, wg = p.q & (Q_G | Q_GJ);
    const dim3 g(blocks), b(256);
    switch ((wa ? 4 : 0) | (wb ? 2 : 0) | (wg ? 1 : 0)) {
        case 1: hipLaunchKernelGGL((near_eval_group_kernel<false, false, true>), g, b, 0, s, p); break;
        case 2: hipLaunchKernelGGL((near_eval_group_kernel<false, true, false>), g, b, 0, s, p); break;
        case 3: hipLaunchKernelGGL((near_eval_group_kernel<false, true, true>), g, b, 0, s, p); break;
        case 4: hipLaunchKernelGGL((near_eval_group_kernel<true, false, false>), g, b, 0, s, p); break;
        case 5: hipLaunchKernelGGL((near_eval_group_kernel<true, false, true>), g, b, 0, s, p); break;
        case 6: hipLaunchKernelGGL((near_eval_group_kernel<true, true, false>), g, b, 0, s, p); break;
        default: hipLaunchKernelGGL((near_eval_group_kernel<true, true, true>), g, b, 0, s, p); break;
    }
}

// The grid covers the capacity at `lanes` lanes a place up to kEvalBlocks blocks, some eight times what the chip holds at
// once, and strides beyond. (A wave that finds no record costs a nanosecond: 75,000 of them, for the default
// capacity of 262,145 points and hardly any record, took 75 us. And the capacity can pass the 2^32 threads of a launch,
// 2^29 records split over eight lanes, which then runs what is left over, without an error.)
constexpr int64_t kEvalBlocks = 16384;
static unsigned near_eval_blocks(const FieldParams &p, int lanes)
{
    return (unsigned)std::min<int64_t>((record_places(p, p.near_cap) * lanes + 255) / 256, kEvalBlocks);
}

void launch_near_eval(hipStream_t s, const FieldParams &p)
{
    if (p.near_cap <= 0) return;
    if (uniform_records(p)) launch_near_eval_g<false>(s, p, near_eval_blocks(p, kRecordSplit));
    else launch_near_eval_group(s, p, (unsigned)std::min<int64_t>((p.near_cap + 3) / 4, 8192));
    if (p.float_records) launch_near_eval_g<true>(s, p, near_eval_blocks(p, p.n_pts < kNearSplitPoints ? kRecordSplit : 1));
}

void launch_near_add(hipStream_t s, const FieldParams &p)
{
    if (p.n_pts <= 0) return;
    hipLaunchKernelGGL(near_add_kernel, dim3((unsigned)((p.n_pts + 255) / 256)), dim3(256), 0, s, p);
}

}  // namespace ccoil
