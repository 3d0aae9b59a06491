// Kernel parameter blocks and launcher declarations (host <-> device contract inside the library).
#pragma once

#include "common.hpp"

namespace ccoil {

// Arithmetic of the quadrature (values of the C ABI precision argument).
enum { kFP64 = 0, kFP32C = 1, kFP32 = 2, kFP64Reference = 3, kFP64IEEE = 4 };
constexpr int kFP64Own = 5;   // field kernels: kFP64's arithmetic at the coils' own nodes (field_rule)
constexpr int kFieldBlock = 256;

// Device-side outcome of the FP32C near pass (read back by the host once the call's work is done).
struct NearState {
    unsigned long long total;   // records (deferred (coil, point) pairs) counted by field_kernel
    unsigned int overflow;      // total > near_cap: the pass was skipped
    unsigned int mismatch;      // near_fill classified a pair differently from field_kernel
    unsigned long long fp64;    // records of kind 0 (FP64 rule)
    // places in the record arrays (the keys' padding counts): the ends of the records of kind 0 that are split over more
    // lanes (the first ones), of kind 0, and of all
    unsigned long long split_end, fp64_end, end;
};

struct FieldParams {
    const CoilDev *coils;
    int32_t n_coils;
    const double *pts;     // AoS xyz
    int64_t n_pts;
    double *A, *E, *B, *G; // AoS outputs (NULL = not requested)
    uint32_t q;            // Q_* mask
    Tables tab;
    int32_t near_fp64;     // FP32C: skip near pairs here, re-evaluate in FP64
    // Rule records (the series modes, large calls): field_kernel evaluates only the series and defers every other
    // (coil, point) pair to the record pass below, which runs the rule on waves of one coil each. A record's kind is
    // 0 for the FP64 rule (FP32C's near pairs; every rule pair in FP64) and 1 for the float rule (FP32C's others);
    // its key, a slot and a coil, is record_key below; n_keys = n_coils * (n_slots + float_records).
    int32_t rule_records;
    int32_t float_records;
    int32_t n_slots;       // key slots of a coil's FP64 records: kRuleClasses, 4 or 2 (record_slot)
    int32_t n_keys;
    // The far field (FP32C, FP64 with CCOIL_FAR_FIELD): each coil's moments (n_coils * kMpCoil doubles, multipole.hpp); a
    // coil with CoilDev::far_d2 > 0 takes its series beyond that distance. NULL: no coil does.
    const double *mp;
    // The order the points are visited in (a spatial sort, so the points of a wave lie close together and a wave
    // mostly takes one branch per coil); NULL: index order. No result depends on it.
    const uint32_t *order;
    // Record pass, stream-ordered with no host readback (so a caller may capture it in a graph): field_kernel counts
    // each point's records (near_counts); an exclusive scan of near_counts gives each point's places in near_vals
    // (near_offsets); near_count, or the series kernel, counts the records of each key (near_hist; coils by
    // CoilDev::near_key, those with the most nodes first); near_key_scan turns near_hist into cursors per key, and stores
    // the total and whether it exceeds near_cap in near_state; near_fill places one record per (coil, point) pair at
    // its key's cursor: the key (near_keys) and point << 32 | place (near_recs); near_eval writes each record's
    // contribution into its place of near_vals (near_width doubles: the requested A, E, B, G in that order);
    // near_add adds a point's values in the order of their places, which is the coils'. The order of records within a
    // key varies from run to run, but a value depends only on its (coil, point) and every sum has a fixed order, so
    // results are bitwise reproducible. When the total exceeds near_cap, near_fill, near_eval and near_add do nothing
    // and the host grows the buffers and runs them again.
    int64_t *near_counts;
    const int64_t *near_offsets;
    uint32_t *near_hist;      // [n_keys + 1] counts per key
    uint32_t *near_cursor;    // [n_keys + 1] next free record of each key
    NearState *near_state;
    int64_t near_cap;
    uint32_t *near_keys;      // record_places(near_cap) keys and records
    const uint32_t *near_coil;               // near_key -> coil index
    uint64_t *near_recs;
    double *near_vals;
    int32_t near_width;
    // Coil chunks (grid y): each block row sums its chunk of coils into partial ([chunk][point][width]: the
    // requested outputs A, E, B, G in that order, 3 or 9 doubles each) and field_reduce_kernel adds the chunks in
    // order.
    int32_t coils_per_chunk;
    int32_t n_chunks;
    int32_t partial_width;
    double *partial;
};

constexpr int64_t kUniformRecordPoints = (int64_t)1 << 17;

// What becomes of a (coil, point) pair: -1 field_kernel evaluates it (the series beyond the far-field distance, or
// the rule in the kernel), 0 an FP64-rule record, 1 a float-rule record. field_kernel, near_count and near_fill all
// classify with this, bitwise alike (to_local and the tests round operation by operation).
__device__ inline int record_kind(const FieldParams &p, const CoilDev &c, double z, double r, bool axis)
{
    if (is_far(c, z, r)) return -1;
    const bool near = p.near_fp64 && is_near(c, z, r, axis);
    if (p.rule_records) return (p.float_records && !near) ? 1 : 0;
    return near ? 0 : -1;
}

// Whether near_eval gives each wave one coil and class at a time (uniform control flow, scalar loads: calls whose
// records are many per key) or each group of lanes its own record (calls with few records, where a wave would hold a
// dozen keys and take them in series: 128 coils at 16,411 points measured 640 us that way, 60 us in groups, while at
// 2^20 points the groups' vector loads are the slower way).
__host__ __device__ inline bool uniform_records(const FieldParams &p)
{
    return p.n_pts >= kUniformRecordPoints;
}

// The sort key of a record: slot, then coil (most nodes first). FP64 records whose serial chain of nodes would outlast
// the rest of the launch come first, and near_eval splits them over more lanes; with two slots that is all. Else
// uniform records are sorted by rule class, the costliest first, so that a wave holds one coil's records of one
// class: the split ones, with the coil's own angular rule and at least kRecordSplit thickness rows of a coil's
// kSplitRows, take the first kSplitSlots slots. (One row a lane leaves more to the set-up and the sum over the lanes than
// it saves: 40 coils of 40 x 10 nodes, 131,072 points, FP32C: 114 us split, 98 not.) Grouped records are sorted by their
// node count in steps of four, the split ones with kGroupSplit nodes or more. Float records follow by coil.
constexpr int kRecordSplit = 8;
constexpr int kSplitRows = 13;
constexpr int kSplitSlots = kRedThk;
constexpr int kGroupSplit = 640;
static_assert(kRedThkN[kRedThk - 1] < kRecordSplit && kRedThkN[kRedThk - 2] >= kRecordSplit, "record_slot");
__device__ inline uint32_t record_slot(const FieldParams &p, const CoilDev &c, int kind, double z, double r)
{
    if (kind) return (uint32_t)p.n_slots;
    const int cls = rule_class(c, z, r);
    if (uniform_records(p)) {
        const int k = cls / (kRedThk + 1), t = cls - k * (kRedThk + 1);
        const bool rows = t == 0 ? c.n_thk >= kRecordSplit : t < kRedThk;   // at least kRecordSplit
        const bool split = k == 0 && rows && c.n_thk >= kSplitRows;
        if (p.n_slots == 2) return split ? 0u : 1u;
        return (uint32_t)(split || (k > 0 && rows) ? cls : k * (kRedThk + 1) + kRedThk);
    }
    const RuleSel s = class_rule(c, cls);
    const int n = s.na * s.nt;
    if (p.n_slots == 2) return n >= kGroupSplit ? 0u : 1u;
    return n >= kGroupSplit ? 0u : n >= kGroupSplit / 4 ? 1u : n >= kGroupSplit / 16 ? 2u : 3u;
}
// Uniform records of all slots start each key at a wave of its own: a wave whose records are of several keys takes them
// in turn, and where classes are rare a wave of a dozen keys and rules outlasted the rest of the launch (40 coils of
// 80 x 20 slow nodes, 131,072 points, series mode: 443 us; in waves of one key 28). key_align: the places that a key's
// records are padded to (near_key_scan marks the padding kNoKey); record_places: the places that n records may take.
constexpr uint32_t kNoKey = 0xffffffffu;
constexpr size_t kRecordBytes = sizeof(uint32_t) + sizeof(uint64_t);   // of one place: its key and its record
__host__ __device__ inline uint32_t key_align(const FieldParams &p, int key)
{
    return p.n_slots != kRuleClasses ? 1u : key < kSplitSlots * p.n_coils ? 64u / kRecordSplit : 64u;
}
__host__ __device__ inline int64_t record_places(const FieldParams &p, int64_t n)
{
    return n + (p.n_slots != kRuleClasses ? 0 : (int64_t)64 * p.n_keys);
}
__device__ inline uint32_t record_key(const FieldParams &p, const CoilDev &c, int kind, double z, double r)
{
    return record_slot(p, c, kind, z, r) * (uint32_t)p.n_coils + (uint32_t)c.near_key;
}

// Adjoint of the summed B field: per-coil gradients of sum_x dL/dB(x) . B(x), 9 per coil in the order
// current, R, a, b, px, py, pz, alpha, beta. Grid: (point blocks, coils); partial sums per (coil, block).
constexpr int kGradTerms = 9;
struct GradParams {
    const CoilDev *coils;
    int32_t n_coils;
    const double *pts;     // AoS xyz
    int64_t n_pts;
    const double *gB;      // dL/dB, AoS (global frame)
    double *partial;       // [n_coils][n_blocks][kGradTerms]
    int32_t n_blocks;
    double *grad;          // [n_coils][kGradTerms]
    Tables tab;
};
void launch_field_grad(hipStream_t s, const GradParams &p, int precision);

void launch_gl_tables(hipStream_t s, double *x, double *w, double *cosv, double *omc, float *xf, float *wf,
                      float *cosf, float *omcf, double *rcos, double *rsin);
// Per-entry products of the tables (after launch_gl_tables on the same stream): wc = w cos, opc = 1 + cos,
// ws = w (1 - cos), ws2 = w (1 - cos)^2, wcs = w cos (1 - cos) (and its float copy wcsf).
void launch_angular_tables(hipStream_t s, const double *x, const double *w, const double *cosv, const double *omc,
                           double *wc, float *wcf, double *opc, float *opcf, double *ws, double *ws2, double *wcs,
                           float *wcsf);
// Zeroes n_words 8-byte words with a kernel (no hipMemsetAsync, so callers may capture it in a graph).
void launch_fill_zero(hipStream_t s, void *p, int64_t n_words);
struct ZeroRanges {       // up to four ranges of words to zero with one launch
    void *p[4];
    int64_t n[4];
};
void launch_fill_zero(hipStream_t s, const ZeroRanges &z);
// split: 1, 4 or 16 lanes per point, or 64 (kFP64).
void launch_field(hipStream_t s, const FieldParams &p, int precision, int split);
void launch_field_reduce(hipStream_t s, const FieldParams &p);   // after launch_field when n_chunks > 1
// Resident 256-thread blocks per CU of the field kernel instance (0 if the runtime cannot tell).
int field_blocks_per_cu(uint32_t q, int precision, int split);
// Whether the series-only kernel counts the record pass's keys (in LDS, 4 bytes per coil of a chunk and slot), so
// that near_count_kernel is not launched: calls with rule records whose coil chunks fit 40 KB, where the kernel's four
// blocks per CU still share the LDS.
__host__ __device__ inline int series_key_words(const FieldParams &p)
{
    return p.coils_per_chunk * (p.n_slots + (p.float_records ? 1 : 0));
}
__host__ __device__ inline bool series_counts_keys(const FieldParams &p)
{
    return p.rule_records && series_key_words(p) <= 10240;
}
// Resident 256-thread blocks per CU of the series-only kernel (the launch of calls with rule records).
int field_series_blocks_per_cu(uint32_t q, int precision);
// Exclusive prefix sum of n counts into offsets (kernel launches only); with temp == NULL only sets temp_bytes.
hipError_t near_scan(hipStream_t s, const int64_t *counts, int64_t *offsets, int64_t n, void *temp,
                     size_t &temp_bytes);
// near_count: the records of each key into near_hist (zeroed before); near_key_scan: the keys' cursors from near_hist,
// and near_state's total, ends and overflow (one small kernel).
void launch_near_count(hipStream_t s, const FieldParams &p);
void launch_near_key_scan(hipStream_t s, const FieldParams &p);
void launch_near_fill(hipStream_t s, const FieldParams &p);
void launch_near_eval(hipStream_t s, const FieldParams &p);
void launch_near_add(hipStream_t s, const FieldParams &p);
// Far-field moments of every coil with CoilDev::far_d2 > 0 and the recurrence header, into mp.
void launch_multipole_moments(hipStream_t s, const CoilDev *coils, int n_coils, const Tables &tab, double *mp);
// The visit order: n <= cap points counting-sorted by the Morton cell of a 2^bits-per-axis grid over their bounding box.
// temp: visit_order_bytes(cap, bits, scan_bytes) bytes, scan_bytes from near_scan for 2^(3 bits) counts.
size_t visit_order_bytes(int64_t cap, int bits, size_t scan_bytes);
int64_t *visit_order_counts(void *temp, int64_t cap);   // the cells' 2^(3 bits) counts, zeroed before the launch
hipError_t launch_visit_order(hipStream_t s, const double *pts, int64_t n, int bits, void *temp, int64_t cap,
                              size_t scan_bytes, uint32_t *order);

}  // namespace ccoil
