// The autotuner: per call size, the launch shape that measured fastest on this device, kept in the context's cache
// and optionally in a text file, so that later calls (and later processes) replay the same choice.
#include "context.hpp"

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <set>
#include <sstream>

using namespace ccoil;

namespace ccoil {

namespace {

bool cache_get(ccoil_ctx ctx, const std::string &key, std::string &value)
{
    auto it = ctx->tuning.find(key);
    if (it == ctx->tuning.end()) return false;
    value = it->second;
    return true;
}

void cache_put(ccoil_ctx ctx, const std::string &key, const std::string &value)
{
    ctx->tuning[key] = value;
    if (ctx->tuning_file.empty()) return;
    std::ofstream f(ctx->tuning_file, std::ios::app);
    if (f) f << key << '\t' << value << '\n';
}

}  // namespace

ccoil_status load_tuning_file(ccoil_ctx ctx, const char *path)
{
    ctx->tuning_file = path ? path : "";
    if (!path) return CCOIL_OK;
    std::ifstream f(path);
    std::string line;
    while (f && std::getline(f, line)) {
        const size_t tab = line.find('\t');
        if (tab == std::string::npos || tab == 0) continue;
        ctx->tuning[line.substr(0, tab)] = line.substr(tab + 1);
    }
    return CCOIL_OK;
}

ccoil_status tune_fields(ccoil_ctx ctx, const ccoil_coils *coils, const double *points, int64_t n_points,
                         uint32_t quantities, int32_t precision, uint32_t flags, double *A, double *B, double *E,
                         double *G, FieldShape &out)
{
    std::vector<CoilDev> hc;
    const std::string msg = pack_coils(coils, false, (quantities & CCOIL_E) != 0, hc);
    if (!msg.empty() || n_points <= 0 || hc.empty()) {   // fields_call reports it, or has nothing to tune
        out = FieldShape();
        return CCOIL_OK;
    }
    int64_t nodes = 0;
    for (const auto &c : hc) nodes += (int64_t)c.n_ang * c.n_thk;
    std::ostringstream k;
    // far: the series' calls have kernels of their own. The kernels' version is part of the key: a shape timed with other
    // kernels is none for these (v2: reduced rules, 64 lanes per point)
    const bool far = (precision == CCOIL_FP32C && !(flags & CCOIL_DIRECT)) ||
                     (precision == CCOIL_FP64 && (flags & CCOIL_FAR_FIELD));
    k << "fields v2 n=" << n_points << " coils=" << hc.size() << " nodes=" << nodes << " q=" << quantities
      << " precision=" << precision << " far=" << far << " near=" << ((flags & CCOIL_NO_NEAR_FP64) ? 0 : 1)
      << " cu=" << ctx->cu_count;
    const std::string key = k.str();
    std::string v;
    if (cache_get(ctx, key, v) && std::sscanf(v.c_str(), "split=%d chunks=%d", &out.split, &out.chunks) == 2)
        return CCOIL_OK;
    // candidates around the rule: every lane count that can fill the chip, 1-4 coil chunks and the rule's chunks
    // with its halves and doubles
    const int64_t nc = (int64_t)hc.size();
    const FieldShape rule = field_shape_rule(ctx, n_points, hc, quantities, precision);
    std::set<std::pair<int, int>> cand;
    std::vector<int> splits = {1, 4};
    if (n_points < kSortedPoints) splits.push_back(16);
    if (n_points < kSortedPoints && precision == CCOIL_FP64) splits.push_back(64);
    for (int s : splits)
        for (int64_t c : {(int64_t)1, (int64_t)2, (int64_t)3, (int64_t)4, (int64_t)rule.chunks,
                          (int64_t)std::max(1, rule.chunks / 2), (int64_t)rule.chunks * 2})
            if (c >= 1 && c <= nc && c <= 65535) cand.insert({s, (int)c});
    cand.insert({rule.split, rule.chunks});
    double best = 1e300;
    FieldShape best_shape = rule;   // every candidate is timed, so one of them replaces it
    for (const auto &c : cand) {
        FieldShape sh;
        sh.split = c.first;
        sh.chunks = c.second;
        ccoil_report rep;
        const ccoil_status st = fields_call(ctx, coils, points, n_points, quantities, precision, flags, A, B, E, G,
                                            &rep, nullptr, &sh);
        if (st != CCOIL_OK) return st;
        if (rep.kernel_ms < best) {   // with what a shape brings along: the visit order, the sum of the chunks
            best = rep.kernel_ms;
            best_shape = sh;
        }
    }
    out = best_shape;
    std::ostringstream o;
    o << "split=" << out.split << " chunks=" << out.chunks;
    cache_put(ctx, key, o.str());
    return CCOIL_OK;
}

ccoil_status tune_pairs(ccoil_ctx ctx, const PairBuild &rule, uint32_t what, int32_t precision,
                        const std::function<ccoil_status(int64_t, double &)> &run, int64_t &target)
{
    std::ostringstream k;
    // v2, reduced: what the target counts, nodes of reduced rules or of the planned ones (build_pairs)
    const bool reduced = precision == CCOIL_FP64 && !rule.own;
    k << "pairs v2 n=" << rule.sorted.size() << " node_pairs=" << rule.node_pairs << " what=" << what
      << " precision=" << precision << " far=" << rule.far << " reduced=" << reduced << " cu=" << ctx->cu_count;
    const std::string key = k.str();
    std::string v;
    long long t = 0;
    if (cache_get(ctx, key, v) && std::sscanf(v.c_str(), "target=%lld", &t) == 1 && t > 0) {
        target = t;
        return CCOIL_OK;
    }
    double best = 1e300;
    target = rule.target;
    // the rule's own target and its neighbours within the range that is worth a launch (lane_target)
    const int64_t least = reduced ? 16 : 256, most = reduced ? 8192 : 32768;
    for (int64_t c : {rule.target / 4, rule.target / 2, rule.target, rule.target * 2}) {
        if (c != rule.target && (c < least || c > most)) continue;
        double ms = 0.0;
        const ccoil_status st = run(c, ms);
        if (st != CCOIL_OK) return st;
        if (ms < best) {
            best = ms;
            target = c;
        }
    }
    cache_put(ctx, key, "target=" + std::to_string(target));
    return CCOIL_OK;
}

}  // namespace ccoil

extern "C" ccoil_status ccoil_set_tuning_file(ccoil_ctx ctx, const char *path)
{
    if (!ctx) return fail(nullptr, CCOIL_ERR_ARGUMENT, "ccoil_set_tuning_file: ctx is NULL");
    return load_tuning_file(ctx, path);
}
