// mc_tune.cpp -- autotuner of the EM work decomposition.
//
// The options that shape the E/M kernels (reduction mode, sessions per work
// item and so sessions per lane, LDS window, lanes per work item) are picked
// for one model type and one training set by measuring graph-replayed EM
// iterations of each candidate on the device: the shape that the planner
// chooses for the set, the reduction mode, then a coordinate search over item
// size, window and workgroup size, each step keeping the fastest.  The starting
// point and the planner's shape are candidates, so the result is slower than
// neither (up to measurement noise).

#include <cstdint>
#include <string>
#include <vector>

#include "mclicks.h"
#include "mc_internal.h"
#include "mc_kernels.h"
#include "mc_model.h"

namespace mc {
namespace {

constexpr int kNumOptions = MC_N_OPTIONS;

struct Trial {
    int model_type, device;
    int64_t n, n_qd;
    const int32_t *query, *pidx;
    const uint8_t *clicks, *len;
    int iterations;
};

// ms per EM iteration of one option set, or a negative value when the
// options are rejected (e.g. a window too small for the model's layout).
// *shape: the sessions per item and lanes that were used.
struct Used {
    int64_t item_sessions, block;
};
mc_status measure(const Trial& tr, const int64_t* opt, double* ms_per_iter, Used* shape) {
    mc_model* m = nullptr;
    mc_status st = mc_model_create(tr.model_type, tr.device, &m);
    if (st != MC_OK) return st;
    for (int o = 0; o < kNumOptions && st == MC_OK; o++) st = mc_model_set_option(m, o, opt[o]);
    if (st == MC_OK) st = mc_init_parameters(m, tr.n, tr.query, tr.pidx, tr.clicks, tr.len, tr.n_qd);
    double ms = 0.0;
    if (st == MC_OK) st = mc_em_graph_timed(m, tr.iterations, &ms);
    *shape = Used{m->item_sessions, m->block};
    mc_model_destroy(m);
    if (st == MC_ERR_INVALID_ARG || st == MC_ERR_UNSUPPORTED) {
        *ms_per_iter = -1.0;
        return MC_OK;
    }
    if (st != MC_OK) return st;
    *ms_per_iter = ms / tr.iterations;
    return MC_OK;
}

}  // namespace
}  // namespace mc

using namespace mc;

extern "C" mc_status mc_autotune(int model_type, int device, int64_t n, const int32_t* query, const int32_t* pidx,
                                 const uint8_t* clicks, const uint8_t* len, int64_t n_qd, int iterations,
                                 int64_t* options, double* best_ms_per_iter, int* n_trials) {
    if (!query || !pidx || !clicks || !options || iterations < 1) {
        set_error("invalid argument");
        return MC_ERR_INVALID_ARG;
    }
    const Trial tr{model_type, device, n, n_qd, query, pidx, clicks, len, iterations};
    std::vector<int64_t> best(options, options + kNumOptions);
    double best_ms = 0.0;
    Used shape{0, 0};
    int trials = 0;
    mc_status st = measure(tr, best.data(), &best_ms, &shape);
    trials++;
    if (st != MC_OK) return st;
    if (best_ms < 0) {
        set_error("the starting options are not valid for this training set");
        return MC_ERR_INVALID_ARG;
    }
    // Tries a set of options; keeps it when faster.
    auto attempt_all = [&](const std::vector<int64_t>& cand) -> mc_status {
        double ms = 0.0;
        Used used{0, 0};
        mc_status s = measure(tr, cand.data(), &ms, &used);
        trials++;
        if (s != MC_OK) return s;
        if (ms >= 0 && ms < best_ms) {
            best = cand;
            best_ms = ms;
            shape = used;
        }
        return MC_OK;
    };
    // Tries `value` for option `o`.
    auto attempt = [&](int o, int64_t value) -> mc_status {
        const int64_t now = o == MC_OPT_ITEM_SESSIONS ? shape.item_sessions
                            : o == MC_OPT_BLOCK       ? shape.block
                                                      : best[(size_t)o];
        if (now == value) return MC_OK;
        std::vector<int64_t> cand = best;
        cand[(size_t)o] = value;
        return attempt_all(cand);
    };
    // The planner's own shape: the only one with windows for queries of more
    // entries than an item window (60,000 UBM sessions on queries of 2,400
    // documents: 15 us per iteration, 32 us the fastest of the others).
    std::vector<int64_t> planned = best;
    for (int o : {MC_OPT_ITEM_SESSIONS, MC_OPT_ITEM_WINDOW, MC_OPT_BLOCK}) planned[(size_t)o] = MC_AUTO;
    if (planned != best && (st = attempt_all(planned)) != MC_OK) return st;
    if ((st = attempt(MC_OPT_REDUCE_MODE, best[MC_OPT_REDUCE_MODE] == MC_REDUCE_SEGMENTED ? MC_REDUCE_ATOMIC
                                                                                            : MC_REDUCE_SEGMENTED)) != MC_OK)
        return st;
    for (int64_t s : {512, 1024, 2048, 4096, 8192, 16384})
        if ((st = attempt(MC_OPT_ITEM_SESSIONS, s)) != MC_OK) return st;
    if (best[MC_OPT_REDUCE_MODE] == MC_REDUCE_SEGMENTED) {
        for (int64_t w : {512, 1024, 1280, 1600, 2048})
            if ((st = attempt(MC_OPT_ITEM_WINDOW, w)) != MC_OK) return st;
        // Lanes per work item.
        for (int64_t b : {256, 512})
            if ((st = attempt(MC_OPT_BLOCK, b)) != MC_OK) return st;
        // Session format of the window items: packed records or rank-major.
        if ((st = attempt(MC_OPT_PACKED, best[MC_OPT_PACKED] ? 0 : 1)) != MC_OK) return st;
    } else {
        for (int64_t b : {256, 512})
            if ((st = attempt(MC_OPT_BLOCK, b)) != MC_OK) return st;
    }
    best[MC_OPT_ITEM_SESSIONS] = shape.item_sessions;
    best[MC_OPT_BLOCK] = shape.block;
    for (int o = 0; o < kNumOptions; o++) options[o] = best[(size_t)o];
    if (best_ms_per_iter) *best_ms_per_iter = best_ms;
    if (n_trials) *n_trials = trials;
    return MC_OK;
}
