// The launch-shape autotuner of the grid search's one-tile kernels (large CMP launches, the
// compensated variant, and windows without a compiled size; other launches take the spread
// kernel, whose shape follows from the launch's size: grid_spread.hpp).
//
// Three knobs (grid_impl.hpp, grid_staged.hpp), none of which changes a result bit:
//  * the parameter tile, candidates per lane (CPL = 1 or 2): two candidates share the
//    trace loop, the geometry broadcast and (16-bit storage) the LDS segment passes, at
//    the price of a second set of window registers;
//  * the t0 tile, 64-sample tiles per workgroup (TT = 1, 2 or 4): the workgroup's four
//    waves split into TT tiles x 4/TT candidate groups, trading the number of workgroups
//    per midpoint (and so how a midpoint's work spreads over the CUs of its XCD) against
//    the candidates each wave walks;
//  * staging (CMP, one t0 tile per workgroup): eight waves walk the traces together and
//    read their windows from the workgroup's LDS copy of each trace's span, instead of
//    each lane (FP32) or each wave (16-bit) reading its own.
// Which shape wins depends on the model, the window size, the storage and the variant.
// Which shape wins also depends on the number of candidates, which the waves take in rounds,
// and on the launch's size.  The first launch for a key (device, model, w, variant, storage,
// and up to 64, up to 128 or more candidates) that is large enough to time reliably runs every
// shape on a leading part of the caller's own batch (its first launch slots, about 8192
// workgroups), timed with HIP events on the caller's stream, and keeps the fastest (ties within
// 1% to the preferred shape); later launches that are large enough themselves reuse it, smaller
// ones take the untuned shape.  The kernels are pure functions
// of their inputs, so the timing runs write the same outputs (accumulating outputs are
// withheld from them by the caller).  No tuning under stream capture (the default shape
// is used), and HSS_AUTOTUNE=0 in the environment turns tuning off.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <tuple>
#include <utility>

#include "launch_util.hpp"

namespace hss {

namespace {
std::mutex tune_mu;
using TuneKey = std::tuple<int, int, int, int, int>;      // device, model, w, variant, storage
std::map<TuneKey, GridShape> pinned_shapes;               // by hss_grid_set_shape
std::map<std::pair<TuneKey, int>, GridShape> timed_shapes;  // by candidate_class() too

constexpr int kCandidateClasses = 3;
int candidate_class(int P) { return P <= 64 ? 0 : (P <= 128 ? 1 : 2); }

bool tuning_enabled() {
    const char *v = std::getenv("HSS_AUTOTUNE");
    return !(v && std::strcmp(v, "0") == 0);
}

// In order of preference: a later shape replaces the best so far only when it is faster by
// more than kTuneMargin, so near-ties (common: two candidates per lane often time within a
// fraction of a percent of one) resolve the same way on every run, to the shape listed
// first -- two candidates per lane first, whose four resident workgroups per CU keep a
// midpoint's traces in the XCD's L2 (one candidate per lane, at six, can fetch many times
// the line past it for the same time).
constexpr GridShape kShapes[] = {{2, 1, 0}, {1, 1, 0}, {2, 2, 0}, {1, 2, 0},
                                 {2, 4, 0}, {1, 4, 0}, {2, 1, 1}, {1, 1, 1}};
constexpr float kTuneMargin = 0.01f;
// workgroups a timing run covers (a leading part of the batch); the warm-up run before it
// (code load) covers a sixteenth of that
constexpr unsigned kTuneBlocks = 8192;
// workgroups of a launch that times reliably (several waves of them per CU)
constexpr unsigned kTuneLeast = 4096;

// The compensated variant's shape without timing.  CMP, up to 9 samples: the staged kernel with
// two candidates.  From 11 on its sums spill with two, or read the stage for few: staged with one
// at 11, and at 13 for few candidates; FP32 takes direct reads once the launch fills the chip.
// 640 samples, 60 traces, direct | staged with one | with two, in ms:
//   FP32, w = 11, 60 midpoints, 300 candidates 1.47 | 1.29 | 1.44, 250 midpoints, 90 candidates
//     1.27 | 1.36 | 1.63, 300 candidates 3.95 | 3.97 | 4.68
//   FP32, w = 13, 16 midpoints, 40 candidates 0.170 | 0.145 | 0.120, 60 midpoints, 90 candidates
//     0.537 | 0.533 | 0.568, 250 midpoints, 300 candidates 4.77 | 5.49 | 5.27
//   FP32, w = 15, 16 midpoints, 40 candidates 0.179 | 0.159 | 0.128, 60 midpoints, 300 candidates
//     1.75 | 1.91 | 1.78, 250 midpoints 5.07 | 7.06 | 5.76
//   FP16, w = 11, 250 midpoints, 300 candidates 5.87 | 4.07 | 4.67
//   FP16, w = 13, 16 midpoints, 40 candidates 0.317 | 0.152 | 0.140, 250 midpoints, 90 candidates
//     1.88 | 1.73 | 1.86, 300 candidates 6.33 | 5.51 | 5.27
//   FP16, w = 15, 16 midpoints, 40 candidates 0.327 | 0.169 | 0.153, 250 midpoints, 40 candidates
//     0.93 | 1.04 | 1.28, 90 candidates 2.03 | 2.24 | 2.06, 300 candidates 6.72 | 7.12 | 5.79
GridShape kahan_shape(int model, int w, int storage, long long tiles, int P) {
    constexpr GridShape direct{1, 1, 0}, staged_one{1, 1, 1}, staged_two{2, 1, 1};
    if (model != HSS_CMP || w < 5 || w > 15) return direct;
    if (w <= 9) return staged_two;
    if (storage == HSS_F32) {
        if (w == 11) return tiles > 768 ? direct : staged_one;
        return tiles > 480 ? direct : staged_two;
    }
    if (w == 11 || (w == 13 && P <= 128)) return staged_one;
    return w == 15 && P <= 64 && tiles > 768 ? direct : staged_two;
}
}  // namespace

int tuned_grid_shape(int model, int w, int variant, int storage, int n_slots, int ntiles, int P,
                     hipStream_t stream, const std::function<int(GridShape, int)> &launch,
                     GridShape *shape_out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = -1;
    const TuneKey key(dev, model, w, variant, storage);
    const auto timed_key = std::make_pair(key, candidate_class(P));
    const unsigned long long blocks = (unsigned long long)n_slots * (unsigned long long)ntiles;
    {
        std::lock_guard<std::mutex> lock(tune_mu);
        auto pin = pinned_shapes.find(key);
        if (pin != pinned_shapes.end()) {
            *shape_out = pin->second;
            return HSS_OK;
        }
        auto it = timed_shapes.find(timed_key);
        if (blocks >= kTuneLeast && it != timed_shapes.end()) {
            *shape_out = it->second;
            return HSS_OK;
        }
    }
    // untuned launches (small, under capture, tuning off): the choice of every tuned line
    // -- two candidates per lane, for CMP with the workgroup-staged traces -- but for the
    // compensated variant, and for up to 24 candidates of FP32 windows of 5 and 7 samples in
    // large launches, where a round or two of the staged kernel's eight waves do not pay for the
    // stage (400 midpoints of 640 samples, 24 candidates, staged | direct, w = 5 0.323 | 0.301,
    // w = 7 0.363 | 0.322 ms; 32 candidates, w = 5 0.382 | 0.397; 60 midpoints, EXACT, w = 5, 24
    // candidates 0.085 | 0.097)
    const bool few = model == HSS_CMP && storage == HSS_F32 && (w == 5 || w == 7) && P <= 24 &&
                     blocks > 1200;
    *shape_out = variant == HSS_KAHAN ? kahan_shape(model, w, storage, (long long)blocks, P)
                                      : GridShape{2, 1, model == HSS_CMP && !few ? 1 : 0};
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
        return HSS_OK;
    if (!tuning_enabled() || blocks < kTuneLeast) return HSS_OK;
    const int slots = (int)std::min<unsigned long long>(
        (unsigned long long)n_slots, (kTuneBlocks + ntiles - 1) / (unsigned)ntiles);
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return HSS_OK;
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return HSS_OK;
    }
    float best_ms = 0.0f;
    GridShape best = *shape_out;
    bool timed = false;
    int rc = HSS_OK;
    for (const GridShape &sh : kShapes) {
        if (sh.staged && model != HSS_CMP) continue;
        rc = launch(sh, std::max(1, slots / 16));  // warm-up (code load)
        if (rc != HSS_OK) break;
        if (hipEventRecord(e0, stream) != hipSuccess) break;
        rc = launch(sh, slots);
        if (rc != HSS_OK) break;
        if (hipEventRecord(e1, stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) break;
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, e0, e1) != hipSuccess) break;
        if (!timed || ms < best_ms * (1.0f - kTuneMargin)) {
            best_ms = ms;
            best = sh;
            timed = true;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != HSS_OK) return rc;
    if (!timed) return HSS_OK;  // a HIP call failed: keep the default, cache nothing
    std::lock_guard<std::mutex> lock(tune_mu);
    timed_shapes[timed_key] = best;
    *shape_out = best;
    return HSS_OK;
}

void tuned_grid_store(int dev, int model, int w, int variant, int storage, GridShape shape) {
    std::lock_guard<std::mutex> lock(tune_mu);
    const TuneKey key(dev, model, w, variant, storage);
    pinned_shapes.erase(key);
    for (int c = 0; c < kCandidateClasses; ++c) timed_shapes.erase({key, c});
    if (shape.cpl != 0) pinned_shapes[key] = shape;
}

// The pinned shape, else the one timed for the most candidates.
GridShape tuned_grid_lookup(int dev, int model, int w, int variant, int storage) {
    std::lock_guard<std::mutex> lock(tune_mu);
    const TuneKey key(dev, model, w, variant, storage);
    auto pin = pinned_shapes.find(key);
    if (pin != pinned_shapes.end()) return pin->second;
    for (int c = kCandidateClasses - 1; c >= 0; --c) {
        auto it = timed_shapes.find({key, c});
        if (it != timed_shapes.end()) return it->second;
    }
    return GridShape{0, 0, 0};
}

bool grid_shape_pinned(int model, int w, int variant, int storage) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lock(tune_mu);
    return pinned_shapes.count(TuneKey(dev, model, w, variant, storage)) != 0;
}

}  // namespace hss

// The launch shape the autotuner chose for a key on the current device (all 0: not yet).
extern "C" int hss_grid_tuned_shape(int model, int w, int variant, int storage, int32_t *cpl,
                                    int32_t *t0_tiles, int32_t *staged) {
    if (!cpl || !t0_tiles || !staged) return HSS_ERR_NULL_POINTER;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return HSS_ERR_NO_DEVICE;
    const hss::GridShape sh = hss::tuned_grid_lookup(dev, model, w, variant, storage);
    *cpl = sh.cpl;
    *t0_tiles = sh.tt;
    *staged = sh.staged;
    return HSS_OK;
}

extern "C" int hss_grid_tuned_config(int model, int w, int variant, int storage, int32_t *cpl) {
    int32_t tt = 0, staged = 0;
    return hss_grid_tuned_shape(model, w, variant, storage, cpl, &tt, &staged);
}

// Pins the launch shape for a key on the current device; cpl = 0 forgets the key (the
// next large launch tunes it again).
extern "C" int hss_grid_set_shape(int model, int w, int variant, int storage, int32_t cpl,
                                  int32_t t0_tiles, int32_t staged) {
    if (cpl < 0 || cpl > 2) return HSS_ERR_INVALID_SIZE;
    if (cpl > 0 && t0_tiles != 1 && t0_tiles != 2 && t0_tiles != 4) return HSS_ERR_INVALID_SIZE;
    if (staged != 0 && staged != 1) return HSS_ERR_INVALID_SIZE;
    if (cpl > 0 && staged && t0_tiles != 1) return HSS_ERR_INVALID_SIZE;
    if (cpl > 0 && staged && model != HSS_CMP) return HSS_ERR_INVALID_MODEL;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return HSS_ERR_NO_DEVICE;
    hss::tuned_grid_store(dev, model, w, variant, storage, hss::GridShape{cpl, t0_tiles, staged});
    return HSS_OK;
}

extern "C" int hss_grid_set_config(int model, int w, int variant, int storage, int32_t cpl) {
    return hss_grid_set_shape(model, w, variant, storage, cpl, 1, 0);
}
