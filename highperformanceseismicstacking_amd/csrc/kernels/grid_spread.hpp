// Grid search spread over the chip: a workgroup takes T consecutive t0 samples (T a power of
// two up to 64), and its 512 lanes split into 512/T candidate groups of two candidates per
// lane and round.  Each lane keeps its running best; lanes that share a sample merge them as
// the other grid kernels do (the larger value, then the lower index), so the results are the
// same bits.
//
// The one-tile kernels give a midpoint of ns samples ns/64 workgroups, one 60-trace gather 16
// of them on 256 CUs, and a workgroup of a large launch runs long enough to leave a tail.
// With T down to 4 a gather fills the chip, and a line's launch ends evenly.  Candidates of
// one lane group are neighbours, so windows stay close together where T is small.  Measured
// (T in brackets; before -> here): one 60-trace gather of 640 samples, 300 candidates [4]
// 1.13 ms -> 69 us, 90 candidates [8] 370 -> 46 us; ZO-CRS, 24 midpoints, BF16 [16] 119 -> 39.9 ms, 200 midpoints 97 -> 82 ms;
// OCT, 30 midpoints, FP16 [4] 188 -> 48 ms (76 without the slopes' order below), 250 midpoints
// 204 -> 101 ms; OCT, 30 midpoints in the reference's order, EXACT 105 -> 60 ms.
// What bounds it then is VALU issue: the 16-bit lanes widen and scale every sample of their own windows, the price of not sharing
// LDS segments.
#pragma once

#include <algorithm>

#include "eval_lanes.hpp"
#include "grid_impl.hpp"

namespace hss {

constexpr int kSpreadWaves = 8;
constexpr int kSpreadThreads = kSpreadWaves * kWave;
// Candidates per lane.
constexpr int spread_cpl(int w) { return w > 15 ? 1 : 2; }
// Register budget, as waves per SIMD (a workgroup is two of them).  Windows of up to 11 samples
// of CMP and ZO-CRS fit six (39.9 against 42.8 ms at four, ZO-CRS, 24 midpoints); OCT, whose
// terms would spill, and wider windows take four (OCT 76 ms, 79 at six; w = 15: 43 against 59
// at two, which leaves one workgroup per CU).
template <int MODEL, int W>
constexpr int spread_min_waves() { return MODEL == HSS_OCT || W > 11 ? 4 : 6; }

// OCT candidates {c, slope}: the smallest d > 0, up to 256, whose slope is candidate 0's (its
// bit pattern), if it divides P; else 1.  Every lane of the wave calls it.
__device__ __forceinline__ int slope_period(const float *__restrict__ params, int P) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t first = __float_as_uint(params[1]);
    for (int d0 = 1; d0 < P && d0 <= 256; d0 += kWave) {
        const int d = d0 + lane;
        const unsigned long long same = __builtin_amdgcn_ballot_w64(
            d < P && __float_as_uint(params[2 * min(d, P - 1) + 1]) == first);
        if (same) {
            const int period = d0 + __builtin_ctzll(same);
            return P % period == 0 ? period : 1;
        }
    }
    return 1;
}

template <int MODEL, int W, int VARIANT, int STORAGE>
__global__ __launch_bounds__(kSpreadThreads)
__attribute__((amdgpu_waves_per_eu(spread_min_waves<MODEL, W>(), 8))) void grid_spread_kernel(GridArgs a) {
    constexpr int NP = MODEL == HSS_CMP ? 1 : (MODEL == HSS_ZOCRS ? 3 : 2);
    constexpr int CPL = spread_cpl(W);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int T = 1 << a.tl;  // t0 samples per workgroup
    const int blk = logical_block(blockIdx.x, gridDim.x);
    const int slot = blk / a.wg_per_mid;
    const int g = launch_midpoint(a.morder, a.nmid, slot);
    if (g < 0) return;  // (the whole workgroup)
    const int s0 = (blk - slot * a.wg_per_mid) * T;
    const int s = s0 + (lane & (T - 1));
    const int ns = a.e.ns;
    const bool active = s < ns;
    const float t0 = (float)s * a.e.dt;
    const EvalCtx e = midpoint_ctx(a.e, a.mbeg, a.mcnt, a.mm0, g);
    const int per_wave = kWave >> a.tl, groups = kSpreadWaves * per_wave;
    const int grp = wave * per_wave + (lane >> a.tl);

    float best = -1.0f, bstack = 0.0f;
    int bidx = -1;
    unsigned long long rejected = 0;
    bool by_runs = false;
    if constexpr (MODEL == HSS_OCT) by_runs = oct_offset_runs_long(e);
    // The candidates in the order the lanes take them: rank -> candidate, a permutation.
    // OCT: where the first slope comes again after `period` candidates (a grid, slope
    // fastest), all candidates of a slope one after the other, so that a wave's candidates
    // displace midpoints alike and its runs visit few traces.
    const int period = MODEL == HSS_OCT ? slope_period(a.params, a.P) : 1;
    const int per_slope = a.P / period;
    auto candidate_of = [&](int rank) {
        if constexpr (MODEL != HSS_OCT) return rank;
        const int sl = rank / per_slope;
        return (rank - sl * per_slope) * period + sl;
    };
    // (a wave whose lanes have no candidate left ends its rounds)
    for (int r0 = 0; r0 + wave * per_wave * CPL < a.P; r0 += groups * CPL) {
        const int q0 = r0 + grp * CPL;
        Candidate k[CPL];
        bool on[CPL];
        int cand[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            on[c] = q0 + c < a.P;
            cand[c] = candidate_of(min(q0 + c, a.P - 1));
            k[c] = load_candidate<MODEL>(a.params, cand[c]);
        }
        float S[CPL], stk[CPL];
        unsigned rej = 0;
        evaluate_lanes<MODEL, W, VARIANT, STORAGE, CPL>(e, t0, t0 * t0, k, on, active, by_runs, S,
                                                        stk, &rej);
        rejected += rej;
        if (!active) continue;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (!on[c]) continue;
            const int q = cand[c];
            if (a.sembl) a.sembl[((size_t)g * ns + s) * a.P + q] = S[c];
            if (a.stack) a.stack[((size_t)g * ns + s) * a.P + q] = stk[c];
            // the first strict maximum, in whatever order the candidates come
            if (S[c] > best || (MODEL == HSS_OCT && S[c] == best && q < bidx)) {
                best = S[c];
                bstack = stk[c];
                bidx = q;
            }
        }
    }
    if (MODEL == HSS_OCT && a.not_used) {
        const unsigned long long tot = wave_sum_u64(rejected);
        if (lane == 0 && tot) atomicAdd(a.not_used + g, tot);
    }

    // the best of the lanes that share a sample: the larger value, then the lower index
    // (as merge_bests), first inside the wave, then over the waves
    auto better = [&](float v, float st, int i) {
        if (i >= 0 && (v > best || (v == best && i < bidx) || bidx < 0)) {
            best = v;
            bstack = st;
            bidx = i;
        }
    };
    for (int off = T; off < kWave; off <<= 1) {
        const float v = __shfl_xor(best, off, kWave), st = __shfl_xor(bstack, off, kWave);
        const int i = __shfl_xor(bidx, off, kWave);
        better(v, st, i);
    }
    __shared__ float sh_best[kSpreadWaves][kWave], sh_stack[kSpreadWaves][kWave];
    __shared__ int sh_idx[kSpreadWaves][kWave];
    sh_best[wave][lane] = best;
    sh_stack[wave][lane] = bstack;
    sh_idx[wave][lane] = bidx;
    __syncthreads();
    if (wave != 0 || lane >= T || !active) return;
#pragma unroll
    for (int v = 1; v < kSpreadWaves; ++v) better(sh_best[v][lane], sh_stack[v][lane], sh_idx[v][lane]);
    float *res = a.result + (size_t)g * (2 + NP) * ns;
    res[s] = bidx >= 0 ? best : -1.0f;
    res[ns + s] = bidx >= 0 ? bstack : 0.0f;
    if (bidx >= 0) {
        const Candidate k = load_candidate<MODEL>(a.params, bidx);
        res[2 * ns + s] = 2 / sqrtf(k.c);
        if constexpr (NP >= 2) res[3 * ns + s] = k.p1;
        if constexpr (NP >= 3) res[4 * ns + s] = k.p2;
    } else {
#pragma unroll
        for (int d = 0; d < NP; ++d) res[(2 + d) * ns + s] = 0.0f;
    }
}

// log2 of T, 2 to 6: the one of least cost, counted in tenths of a wave's pass over a list
// (64 samples x candidates times CPL).
//  - Work: the passes of all waves.  A workgroup whose candidates fill few of its waves holds
//    its slot on a CU all the same, about 3.4 passes a round (CMP, 74 midpoints, 36 candidates:
//    0.750/0.413/0.266/0.244/0.265 ms for T = 4 to 64); an OCT workgroup spends 4.2 passes on
//    its run list.
//  - Passes of different T cost differently: for ZO-CRS 51/45/41.9/41.4 ms at 64/32/16/8 (100
//    midpoints), for OCT, where a wave of few samples and many candidates of one slope keeps
//    few traces of a run, 56/50.4/48.2 ms at 16/8/4 (30 midpoints, 1024 candidates).
//  - Latency: rounds follow each other, some 25 us each where the chip is idle, about what
//    1200 passes take when it is not (CMP, one midpoint, 300 candidates: 0.068/0.094/0.149/
//    0.251/0.487 ms for T = 4 to 64).
// Against T from the number of workgroups alone: CMP, one midpoint, 90 candidates 0.098 ->
// 0.046 ms, 8 midpoints, 40 candidates 0.094 -> 0.052; ZO-CRS, 4 midpoints, 36 candidates
// 1.13 -> 0.43; OCT, 16 midpoints, 32 candidates 1.51 -> 0.81; 144 candidates 3.13 -> 3.63.
inline int spread_tl(int model, int n_slots, int ns, int w, int P) {
    static constexpr int kPassCost[3][5] = {
        {108, 106, 104, 102, 100}, {105, 99, 100, 107, 122}, {100, 111, 127, 145, 170}};
    const int *cost = kPassCost[model == HSS_CMP ? 0 : (model == HSS_ZOCRS ? 1 : 2)];
    int tl = 2;
    double least = 0.0;
    for (int t = 2; t <= 6; ++t) {
        const int per_wave = (kWave >> t) * spread_cpl(w);
        const double waves = (double)((P - 1) / per_wave + 1);
        const double rounds = (double)((P - 1) / (per_wave * kSpreadWaves) + 1);
        const double wgs = (double)n_slots * (double)((ns + (1 << t) - 1) >> t);
        const double passes = model == HSS_OCT ? waves + 4.2 : std::max(waves, 3.4 * rounds);
        const double c = wgs * passes * cost[t - 2] + 120000.0 * rounds;
        if (t == 2 || c < least) {
            least = c;
            tl = t;
        }
    }
    return tl;
}

// Whether a launch takes this kernel when no shape is pinned for it: ZO-CRS and OCT always
// (measured faster at every size, above), CMP below the size where the staged kernel, which
// reads and widens a sample once for many windows, has enough workgroups (640 samples, staged
// | spread, in ms: FP32, 250 tiles, 11 samples P = 90 0.188 | 0.170, P = 300 0.512 | 0.453,
// 15 samples P = 300 0.590 | 0.588; 500 tiles, 11 samples P = 90 0.272 | 0.302, P = 300
// 0.800 | 0.833; FP16, 15 samples, 80 tiles P = 300 0.526 | 0.284, 250 tiles 0.581 | 0.727).
inline bool spread_wanted(int model, int storage, long long tiles) {
    if (model != HSS_CMP) return true;
    return tiles <= (storage == HSS_F32 ? 320 : 160);
}

// false: this window, variant or trace length has no such kernel.
template <int MODEL>
bool launch_grid_spread(const GridArgs &a, int n_slots, int variant, int storage, int tl,
                        hipStream_t stream, int *status) {
    if (variant == HSS_KAHAN || a.e.ns <= a.e.w ||
        !fast_index_verified(a.e.dt, a.e.tau, stream))
        return false;
    GridArgs la = a;
    la.tl = tl;
    la.wg_per_mid = (a.e.ns + (1 << tl) - 1) >> tl;
    const unsigned long long blocks = (unsigned long long)n_slots * la.wg_per_mid;
    if (blocks == 0 || blocks > 0x7fffffffull) return false;
    bool done = false;
    const int rc = dispatch_storage(storage, [&](auto S) {
        dispatch_variant(variant, [&](auto V) {
            dispatch_window(a.e.w, true, [&](auto Wc) {
                constexpr int WW = decltype(Wc)::value, VV = decltype(V)::value,
                              SS = decltype(S)::value;
                if constexpr (WW > 0 && VV != HSS_KAHAN) {
                    hipLaunchKernelGGL((grid_spread_kernel<MODEL, WW, VV, SS>),
                                       dim3((unsigned)blocks), dim3(kSpreadThreads), 0, stream, la);
                    done = true;
                }
            });
        });
    });
    *status = rc != HSS_OK ? rc : (done ? hip_status(hipGetLastError()) : HSS_OK);
    return done;
}

bool launch_spread_cmp(const GridArgs &a, int n_slots, int variant, int storage, int tl,
                       hipStream_t stream, int *status);
bool launch_spread_zocrs(const GridArgs &a, int n_slots, int variant, int storage, int tl,
                         hipStream_t stream, int *status);
bool launch_spread_oct(const GridArgs &a, int n_slots, int variant, int storage, int tl,
                       hipStream_t stream, int *status);

}  // namespace hss
