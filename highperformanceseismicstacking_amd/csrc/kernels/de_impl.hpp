// Differential evolution over the traveltime parameters, one population per (midpoint, t0),
// every generation inside one launch.
//
// Reference behaviour (common/differential_evolution.cu:19-155 driven by
// DifferentialEvolutionAlgorithm.cpp:21-81): start x = lo + U*(hi-lo); evaluate; then
// for G-1 generations mutate per parameter from donors floor(U*(NP-1)) with F = 0.85 and
// clamp, cross over with CR = 0.5 and a forced index l = floor(U*(D-1)), evaluate the
// trials and keep a trial on strict '>' of its semblance; finally report the first best
// individual (cmp|zocrs|oct/differential_evolution.cu selectBestIndividuals*).  The
// reference draws from curand seeded with time(); here the uniforms come from
// Philox4x32-10 with counter {s, stream, individual, gen<<4 | block} and key = seed, the
// layout the CPU oracle uses, so runs are reproducible and checkable.
//
// MI355X mapping: one workgroup = (midpoint, 64 consecutive t0); lane l of every wave
// owns population s = tile*64 + l; wave v of V handles individuals v, v+V, ...  The
// populations live in a caller-provided workspace, double buffered (trials of generation
// g read generation g's individuals only), lane-fastest so every access is a 256-byte
// coalesced row; one workgroup barrier separates generations.
#pragma once

#include <cstddef>

#include "eval_compact.hpp"
#include "eval_runs.hpp"
#include "grid_impl.hpp"
#include "launch_util.hpp"

namespace hss {

// Launch shape of de_semblance_kernel, which runs large ZO-CRS launches and every model's
// compensated and non-compiled windows (de_spread_kernel below takes the rest), chosen by
// timing a ZO-CRS line (200 midpoints, ~930 traces each, NP 32, G 50, BF16).  ZO-CRS with a
// compiled window of up to 11 samples:
//  * de_cpl: two individuals per lane in one trace loop interleave two independent
//    traveltime/window chains, which hides their latency better than more resident waves
//    do (-6%; three were slower);
//  * de_min_occupancy: eight waves per SIMD, 64 VGPRs: the traveltime terms are kept across
//    a midpoint's traces, the trace loop is short and waits on memory, and more resident
//    waves pay for the spills of the per-generation code (6/7/8 waves 559/557/536 ms);
//  * de_waves: eight waves, so that four whole workgroups fill a CU's wave slots.
// The others keep one individual per lane and the compiler's own register budget.
template <int MODEL>
constexpr int de_waves() { return 8; }
template <int MODEL, int W, int VARIANT>
constexpr bool de_tuned() {
    return MODEL == HSS_ZOCRS && VARIANT != HSS_KAHAN && W != 0 && W <= 11;
}
template <int MODEL, int W, int VARIANT>
constexpr int de_cpl() { return de_tuned<MODEL, W, VARIANT>() ? 2 : 1; }
template <int MODEL, int W, int VARIANT>
constexpr int de_min_occupancy() { return de_tuned<MODEL, W, VARIANT>() ? 8 : 1; }
constexpr int kDeWavesMax = 8;
// Every lane carries its own individual, so a trace's windows spread over far more than
// one wave segment; DE reads 16-bit windows per lane (Window::add16) instead.
constexpr bool kDeSegments = false;
// OCT: DE keeps the offset-dependent half of the traveltime across consecutive traces
// with the same half offset (the host layer groups the lists of the non-exact variants by
// offset).  Any order gives the bits of computing every trace afresh; in the reference's
// (m, h) order nothing is shared.
constexpr bool kDeOctKeep = true;
// OCT: the aperture test of a run of traces first, then each lane's kept traces only
// (eval_compact.hpp); same bits as evaluate_n.  Not for HSS_KAHAN.
template <int MODEL, int VARIANT>
constexpr bool de_compact() { return MODEL == HSS_OCT && kDeOctKeep && VARIANT != HSS_KAHAN; }
constexpr float kDeF = 0.85f;   // F_FAC, common/include/gpu/interface.h:5
constexpr float kDeCR = 0.5f;   // CR, common/include/gpu/interface.h:6

struct DeArgs {
    EvalCtx e;
    const int *mbeg;
    const int *mcnt;
    const float *mm0;
    const int *morder;  // launch order (launch_midpoint) or NULL
    int nmid;
    int NP, G;
    int gen_begin, gen_end;  // generations run by this launch; the workspace carries the rest
    float lo[3], hi[3];
    uint32_t key0, key1, stream_base;
    int ntiles;
    int tl;           // de_spread_kernel: log2 of the t0 samples per workgroup
    float *ws;        // [n*ntiles][2][NP][D+2][64]
    float *result;    // [n][2+D][ns]
    float *pop_x;     // [n][ns][NP][D] or NULL
    float *pop_fx;    // [n][ns][NP][2] or NULL
    unsigned long long *not_used;  // [n] OCT rejections, accumulated, or NULL
};

// Philox4x32-10 (Salmon et al., SC'11).
__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                              uint32_t k0, uint32_t k1, uint32_t out[4]) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t lo0 = 0xD2511F53u * c0, hi0 = __umulhi(0xD2511F53u, c0);
        const uint32_t lo1 = 0xCD9E8D57u * c2, hi1 = __umulhi(0xCD9E8D57u, c2);
        c0 = hi1 ^ c1 ^ k0;
        c1 = lo1;
        c2 = hi0 ^ c3 ^ k1;
        c3 = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0;
    out[1] = c1;
    out[2] = c2;
    out[3] = c3;
}

// 24-bit uniform in (0, 1].
__device__ __forceinline__ float u01(uint32_t x) {
    return ((float)(x >> 8) + 1.0f) * 5.9604644775390625e-08f;
}

// The first nq uniforms of (s, stream, i, gen).
template <int NQ>
__device__ __forceinline__ void de_uniforms(const DeArgs &a, uint32_t s, uint32_t stream, int i,
                                            int gen, float *u) {
#pragma unroll
    for (int b = 0; b * 4 < NQ; ++b) {
        uint32_t r[4];
        philox4x32_10(s, stream, (uint32_t)i, ((uint32_t)gen << 4) | (uint32_t)b, a.key0, a.key1, r);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (b * 4 + q < NQ) u[b * 4 + q] = u01(r[q]);
    }
}

// Storage-form candidate of an individual in v space (cmp|zocrs|oct/differential_evolution.cu:
// c = 4/v^2, the other parameters as they are).
template <int MODEL>
__device__ __forceinline__ Candidate de_candidate(const float *x) {
    Candidate k{0.0f, 0.0f, 0.0f};
    const float v = x[0];
    k.c = 4.0f / (v * v);
    if constexpr (MODEL == HSS_ZOCRS) {
        k.p1 = x[1];
        k.p2 = x[2];
    } else if constexpr (MODEL == HSS_OCT) {
        k.p1 = x[1];
    }
    return k;
}

// The end of a run for sample s of midpoint g: the first best individual, and the population.
template <int D, class Rec>
__device__ __forceinline__ void de_report(const DeArgs &a, int g, int s, const Rec &rec) {
    const int ns = a.e.ns, NP = a.NP;
    const int cur = (a.G - 1) & 1;
    // selectBestIndividuals*: first strict maximum of S over the population
    float best = -1.0f, bstack = 0.0f;
    int bi = -1;
    for (int i = 0; i < NP; ++i) {
        const float S = *rec(cur, i, D);
        if (S > best) {
            best = S;
            bstack = *rec(cur, i, D + 1);
            bi = i;
        }
    }
    float *res = a.result + (size_t)g * (2 + D) * ns;
    res[s] = best;
    res[ns + s] = bi >= 0 ? bstack : 0.0f;
#pragma unroll
    for (int d = 0; d < D; ++d) res[(2 + d) * ns + s] = bi >= 0 ? *rec(cur, bi, d) : 0.0f;
    if (a.pop_x) {
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int d = 0; d < D; ++d)
                a.pop_x[(((size_t)g * ns + s) * NP + i) * D + d] = *rec(cur, i, d);
    }
    if (a.pop_fx) {
        for (int i = 0; i < NP; ++i) {
            a.pop_fx[(((size_t)g * ns + s) * NP + i) * 2] = *rec(cur, i, D);
            a.pop_fx[(((size_t)g * ns + s) * NP + i) * 2 + 1] = *rec(cur, i, D + 1);
        }
    }
}

template <int MODEL, int W, int VARIANT, int STORAGE>
__global__ __launch_bounds__(kDeWavesMax * kWave)
__attribute__((amdgpu_waves_per_eu(de_min_occupancy<MODEL, W, VARIANT>(), 8))) void de_semblance_kernel(DeArgs a) {
    constexpr int kDeWaves = de_waves<MODEL>();
    constexpr int D = MODEL == HSS_CMP ? 1 : (MODEL == HSS_ZOCRS ? 3 : 2);
    constexpr int REC = D + 2;  // D parameters, S, stack
    const int lane = threadIdx.x & (kWave - 1);
    // The wave index is uniform (readfirstlane), so the individual loops, their bounds and
    // the donors' rows are scalar work.  What outlives an evaluation -- the trials, the
    // lane's workspace column, its sample -- is kept in LDS or recomputed from the thread
    // index where it is used (thread_index_here), so that the registers of the budget go
    // to the trace walk and nothing is spilled: a spill slot is per-lane memory that takes
    // L2 from the traces (this kernel waits on its trace reads).
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int blk = logical_block(blockIdx.x, gridDim.x);
    const int slot = blk / a.ntiles;
    const int tile = blk - slot * a.ntiles;
    const int g = launch_midpoint(a.morder, a.nmid, slot);
    if (g < 0) return;
    const int s = tile * kWave + lane;
    const int ns = a.e.ns;
    const bool active = s < ns;
    const float t0 = (float)s * a.e.dt;
    const float t0sq = t0 * t0;
    const EvalCtx e = midpoint_ctx(a.e, a.mbeg, a.mcnt, a.mm0, g);
    const uint32_t stream = a.stream_base + (uint32_t)g;
    const int NP = a.NP;
    float *const base = a.ws + ((size_t)g * a.ntiles + tile) * 2 * NP * REC * kWave;
    auto rec = [&](int buf, int i, int f) -> float * {
        return base + ((size_t)(buf * NP + i) * REC + f) * kWave +
               (thread_index_here() & (kWave - 1));
    };
    // the lane's sample, as the counter of its random stream
    auto sample_here = [&]() {
        return (uint32_t)(tile * kWave + (thread_index_here() & (kWave - 1)));
    };

    __shared__ float seg_lds[kDeWaves][kSegFloats];
    // OCT: the midpoint's offset runs, or (lists without them) the waves' records of a chunk
    // of traces (uniform over the workgroup)
    union OctLists {
        OctRuns runs;
        OctTraceRec chunk[kDeWaves][kWave];
    };
    __shared__ std::conditional_t<de_compact<MODEL, VARIANT>(), OctLists, int> oct_lists;
    bool by_runs = false;
    if constexpr (de_compact<MODEL, VARIANT>())
        by_runs = load_oct_runs(e, STORAGE == HSS_F32 ? 4 : 2, oct_lists.runs);
    constexpr int CPL = de_cpl<MODEL, W, VARIANT>();
    // the individuals a lane evaluates together, from their drawing to their selection
    __shared__ float held[CPL * D][kDeWaves * kWave];
    uint64_t rejected = 0;  // the wave's rejections (uniform)
    auto eval = [&](const Candidate (&kc)[CPL], const bool (&on)[CPL], float (&S)[CPL],
                    float (&stk)[CPL]) {
        unsigned rej = 0;  // on the wave's lowest active lane
        if constexpr (de_compact<MODEL, VARIANT>()) {
            if (by_runs)
                evaluate_oct_runs<W, VARIANT, STORAGE, false, CPL>(e, oct_lists.runs, t0, kc, on,
                                                                   0.0f, active, S, stk, &rej);
            else
                evaluate_oct_compact<W, VARIANT, STORAGE, false, CPL>(
                    e, t0, kc, on, 0.0f, active, oct_lists.chunk[wave], S, stk, &rej);
        } else if (STORAGE == HSS_BF16 && e.scale == nullptr)
            // a BF16 line stored without scales: its windows summed as FP32 windows (one
            // form per code path, chosen outside the trace loop)
            evaluate_n<MODEL, W, VARIANT, STORAGE, false, CPL, kDeSegments, kDeOctKeep, false>(
                e, t0, t0sq, kc, on, 0.0f, active, seg_lds[wave], S, stk, &rej);
        else
            evaluate_n<MODEL, W, VARIANT, STORAGE, false, CPL, kDeSegments, kDeOctKeep>(
                e, t0, t0sq, kc, on, 0.0f, active, seg_lds[wave], S, stk, &rej);
        if constexpr (MODEL == HSS_OCT) {
            // the wave's total, summed over the lanes that hold a count (readlane: uniform)
            for (uint64_t m = __builtin_amdgcn_ballot_w64(rej != 0u); m; m &= m - 1)
                rejected += (uint32_t)__builtin_amdgcn_readlane((int)rej, __builtin_ctzll(m));
        }
    };
    // Generation g's population lives in buffer g & 1 of the workspace, so a run split
    // over several launches ([gen_begin, gen_end) each) gives the same result as one.
    // generation 0: the start population (startPopulations) and its fitness
    // A wave evaluates CPL individuals i0, i0+V, ... at a time (one trace loop for all);
    // a slot past NP is evaluated on individual i0's data and discarded.
    for (int i0 = wave; a.gen_begin == 0 && i0 < NP; i0 += kDeWaves * CPL) {
        Candidate kc[CPL];
        bool on[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int i = i0 + c * kDeWaves;
            on[c] = i < NP;
            float u[4];
            de_uniforms<D>(a, sample_here(), stream, on[c] ? i : i0, 0, u);
            float x[D];
            const int t = thread_index_here();
#pragma unroll
            for (int d = 0; d < D; ++d) {
                x[d] = a.lo[d] + u[d] * (a.hi[d] - a.lo[d]);
                held[c * D + d][t] = x[d];
            }
            kc[c] = de_candidate<MODEL>(x);
        }
        float S[CPL], stk[CPL];
        eval(kc, on, S, stk);
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (!on[c]) continue;
            const int i = i0 + c * kDeWaves;
            const int t = thread_index_here();
#pragma unroll
            for (int d = 0; d < D; ++d) *rec(0, i, d) = held[c * D + d][t];
            *rec(0, i, D) = S[c];
            *rec(0, i, D + 1) = stk[c];
        }
    }
    __syncthreads();

    for (int gen = a.gen_begin > 1 ? a.gen_begin : 1; gen < a.gen_end; ++gen) {
        const int cur = (gen - 1) & 1;
        for (int i0 = wave; i0 < NP; i0 += kDeWaves * CPL) {
            Candidate kc[CPL];
            bool on[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const int i1 = i0 + c * kDeWaves;
                on[c] = i1 < NP;
                const int i = on[c] ? i1 : i0;
                constexpr int NQ = 4 * D + 1;
                float u[NQ];
                de_uniforms<NQ>(a, sample_here(), stream, i, gen, u);
                int np1i = NP - 1;  // donors are drawn from NP - 1 (converted where used)
                __asm__ volatile("" : "+s"(np1i));
                const float np1 = (float)np1i;
                // mutatePopulations (common/differential_evolution.cu:43-89)
                float mutant[D];
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const unsigned r1 = (unsigned)(u[3 * d] * np1);
                    const unsigned r2 = (unsigned)(u[3 * d + 1] * np1);
                    const unsigned r3 = (unsigned)(u[3 * d + 2] * np1);
                    float nv = *rec(cur, r1, d) + kDeF * (*rec(cur, r2, d) - *rec(cur, r3, d));
                    // the bounds as opaque scalars: canonicalized at each use (one operation)
                    // rather than once into vector registers held through the evaluation
                    int hb = __builtin_amdgcn_readfirstlane(__float_as_int(a.hi[d]));
                    int lb = __builtin_amdgcn_readfirstlane(__float_as_int(a.lo[d]));
                    __asm__ volatile("" : "+s"(hb), "+s"(lb));
                    nv = fminf(nv, __int_as_float(hb));
                    nv = fmaxf(nv, __int_as_float(lb));
                    mutant[d] = nv;
                }
                // crossoverPopulations (common/differential_evolution.cu:91-122)
                const unsigned l = (unsigned)(u[3 * D] * (float)(D - 1));
                float trial[D];
                const int t = thread_index_here();
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const float r = u[3 * D + 1 + d];
                    trial[d] = (r > kDeCR && l != (unsigned)d) ? *rec(cur, i, d) : mutant[d];
                    held[c * D + d][t] = trial[d];
                }
                kc[c] = de_candidate<MODEL>(trial);
            }
            float S[CPL], stk[CPL];
            eval(kc, on, S, stk);
            // nextGeneration (common/differential_evolution.cu:124-155): strict '>'
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                if (!on[c]) continue;
                const int i = i0 + c * kDeWaves;
                const bool take = S[c] > *rec(cur, i, D);
                const int t = thread_index_here();
#pragma unroll
                for (int d = 0; d < D; ++d)
                    *rec(cur ^ 1, i, d) = take ? held[c * D + d][t] : *rec(cur, i, d);
                *rec(cur ^ 1, i, D) = take ? S[c] : *rec(cur, i, D);
                *rec(cur ^ 1, i, D + 1) = take ? stk[c] : *rec(cur, i, D + 1);
            }
        }
        __syncthreads();
    }

    if (MODEL == HSS_OCT && a.not_used) {
        if ((thread_index_here() & (kWave - 1)) == 0 && rejected)
            atomicAdd(a.not_used + g, (unsigned long long)rejected);
    }
    if (a.gen_end < a.G || wave != 0 || !active) return;
    de_report<D>(a, g, s, rec);
}

// The same run spread over more of the chip: a workgroup takes T = 16 consecutive t0 samples
// (de_spread_shape), and a wave's lanes split into four groups with an individual each, so that
// (with up to twelve waves) the whole population of a sample is evaluated at once, one
// individual per lane.  Workspace rows, random streams, donors and selections are those of
// de_semblance_kernel, so the results are the same bits, and a run may change kernels between
// generation ranges.
//
// One midpoint has ns/64 workgroups in de_semblance_kernel and each wave evaluates its
// individuals one pair after the other: 1001 samples, NP = 32, took 54.4 ms on 16 CUs
// (ZO-CRS, FP32, G = 50) where this kernel takes 15.1.  For CMP and OCT it is the faster one
// at every size (OCT, NP = 48, 24 midpoints 88.0 -> 68.4 ms, NP = 32, 128 midpoints 58.5 ->
// 44.6 ms; CMP, 60 midpoints 6.2 -> 5.1 ms): one candidate's registers and windows per lane,
// neighbouring lanes on neighbouring samples of one individual, short workgroups.  Two
// individuals per lane share ZO-CRS's long trace loop better once the chip is full (128
// midpoints: 62.3 against 67.5 ms here; 32 midpoints, 512 workgroups: 90.5 against 88.4), so
// it keeps de_semblance_kernel above 512 workgroups of it.  (OCT at T = 8/16/32: 77.8/68.4/
// 72.6 ms; at eight waves, two passes over 48 individuals, 84.7; at five waves per SIMD 88.8.)
constexpr int kDeSpreadWaves = 12;
template <int MODEL>
constexpr bool de_spread_always() { return MODEL != HSS_ZOCRS; }

template <int MODEL, int W, int VARIANT, int STORAGE>
__global__ __launch_bounds__(kDeSpreadWaves * kWave)
__attribute__((amdgpu_waves_per_eu(6, 8))) void de_spread_kernel(DeArgs a) {
    constexpr int D = MODEL == HSS_CMP ? 1 : (MODEL == HSS_ZOCRS ? 3 : 2);
    constexpr int REC = D + 2;  // D parameters, S, stack
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int T = 1 << a.tl;
    const int wg_per_mid = (a.e.ns + T - 1) / T;
    const int blk = logical_block(blockIdx.x, gridDim.x);
    const int slot = blk / wg_per_mid;
    const int g = launch_midpoint(a.morder, a.nmid, slot);
    if (g < 0) return;  // (the whole workgroup)
    const int s0 = (blk - slot * wg_per_mid) * T;
    const int s = s0 + (lane & (T - 1));
    const int ns = a.e.ns;
    const bool active = s < ns;
    const float t0 = (float)s * a.e.dt;
    const EvalCtx e = midpoint_ctx(a.e, a.mbeg, a.mcnt, a.mm0, g);
    const uint32_t stream = a.stream_base + (uint32_t)g;
    const int NP = a.NP;
    const int per_wave = kWave >> a.tl;
    const int per_pass = per_wave * ((int)blockDim.x / kWave);
    const int first = wave * per_wave + (lane >> a.tl);  // the lane's individual of a pass
    // the workspace column of sample s in de_semblance_kernel's 64-sample tiles
    float *const column = a.ws +
                          ((size_t)g * a.ntiles + s0 / kWave) * 2 * NP * REC * kWave + s % kWave;
    auto rec = [&](int buf, int i, int f) -> float * {
        return column + ((size_t)(buf * NP + i) * REC + f) * kWave;
    };
    // OCT: the midpoint's offset runs, or, for lists that do not fit them, the waves' records of
    // a chunk of traces for the compacted walk, where the list has runs at all (in the
    // reference's order its two passes find little to skip, and evaluate_n is faster).  150
    // midpoints, NP = 48, two generations, evaluate_n | compacted walk, in ms: grouped lists of
    // ~3700 traces, FP16 77.7 | 62.2, ~4600, FP16 96.9 | 75.4, FP32 78.0 | 64.0; ~2400 in the
    // reference's order, FP32 EXACT 115.8 | 124.1.
    union OctLists {
        OctRuns runs;
        OctTraceRec chunk[kDeSpreadWaves][kWave];
    };
    static_assert(sizeof(OctLists::chunk) <= offsetof(OctRuns, n),
                  "a wave may write its records while another still reads runs.n");
    __shared__ std::conditional_t<de_compact<MODEL, VARIANT>(), OctLists, int> oct_lists;
    bool by_runs = false;
    if constexpr (de_compact<MODEL, VARIANT>())
        by_runs = load_oct_runs(e, STORAGE == HSS_F32 ? 4 : 2, oct_lists.runs);
    bool compact = false;
    if constexpr (de_compact<MODEL, VARIANT>()) compact = !by_runs && oct_offset_runs_long(e);
    uint64_t rejected = 0;  // the wave's rejections (uniform)
    auto eval = [&](const Candidate &k, bool on, float *S, float *stk) {
        const Candidate kc[1] = {k};
        const bool on1[1] = {on};
        float S1[1], T1[1];
        unsigned rej = 0;  // on the wave's lowest active lane
        const bool live = active && on;
        if constexpr (de_compact<MODEL, VARIANT>()) {
            if (by_runs)
                evaluate_oct_runs<W, VARIANT, STORAGE, false, 1>(e, oct_lists.runs, t0, kc, on1,
                                                                 0.0f, live, S1, T1, &rej);
            else if (compact)
                evaluate_oct_compact<W, VARIANT, STORAGE, false, 1>(
                    e, t0, kc, on1, 0.0f, live, oct_lists.chunk[wave], S1, T1, &rej);
            else
                evaluate_n<MODEL, W, VARIANT, STORAGE, false, 1, kDeSegments, kDeOctKeep>(
                    e, t0, t0 * t0, kc, on1, 0.0f, live, nullptr, S1, T1, &rej);
        } else if (STORAGE == HSS_BF16 && e.scale == nullptr)
            evaluate_n<MODEL, W, VARIANT, STORAGE, false, 1, kDeSegments, kDeOctKeep, false>(
                e, t0, t0 * t0, kc, on1, 0.0f, live, nullptr, S1, T1, &rej);
        else
            evaluate_n<MODEL, W, VARIANT, STORAGE, false, 1, kDeSegments, kDeOctKeep>(
                e, t0, t0 * t0, kc, on1, 0.0f, live, nullptr, S1, T1, &rej);
        if constexpr (MODEL == HSS_OCT) {
            for (uint64_t m = __builtin_amdgcn_ballot_w64(rej != 0u); m; m &= m - 1)
                rejected += (uint32_t)__builtin_amdgcn_readlane((int)rej, __builtin_ctzll(m));
        }
        *S = S1[0];
        *stk = T1[0];
    };
    for (int gen = a.gen_begin; gen < a.gen_end; ++gen) {
        const int cur = (gen - 1) & 1, next = gen & 1;
        for (int p0 = 0; p0 < NP; p0 += per_pass) {
            if (p0 + wave * per_wave >= NP) continue;  // (the whole wave)
            // (a lane past the population works on the last individual and keeps nothing; so
            // does one past the trace, whose column lies in the last tile's padding)
            const bool on = p0 + first < NP;
            const int i = min(p0 + first, NP - 1);
            float x[D];
            if (gen == 0) {
                float u[4];
                de_uniforms<D>(a, (uint32_t)s, stream, i, 0, u);
#pragma unroll
                for (int d = 0; d < D; ++d) x[d] = a.lo[d] + u[d] * (a.hi[d] - a.lo[d]);
            } else {
                constexpr int NQ = 4 * D + 1;
                float u[NQ];
                de_uniforms<NQ>(a, (uint32_t)s, stream, i, gen, u);
                const float np1 = (float)(NP - 1);
                const unsigned l = (unsigned)(u[3 * D] * (float)(D - 1));
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const unsigned r1 = (unsigned)(u[3 * d] * np1);
                    const unsigned r2 = (unsigned)(u[3 * d + 1] * np1);
                    const unsigned r3 = (unsigned)(u[3 * d + 2] * np1);
                    float nv = *rec(cur, r1, d) + kDeF * (*rec(cur, r2, d) - *rec(cur, r3, d));
                    nv = fminf(nv, a.hi[d]);
                    nv = fmaxf(nv, a.lo[d]);
                    const float r = u[3 * D + 1 + d];
                    x[d] = (r > kDeCR && l != (unsigned)d) ? *rec(cur, i, d) : nv;
                }
            }
            float S, stk;
            eval(de_candidate<MODEL>(x), on, &S, &stk);
            if (!on || !active) continue;
            if (gen > 0 && !(S > *rec(cur, i, D))) {
#pragma unroll
                for (int f = 0; f < REC; ++f) *rec(next, i, f) = *rec(cur, i, f);
            } else {
#pragma unroll
                for (int d = 0; d < D; ++d) *rec(next, i, d) = x[d];
                *rec(next, i, D) = S;
                *rec(next, i, D + 1) = stk;
            }
        }
        __syncthreads();
    }
    if (MODEL == HSS_OCT && a.not_used) {
        if (lane == 0 && rejected) atomicAdd(a.not_used + g, (unsigned long long)rejected);
    }
    // the lanes of the first group report their samples
    if (a.gen_end < a.G || first != 0 || !active) return;
    de_report<D>(a, g, s, rec);
}

// The shape of a de_spread_kernel launch: T = 2^tl samples per workgroup, and its waves.  A CU's
// four SIMDs share them, so more than four are a multiple of four: as many as take the
// population in the fewest passes, the last ones idle.  (Five to seven or nine to eleven load the
// SIMDs unevenly: 100 midpoints, 8 generations, nine | twelve waves for a population of 36, CMP,
// FP32 3.65 | 3.39 ms; OCT, 30 midpoints, FP16, 4 generations 6.5 | 5.9; ZO-CRS, 20 midpoints,
// BF16, ten | twelve for 40 8.4 | 6.5.)  CMP launches that fill the chip take workgroups of four,
// which leave the SIMDs even whatever the population (300 midpoints, 6 generations, 36
// individuals, nine | twelve | four waves: FP16 10.6 | 9.5 | 7.7 ms, EXACT 16.7 | 14.9 | 12.1; 48
// individuals, twelve | four: FP16 10.3 | 9.6), FP32 ones once they are large (100 midpoints, 36
// individuals, twelve | four 3.39 | 3.56, 300 midpoints 7.70 | 7.40); 17 to 24 individuals of a
// 16-bit line then go eight at a time, not sixteen (FP16, w = 5, 120 midpoints, 20 individuals
// 2.51 | 2.22 ms).
struct DeSpreadShape {
    int tl, waves;
};
inline DeSpreadShape de_spread_shape(int model, int storage, int NP, long long n_mid, int ns) {
    constexpr int tl = 4, per_wave = kWave >> tl;
    const int need = (NP + per_wave - 1) / per_wave;
    if (need <= 4) return {tl, need};
    const long long workgroups = n_mid * ((ns + (1 << tl) - 1) >> tl);
    if (model == HSS_CMP && workgroups >= (storage == HSS_F32 || need % 4 == 0 ? 8192 : 1536))
        return {need <= 6 && storage != HSS_F32 ? tl + 1 : tl, 4};
    const int passes = (need + kDeSpreadWaves - 1) / kDeSpreadWaves;
    return {tl, ((need + passes - 1) / passes + 3) / 4 * 4};
}

// Whether ZO-CRS takes de_spread_kernel: up to 512 workgroups of de_semblance_kernel, 400 where
// some of its waves idle or, three of them, load the SIMDs unevenly (BF16, 36 individuals on nine
// of twelve waves, it | de_semblance_kernel: 30 midpoints, 480 workgroups 11.7 | 10.3 ms, 24 of
// them, FP32, 5.2 | 6.7).
constexpr long long kDeSpreadZocrsTiles = 512, kDeSpreadZocrsTilesIdle = 400;
inline bool de_spread_zocrs(long long tiles, int NP, DeSpreadShape shape) {
    const int need = (NP + (kWave >> shape.tl) - 1) / (kWave >> shape.tl);
    const bool even = need % shape.waves == 0 && shape.waves != 3;
    return tiles <= (even ? kDeSpreadZocrsTiles : kDeSpreadZocrsTilesIdle);
}

template <int MODEL>
int launch_de(const DeArgs &args, int n_mid, int variant, int storage, hipStream_t stream) {
    int st = HSS_OK;
    DeArgs a = args;
    const unsigned blocks = (unsigned)n_mid * (unsigned)a.ntiles;
    if (blocks == 0) return HSS_OK;
    const DeSpreadShape shape = de_spread_shape(MODEL, storage, a.NP, n_mid, a.e.ns);
    a.tl = shape.tl;
    const long long spread = (long long)n_mid * ((a.e.ns + (1 << a.tl) - 1) >> a.tl);
    const bool spread_it = (de_spread_always<MODEL>() || de_spread_zocrs(blocks, a.NP, shape)) &&
                           spread <= 0x7fffffffll;
    int st_launch = HSS_OK;
    int rc = dispatch_storage(storage, [&](auto S) {
        st = dispatch_variant(variant, [&](auto V) {
            dispatch_window(a.e.w, fast_index_verified(a.e.dt, a.e.tau, stream), [&](auto Wc) {
                constexpr int VV = decltype(V)::value, SS = decltype(S)::value,
                              WW = window_of<decltype(Wc)::value, VV, true>();
                if constexpr (WW > 0 && VV != HSS_KAHAN) {
                    if (spread_it) {
                        hipLaunchKernelGGL((de_spread_kernel<MODEL, WW, VV, SS>),
                                           dim3((unsigned)spread), dim3(shape.waves * kWave), 0, stream,
                                           a);
                        return;
                    }
                }
                // (CMP and OCT are spread: what is left is compensated or has no compiled
                // window)
                if constexpr (!(de_spread_always<MODEL>() && WW > 0 && VV != HSS_KAHAN))
                    hipLaunchKernelGGL((de_semblance_kernel<MODEL, WW, VV, SS>), dim3(blocks),
                                       dim3(de_waves<MODEL>() * kWave), 0, stream, a);
                else
                    st_launch = HSS_ERR_INVALID_SIZE;  // 2^31 workgroups: no workspace holds them
            });
        });
    });
    if (rc != HSS_OK) return rc;
    if (st != HSS_OK) return st;
    if (st_launch != HSS_OK) return st_launch;
    return hip_status(hipGetLastError());
}

int launch_de_cmp(const DeArgs &a, int n_mid, int variant, int storage, hipStream_t stream);
int launch_de_zocrs(const DeArgs &a, int n_mid, int variant, int storage, hipStream_t stream);
int launch_de_oct(const DeArgs &a, int n_mid, int variant, int storage, hipStream_t stream);

}  // namespace hss
