// CMP grid search with the traces staged in LDS for the whole workgroup.
//
// The grid kernel (grid_impl.hpp) lets every wave read its own windows: FP32 lanes with
// 16-byte loads (the texture-address unit is then the busiest unit after the VALU), 16-bit
// storage through a per-wave LDS segment that each wave loads and decodes for itself.
// Here the eight waves of a workgroup (one 64-sample t0 tile of a midpoint) take their
// candidates in rounds -- round r: wave v evaluates the CPL candidates starting at
// (8r + v)*CPL -- and walk the midpoint's traces together, a block at a time.  For each trace
// of a block the workgroup first loads, decodes and scales into LDS the samples that any
// window of the round can read, then every lane reads its windows from there.  (Blocks of
// 32 traces; HSS_KAHAN: 16.)  Eight waves rather than four halve the staging per candidate
// and the length of a workgroup, and with it the launch's tail: 10.2 -> 9.7 ms on a
// 150-midpoint line (w = 11, 512 candidates), 52.0 -> 50.9 ms on a 256-midpoint one (FP16,
// w = 15, 1024 candidates).
//
// The staged span of a trace follows from monotonicity (CMP: t = sqrt(t0^2 + c h^2) and
// every operation of the index chain are nondecreasing in t0 and in c): the smallest
// window start of the round is at the tile's first t0 and the round's smallest c, the
// largest at its last t0 and largest c.  When both corners' windows lie inside the trace,
// every lane's do, and the trace loop is straight-line code: no bounds tests, no lane masks,
// both candidates' index chains interleaved (lanes past the last sample repeat it).  Traces
// whose span crosses the trace's ends keep the tests; a trace whose span exceeds the stage
// is read directly.  Each lane adds its traces in the same order with the same operations
// on the same values as the grid kernel, so the results are the same bits (HSS_KAHAN's
// chunk boundaries are the same 16-trace blocks).
//
// What bounds it: VALU issue.  On the 256-midpoint line the straight-line loop is 147 VALU
// instructions per trace and two candidates (120 of them the windows), 322 issue cycles at
// the rates of window.hpp; the launch takes 395 cycles per trace and two candidates, with
// the VALU issuing 93% of the time.  Before (four waves, masked lanes, dword stage loads)
// 485 cycles; 61.0 -> 50.9 ms.
#pragma once

#include "grid_impl.hpp"

namespace hss {

// Samples staged per trace: 128, four per lane, two traces per wave and load.  The C5 line's spans (a 64-sample t0 tile plus the window and the moveout
// across the round's candidates) fit; a 256-sample stage was 4.7% slower (more LDS per
// workgroup, one workgroup fewer per CU).
constexpr int kStagedWaves = 8;
constexpr int kStagedThreads = kStagedWaves * kWave;
constexpr int kStageCap = 128;
constexpr int kStageLaneSamples = 4;
constexpr int kStageRowLanes = kStageCap / kStageLaneSamples;  // lanes that load one trace
constexpr int kStageRowsPerWave = kWave / kStageRowLanes;
// Traces per stage: 32 (16 KB of LDS; 48 was no faster, 16 was 3% slower on the C5 line),
// and for HSS_KAHAN its compensation chunk, since its sums are flushed at those fixed
// trace blocks.
template <int VARIANT>
constexpr int stage_traces() { return VARIANT == HSS_KAHAN ? kKahanChunk : 32; }

// Register budget, as waves per SIMD.  A workgroup is two waves per SIMD, so budgets between
// four and six waves buy nothing.  Windows of up to 11 samples fit six (11 samples spill 28
// bytes outside the trace loop; 9.57 ms at six against 9.73 at four on a 150-midpoint line),
// wider ones take four without spills (50.9 against 52.4 ms at six on a 256-midpoint line).
// Inside the trace loop nothing may be spilled: a spill slot is per-lane memory that stays
// in L2 beside the traces.  Hence the running best in LDS, the uniform values in scalar
// registers and thread_index_here().  HSS_KAHAN keeps the grid kernel's budget.
template <int W, int VARIANT, int CPL>
constexpr int staged_min_waves() {
    if (VARIANT == HSS_KAHAN) return grid_min_waves<VARIANT, CPL>();
    return W == 0 ? 2 : (W <= 11 ? 6 : 4);
}

// The running best of each thread, in LDS.
struct RunBest {
    float best[kStagedThreads];
    float stack[kStagedThreads];
    int idx[kStagedThreads];
};

// What the trace loop needs of one staged trace: h^2 and the LDS address at which sample
// index k's window starts, minus 8*k.
struct StagedTrace {
    float h2;
    uint32_t row;
};

template <int W, int VARIANT, int STORAGE, int CPL>
__global__ __launch_bounds__(kStagedThreads)
__attribute__((amdgpu_waves_per_eu(staged_min_waves<W, VARIANT, CPL>(), 8))) void grid_staged_kernel(
    GridArgs a) {
    using Reader = SampleReader<STORAGE>;
    constexpr bool FASTIDX = W != 0;
    const int lane = threadIdx.x & (kWave - 1);
    // wave-uniform values go through readfirstlane so that they live in scalar registers
    // (the round's candidates are then scalar loads; gfx950 has no scalar float ALU, so a
    // uniform float otherwise takes a vector register for the whole kernel)
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int blk = logical_block(blockIdx.x, gridDim.x);
    const int slot = blk / a.ntiles;
    const int tile = blk - slot * a.ntiles;
    const int g = launch_midpoint(a.morder, a.nmid, slot);
    if (g < 0) return;  // (the whole workgroup)
    const int s = tile * kWave + lane;
    const int ns = a.e.ns;
    const bool active = s < ns;
    // lanes past the last sample follow it: they read what it reads and write nothing
    const float t0 = (float)min(s, ns - 1) * a.e.dt;
    const float t0sq = t0 * t0;
    const EvalCtx e = midpoint_ctx(a.e, a.mbeg, a.mcnt, a.mm0, g);
    const bool scaled = (STORAGE != HSS_F32) && e.scale != nullptr;
    Reader rd{(decltype(Reader::p))e.samples};
    // the tile's first and last t0 (the span's corners)
    const float t0a = (float)(tile * kWave) * e.dt;
    const float t0b = (float)min(tile * kWave + kWave - 1, ns - 1) * e.dt;
    const float t0a_sq = uniform_f(t0a * t0a), t0b_sq = uniform_f(t0b * t0b);
    // the midpoint's [ns][P] slabs of the optional cubes (the host keeps ns * P below 2^32)
    float *const sembl_g = a.sembl ? a.sembl + (size_t)g * ns * a.P : nullptr;
    float *const stack_g = a.stack ? a.stack + (size_t)g * ns * a.P : nullptr;

    constexpr int ST = stage_traces<VARIANT>();
    static_assert(2 * ST <= kWave, "a block's span corners are one wave's lanes");
    static_assert(ST % (kStagedWaves * kStageRowsPerWave) == 0, "whole loads");
    // stage[jj][i] = samples i and i + 1 of trace jj's span: a window that starts at any i is
    // (W + 1)/2 aligned 8-byte reads, 16 bytes apart
    __shared__ alignas(16) float2 stage[ST][kStageCap];
    __shared__ StagedTrace meta[ST + 1];
    // the lane's running best (first strict maximum over its candidates in order), kept in
    // LDS rather than in registers, which the window sums of two candidates use up; each
    // thread reads and writes only its own slots
    __shared__ RunBest run;
    run.best[threadIdx.x] = -1.0f;
    run.stack[threadIdx.x] = 0.0f;
    run.idx[threadIdx.x] = -1;
    if (threadIdx.x == 0) meta[ST] = StagedTrace{0.0f, 0u};
    const float dt_v = vector_f(e.dt), inv_v = vector_f(e.inv_dt);

    const int per_round = kStagedWaves * CPL;
    const int rounds = (a.P + per_round - 1) / per_round;
    for (int r = 0; r < rounds; ++r) {
        const int q0 = (r * kStagedWaves + wave) * CPL;
        float kc[CPL];
        bool on[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            on[c] = q0 + c < a.P;
            kc[c] = vector_f(a.params[on[c] ? q0 + c : min(q0, a.P - 1)]);
        }
        // the round's range of c (all waves: the same candidates, the same values)
        float cmin = INFINITY, cmax = -INFINITY;
        bool c_ok = true;  // no NaN among them
        const int qa = r * per_round, qb = min(a.P, qa + per_round);
        for (int q = qa; q < qb; ++q) {
            const float c = a.params[q];
            cmin = fminf(cmin, c);
            cmax = fmaxf(cmax, c);
            c_ok = c_ok && c == c;
        }
        Window<W, VARIANT> acc[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[c].reset();

        for (int j0 = 0; j0 < e.cnt; j0 += ST) {
            const int nj = min(ST, e.cnt - j0);
            // lanes jj and ST + jj < 2*ST: trace j0 + jj's geometry, scale and staged span;
            // the first of the two works out the span's lower corner, the second its upper
            const int ln = thread_index_here() & (kWave - 1);
            const int tr = ln & (ST - 1);
            const bool upper = (ln & ST) != 0;
            const bool have = tr < nj;
            const int ti_l = have ? (e.midx ? e.midx[e.beg + j0 + tr] : e.beg + j0 + tr) : 0;
            const float h2_l = have ? e.hoff2[ti_l] : 0.0f;
            const float sc_l = (scaled && have) ? e.scale[ti_l] : 1.0f;
            int base_l;
            unsigned long long fit, clean;  // bit jj: trace j0 + jj
            {
                const float x = (upper ? t0b_sq : t0a_sq) + (upper ? cmax : cmin) * h2_l;
                const float t = sqrt_time<FASTIDX, false>(x);
                float ti;
                if constexpr (FASTIDX) ti = div_rn(t, e.dt, e.inv_dt);
                else ti = t / e.dt;
                // the corner's sample index (the span needs the order only: lanes use
                // indices inside (lo, hi) of index_bounds()); a corner that has none, or
                // whose root sqrt_rn_big does not give, stands for the whole trace
                const bool usable = x >= 0x1.0p-96f && x < INFINITY;
                const int none = upper ? 1 << 24 : -1;
                const int k = usable ? (int)fminf(fmaxf(ti, -1.0f), 16777216.0f) : none;
                const bool in = usable && ti > e.ib.lo && ti < e.ib.hi;
                const int kx = __shfl_xor(2 * k + (in ? 1 : 0), ST, kWave);
                const int ka = upper ? (kx >> 1) : k, kb = upper ? k : (kx >> 1);
                // windows run from k - tau to k + tau + 1, inside the trace
                const int first = max(ka - e.tau, 0), end = min(kb + e.tau + 2, ns);
                base_l = min(first, ns - kStageCap);
                if (STORAGE != HSS_F32 && ((((ti_l & ns) ^ base_l) & 1) != 0))
                    // 16-bit samples are loaded in aligned words: an even flat index
                    base_l += base_l < first ? 1 : -1;
                // (monotone in c only for h^2 >= 0)
                const bool ok = have && ns >= kStageCap && h2_l >= 0.0f && end - base_l <= kStageCap;
                fit = __builtin_amdgcn_ballot_w64(ok) & ((1ull << ST) - 1);
                // every window of the trace lies inside it: no bounds tests
                clean = W == 0 || !c_ok ? 0
                                        : __builtin_amdgcn_ballot_w64(in && (kx & 1)) & fit;
            }
            if constexpr (VARIANT == HSS_KAHAN) {
                if (j0 > 0) {
#pragma unroll
                    for (int c = 0; c < CPL; ++c) acc[c].flush(e.w);
                }
            }
            if (fit != 0) {
                constexpr int LOADS = ST / (kStagedWaves * kStageRowsPerWave);
                const size_t off_l = (size_t)ti_l * (size_t)ns + (size_t)(ptrdiff_t)base_l;
                const int col = (ln & (kStageRowLanes - 1)) * kStageLaneSamples;
                // The sample after the lane's own four (the last lane's would lie past the
                // stage, where no window reads)
                const int after = min(col + kStageLaneSamples, kStageCap - 1);
                auto row_of = [&](int i) {  // the trace this lane helps load in load i
                    return (i * kStagedWaves + wave) * kStageRowsPerWave + ln / kStageRowLanes;
                };
                auto offset_of = [&](int row) {
                    return (size_t)(uint32_t)__shfl((int)(off_l >> 32), row, kWave) << 32 |
                           (uint32_t)__shfl((int)off_l, row, kWave);
                };
                // all of the block's loads first, then the (decoded and scaled) samples into
                // LDS: one wait, not one per trace
                constexpr bool F32S = STORAGE == HSS_F32;
                constexpr int RAW = F32S ? kStageLaneSamples + 1 : kStageLaneSamples / 2 + 1;
                uint32_t raw[LOADS][RAW];
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    const int row = row_of(i);
                    const size_t off = offset_of(row);
#pragma unroll
                    for (int q = 0; q < RAW; ++q) raw[i][q] = 0;
                    if ((fit >> row) & 1) {
                        if constexpr (F32S) {
                            const uint32_t *src = (const uint32_t *)e.samples + off;
#pragma unroll
                            for (int q = 0; q < RAW - 1; ++q) raw[i][q] = src[col + q];
                            raw[i][RAW - 1] = src[after];
                        } else {
                            const uint32_t *src =
                                (const uint32_t *)((const uint16_t *)e.samples + off);
#pragma unroll
                            for (int q = 0; q < RAW - 1; ++q) raw[i][q] = src[col / 2 + q];
                            raw[i][RAW - 1] = src[after / 2];
                        }
                    }
                }
                __syncthreads();  // every wave has read the previous staged block
                if (wave == 0 && ln < nj)
                    meta[ln] = StagedTrace{
                        h2_l, (uint32_t)(size_t)((const LdsFloat *)&stage[0][0]) +
                                  8u * (uint32_t)(kStageCap * ln - base_l - e.tau)};
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    const int row = row_of(i);
                    float v[kStageLaneSamples + 1];
                    if constexpr (F32S) {
#pragma unroll
                        for (int q = 0; q < RAW; ++q) v[q] = __uint_as_float(raw[i][q]);
                    } else {
                        // as the wave segments decode and scale
                        const float sc = __shfl(sc_l, row, kWave);
#pragma unroll
                        for (int q = 0; q <= kStageLaneSamples; ++q) {
                            const uint32_t d = raw[i][q / 2];
                            if constexpr (STORAGE == HSS_F16)
                                v[q] = (float)__builtin_bit_cast(
                                           _Float16, (uint16_t)((q & 1) ? d >> 16 : d & 0xffffu)) * sc;
                            else
                                v[q] = __uint_as_float((q & 1) ? d & 0xffff0000u : d << 16) * sc;
                        }
                    }
                    float4 *dst = (float4 *)&stage[row][col];
                    dst[0] = float4{v[0], v[1], v[1], v[2]};
                    dst[1] = float4{v[2], v[3], v[3], v[4]};
                }
                __syncthreads();
            }
            // One read path per loop, chosen for the whole workgroup (every wave computes the
            // same spans): runs of consecutive traces that are staged with all their windows
            // inside the trace, staged, or read directly.
            for (int jj = 0; jj < nj;) {
                const bool cl = (clean >> jj) & 1, ft = (fit >> jj) & 1;
                const unsigned long long same = cl ? clean : (ft ? fit & ~clean : ~fit);
                const int je = min(nj, jj + (int)__builtin_ctzll(~(same >> jj) | (1ull << ST)));
                if (W > 0 && cl) {
                    // every lane's windows of both candidates, no masks: index, read, sum
#pragma unroll
                    for (int c = 0; c < CPL; ++c) acc[c].used += (unsigned)(je - jj);
                    for (; jj < je; ++jj) {
                        const StagedTrace m = meta[jj];
                        LdsPair *at[CPL];
                        float f[CPL];
#pragma unroll
                        for (int c = 0; c < CPL; ++c) {
                            const float t = sqrt_rn_big(t0sq + kc[c] * m.h2);
                            const float ti = div_rn(t, dt_v, inv_v);
                            f[c] = __builtin_amdgcn_fractf(ti);
                            at[c] = (LdsPair *)(size_t)(m.row + 8u * (uint32_t)(int)ti);
                        }
#pragma unroll
                        for (int c = 0; c < CPL; ++c) {
                            acc[c].sum_pairs(at[c], f[c], e.w, c);
                        }
                    }
                    continue;
                }
                // the lane's sample index, weight and inclusion
                auto index = [&](float h2, int (&kk)[CPL], float (&f)[CPL], bool (&use)[CPL]) {
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        const float t = sqrt_time<FASTIDX, false>(t0sq + kc[c] * h2);
                        const bool in =
                            window_k<FASTIDX>(t, e.dt, e.inv_dt, e.ib, &kk[c], &f[c]);
                        use[c] = in & active & on[c];
                    }
                };
                int kk[CPL];
                float f[CPL];
                bool use[CPL];
                if (ft) {
                    for (; jj < je; ++jj) {
                        const StagedTrace m = meta[jj];
                        index(m.h2, kk, f, use);
#pragma unroll
                        for (int c = 0; c < CPL; ++c) {
                            if (!use[c]) continue;
                            acc[c].sum_pairs((LdsPair *)(size_t)(m.row + 8u * (uint32_t)kk[c]),
                                             f[c], e.w, c);
                            acc[c].used++;
                        }
                    }
                } else {
                    for (; jj < je; ++jj) {
                        const size_t trace0 =
                            (size_t)__builtin_amdgcn_readlane(ti_l, jj) * (size_t)ns;
                        const float sc = bcast(sc_l, jj);
                        index(bcast(h2_l, jj), kk, f, use);
#pragma unroll
                        for (int c = 0; c < CPL; ++c) {
                            if (!use[c]) continue;
                            if constexpr (STORAGE == HSS_F32)
                                acc[c].add_row((const float *)e.samples + trace0 - (size_t)e.tau,
                                               (unsigned)kk[c], f[c], e.w, c);
                            else
                                acc[c].add(rd, trace0 + (size_t)(kk[c] - e.tau), f[c], sc, true,
                                           e.w);
                        }
                    }
                }
            }
        }
        float S[CPL], stk[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[c].reduce(e.w, &S[c], &stk[c]);
        if (active) {
            const int t = thread_index_here();
            const uint32_t cube_row = (uint32_t)(tile * kWave + (t & (kWave - 1))) * (uint32_t)a.P;
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                if (!on[c]) continue;
                const int q = q0 + c;
                if (sembl_g) sembl_g[cube_row + (uint32_t)q] = S[c];
                if (stack_g) stack_g[cube_row + (uint32_t)q] = stk[c];
                if (S[c] > run.best[t]) {
                    run.best[t] = S[c];
                    run.stack[t] = stk[c];
                    run.idx[t] = q;
                }
            }
        }
    }

    // the waves' bests of each t0, as merge_bests merges them (the largest value, the
    // smallest candidate index among equal values)
    __syncthreads();
    if (wave != 0 || !active) return;
    const int ln = thread_index_here() & (kWave - 1);
    float B = -1.0f, BS = 0.0f;
    int BI = -1;
#pragma unroll
    for (int v = 0; v < kStagedWaves; ++v) {
        const int iv = run.idx[v * kWave + ln];
        const float sv = run.best[v * kWave + ln];
        if (iv >= 0 && (sv > B || (sv == B && iv < BI))) {
            B = sv;
            BS = run.stack[v * kWave + ln];
            BI = iv;
        }
    }
    const int so = tile * kWave + ln;  // the lane's sample
    float *res = a.result + (size_t)g * 3 * ns;
    res[so] = B;
    res[ns + so] = BI >= 0 ? BS : 0.0f;
    res[2 * ns + so] = BI >= 0 ? 2 / sqrtf(load_candidate<HSS_CMP>(a.params, BI).c) : 0.0f;
}

// Whether few candidates go one to a lane.  A round of the eight waves is eight candidates
// then and sixteen with two, so with two P = 24 costs what 32 does.  Two are up to 12% cheaper
// per candidate of a full round, except in 16 bits or from 13 samples on with few rounds
// (640 samples, 60 traces, two | one, in ms: 250 midpoints, FP32, 11 samples P = 24 0.421 |
// 0.339, 52 0.816 | 0.716, 64 0.816 | 0.815, 72 0.980 | 0.899, 128 1.454 | 1.532, 512 5.20 |
// 5.52; FP32, 5 samples P = 64 0.543 | 0.570; FP16, 15 samples P = 28 0.683 | 0.578, 64
// 1.098 | 0.970, 128 1.816 | 1.800, 512 6.23 | 6.42).
inline bool staged_one_candidate(int w, int storage, int P) {
    const int one = (P + kStagedWaves - 1) / kStagedWaves;
    const int two = 2 * ((P + 2 * kStagedWaves - 1) / (2 * kStagedWaves));
    return 11 * one < 10 * two || (P <= 64 && (storage != HSS_F32 || w >= 13));
}

// Host launcher: one workgroup per (launch slot, t0 tile) (a.tt must be 1).
int launch_grid_cmp_staged(const GridArgs &a, int n_slots, int variant, int storage, int cpl,
                           hipStream_t stream);

}  // namespace hss
