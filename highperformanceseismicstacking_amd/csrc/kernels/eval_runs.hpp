// OCT evaluation over whole offset runs, for lanes that carry their own candidates
// (differential evolution, stretch-free search).
//
// In an OCT evaluation most traces fall outside the aperture |m - mh| <= apm around the
// candidate's displaced midpoint mh, and with one candidate per lane every lane has its own
// mh.  When a midpoint's list is grouped by half offset and each group ("run") is in
// midpoint order, the traces a lane keeps of a run are consecutive: m - mh rounds
// monotonically in m, so the two ends of the kept range come from two binary searches, and
// the lane walks lo .. hi - 1.  A wave makes as many steps per run as its busiest lane
// keeps.  (The walk over 64-trace chunks in eval_compact.hpp, the form for every other list,
// tests every trace and makes that many steps per chunk, and a run of ~134 traces spans
// three or four chunks: three times the steps.)
//
// The workgroup's waves share one midpoint, so its runs and its traces' midpoints sit in
// LDS once per workgroup (load_oct_runs).  A lane adds its kept traces in the same order and
// computes every value with the same operations as evaluate_n, so the results are the same
// bits (HSS_EXACT and HSS_FAST; HSS_KAHAN flushes its chunk sums at fixed trace blocks of
// the list and stays on evaluate_n).
#pragma once

#include "eval.hpp"

namespace hss {

// Traces of a midpoint that fit: 42 KB of LDS, three workgroups per CU with what differential
// evolution keeps there besides.
constexpr int kRunTraces = 3584;
constexpr int kRunsMax = 255;

struct OctRunTrace {
    float m;
    int ti;
};

struct OctRuns {
    OctRunTrace trace[kRunTraces];
    float scale[kRunTraces];  // 16-bit storage (1 on a line without scales)
    int start[kRunsMax + 1];  // [n] = the midpoint's trace count
    float h[kRunsMax + 1];
    int n;
};

// Whether a line's samples can be addressed from 24-bit trace numbers and row lengths and
// 32-bit byte offsets (evaluate_oct_runs does).
__device__ __forceinline__ bool oct_runs_addressable(const EvalCtx &e, int sample_bytes) {
    const uint64_t row = (uint64_t)e.ns * (uint64_t)sample_bytes;
    return e.ntr < (1 << 24) && row < (1u << 24) && (uint64_t)e.ntr * row <= 0xffffff00ull;
}

// Fills `r` with the midpoint's traces and runs; false (for the whole workgroup) when the
// list does not fit, is not in midpoint order inside a run, or its runs average fewer than
// four traces (lists in the reference's order).  Every thread of the workgroup calls it; it
// ends in a barrier.
__device__ __forceinline__ bool load_oct_runs(const EvalCtx &e, int sample_bytes, OctRuns &r) {
    const int tid = (int)threadIdx.x, nthreads = (int)blockDim.x;
    const int lane = tid & (kWave - 1);
    bool ok = e.cnt <= kRunTraces && oct_runs_addressable(e, sample_bytes);
    if (ok) {  // (uniform)
        bool sorted = true;
        for (int j = tid; j < e.cnt; j += nthreads) {
            const int ti = e.midx ? e.midx[e.beg + j] : e.beg + j;
            const float m = e.mid[ti];
            r.trace[j] = OctRunTrace{m, ti};
            if (sample_bytes == 2) r.scale[j] = e.scale ? e.scale[ti] : 1.0f;
            sorted = sorted && m == m;
            if (j > 0) {
                const int tp = e.midx ? e.midx[e.beg + j - 1] : e.beg + j - 1;
                const bool same = __float_as_uint(e.hoff[ti]) == __float_as_uint(e.hoff[tp]);
                sorted = sorted && (!same || m >= e.mid[tp]);
            }
        }
        ok = !__syncthreads_or(!sorted);
    }
    if (ok && tid < kWave) {
        // the first wave lists the runs (one offset bit pattern each)
        int n = 0;
        for (int j0 = 0; j0 < e.cnt; j0 += kWave) {
            const int j = j0 + lane;
            bool first = false;
            float h = 0.0f;
            if (j < e.cnt) {
                h = e.hoff[r.trace[j].ti];
                first = j == 0 || __float_as_uint(h) != __float_as_uint(e.hoff[r.trace[j - 1].ti]);
            }
            const unsigned long long mask = __builtin_amdgcn_ballot_w64(first);
            const int at = n + __builtin_popcountll(mask & ((1ull << lane) - 1));
            if (first && at < kRunsMax) {
                r.start[at] = j;
                r.h[at] = h;
            }
            n += __builtin_popcountll(mask);
        }
        if (lane == 0) {
            r.n = n <= kRunsMax && 4 * n <= e.cnt ? n : -1;
            if (n <= kRunsMax) r.start[n] = e.cnt;
        }
    }
    __syncthreads();
    return ok && r.n >= 0;
}

// The traces lo .. hi - 1 of a run beg .. end - 1 that a lane's aperture keeps.
struct OctKept {
    int lo, hi;
};

// Up to lo traces have m - mh < -apm, up to hi traces do not have m - mh > apm: the kept ones
// are those evaluate_n keeps, !(|m - mh| > apm) (a NaN mh fails both tests: every trace kept,
// as in the reference).  `on`: the lane has a candidate here.
__device__ __forceinline__ OctKept oct_kept_range(const OctRuns &r, int beg, int end,
                                                  const OctMid &om, float apm, bool on) {
    OctKept k{beg, beg};
    for (int bit = 1 << (31 - __builtin_clz(end - beg)); bit > 0; bit >>= 1) {
        const float dl = r.trace[min(k.lo + bit, end) - 1].m - om.mh;
        const float dh = r.trace[min(k.hi + bit, end) - 1].m - om.mh;
        k.lo += ((k.lo + bit <= end) & (dl < -apm)) ? bit : 0;
        k.hi += ((k.hi + bit <= end) & !(dh > apm)) ? bit : 0;
    }
    if (om.bad | !on) k.hi = k.lo;
    return k;
}

// The largest `count` (at most `most`) of the wave's lanes, by binary lifting on ballots, so
// that the walk is a counted, wave-uniform loop.
__device__ __forceinline__ int wave_max_steps(int count, int most) {
    int steps = 0;
    for (int bit = 1 << (31 - __builtin_clz(most)); bit > 0; bit >>= 1)
        if (__builtin_amdgcn_ballot_w64(count >= steps + bit) != 0) steps += bit;
    return steps;
}

template <int W, int VARIANT, int STORAGE, bool SHIFT, int CPL>
__device__ __forceinline__ void evaluate_oct_runs(const EvalCtx &e, const OctRuns &runs, float t0,
                                                  const Candidate (&k)[CPL], const bool (&on)[CPL],
                                                  float shift, bool active, float (&S)[CPL],
                                                  float (&stack)[CPL], unsigned *rejected) {
    static_assert(VARIANT != HSS_KAHAN, "the compensated variant uses evaluate_n");
    using Reader = SampleReader<STORAGE>;
    constexpr bool FASTIDX = W != 0;
    const bool scaled = (STORAGE != HSS_F32) && e.scale != nullptr;
    Window<W, VARIANT> acc[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[c].reset();
    unsigned rej = 0;  // the lane's own
    OctCand oc[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) oc[c] = oct_cand(t0, e.h0, k[c]);
    const unsigned row_bytes = (unsigned)e.ns * (STORAGE == HSS_F32 ? 4u : 2u);
    const int nruns = runs.n;
    for (int r = 0; r < nruns; ++r) {
        const int beg = __builtin_amdgcn_readfirstlane(runs.start[r]);
        const int end = __builtin_amdgcn_readfirstlane(runs.start[r + 1]);
        const OctTrace ot = oct_trace<FASTIDX>(uniform_f(runs.h[r]), 0.0f, e.h0);
        OctMid om[CPL];
        int lo[CPL], hi[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            om[c] = oct_mid<FASTIDX>(ot, oc[c], e.m0);
            const OctKept k = oct_kept_range(runs, beg, end, om[c], e.apm, on[c] & active);
            lo[c] = k.lo;
            hi[c] = k.hi;
        }
        OctTime otm[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (on[c] & active) rej += (unsigned)(end - beg - max(hi[c] - lo[c], 0));
            otm[c] = OctTime{0.0f, 0.0f, true};
            if (__builtin_amdgcn_ballot_w64(hi[c] > lo[c]) != 0)
                otm[c] = oct_time_terms<FASTIDX>(ot, oc[c], e.m0, om[c]);
            if (otm[c].bad) hi[c] = lo[c];
        }
        int most = 0;
#pragma unroll
        for (int c = 0; c < CPL; ++c) most = max(most, hi[c] - lo[c]);
        const int steps = wave_max_steps(most, end - beg);
        for (int step = 0; step < steps; ++step) {
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const bool has = lo[c] < hi[c];
                const int j = min(lo[c], end - 1);
                const OctRunTrace tr = runs.trace[j];
                lo[c] += 1;
                float tt = otm[c].th + otm[c].ah * (tr.m - om[c].mh);
                if constexpr (SHIFT) tt = tt + shift;
                int kk;
                float f;
                const bool in = window_k<FASTIDX>(tt, e.dt, e.inv_dt, e.ib, &kk, &f);
                if (has & in) {
                    // the window's first byte (24-bit product: see oct_runs_addressable)
                    const uint32_t row = __umul24((unsigned)tr.ti, row_bytes);
                    const uint32_t first = (uint32_t)(kk - e.tau);  // >= 0: the window is inside
                    if constexpr (STORAGE == HSS_F32) {
                        acc[c].add_row((const float *)at_bytes(e.samples, row + 4u * first), 0u, f,
                                       e.w, c);
                    } else {
                        const float sc = runs.scale[j];
                        const uint32_t at = (row >> 1) + first;
                        if constexpr (W > 0) {
                            acc[c].template add16<STORAGE>((const uint32_t *)e.samples, 0u, at, f,
                                                           sc, c);
                        } else {
                            const Reader rd{(decltype(Reader::p))e.samples};
                            acc[c].add(rd, (size_t)at, f, sc, scaled, e.w);
                        }
                    }
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[c].reduce(e.w, &S[c], &stack[c]);
    // the wave's count goes to its lowest active lane
    const unsigned total = wave_sum_u32(active ? rej : 0u);
    const unsigned long long act = __builtin_amdgcn_ballot_w64(active);
    const int lane = threadIdx.x & (kWave - 1);
    *rejected += (act != 0 && lane == __builtin_ctzll(act)) ? total : 0u;
}

}  // namespace hss
