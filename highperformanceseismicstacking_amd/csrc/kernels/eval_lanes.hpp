// A grid evaluation in which every lane carries its own candidates (grid_spread.hpp).
//
// evaluate_n with per-lane candidates, window reads by every lane for itself and three
// differences, none of which changes a bit of a result:
//  * both candidates' windows are requested before the first is summed (a lane without a
//    window reads the trace's first one), in straight-line code;
//  * uniform values of the index chain sit in vector registers (window.hpp);
//  * OCT, lists in offset runs: a run only visits the traces that some lane's aperture keeps.
//    With the smallest and largest displaced midpoint of the wave's lanes, m - mh < -apm for
//    the smallest or m - mh > apm for the largest rejects a trace for every lane (the
//    difference rounds monotonically in mh); about three traces in four drop out this way.
#pragma once

#include "eval.hpp"

namespace hss {

// The smallest (largest) value over the wave's lanes.
__device__ __forceinline__ float wave_min_f(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fminf(x, __shfl_xor(x, off, kWave));
    return x;
}
__device__ __forceinline__ float wave_max_f(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, kWave));
    return x;
}

// by_runs (OCT, uniform): the list comes in offset runs (oct_offset_runs_long).  *rejected
// gets the lane's own number of OCT rejections.  Traces must be longer than the window.
template <int MODEL, int W, int VARIANT, int STORAGE, int CPL>
__device__ __forceinline__ void evaluate_lanes(const EvalCtx &e, float t0, float t0sq,
                                               const Candidate (&k)[CPL], const bool (&on)[CPL],
                                               bool active, bool by_runs, float (&S)[CPL],
                                               float (&stack)[CPL], unsigned *rejected) {
    static_assert(W > 0 && VARIANT != HSS_KAHAN, "compiled windows, plain sums");
    const bool scaled = (STORAGE != HSS_F32) && e.scale != nullptr;
    Window<W, VARIANT> acc[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[c].reset();
    unsigned rej = 0;
    const int lane = threadIdx.x & (kWave - 1);
    const float dt_v = vector_f(e.dt), inv_v = vector_f(e.inv_dt);
    OctCand oc[CPL];
    if constexpr (MODEL == HSS_OCT) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) oc[c] = oct_cand(t0, e.h0, k[c]);
    }
    float zmid[CPL];  // ZO-CRS: the midpoint part, kept across a midpoint's traces
    uint32_t zkey = 0;
    bool zvalid = false;
    for (int j0 = 0; j0 < e.cnt; j0 += kWave) {
        const int mine = j0 + lane;
        const bool have = mine < e.cnt;
        const int ti_l = have ? (e.midx ? e.midx[e.beg + mine] : e.beg + mine) : 0;
        const TraceGeom g_l = have ? load_geom<MODEL>(e.mid, e.hoff, e.hoff2, ti_l)
                                   : TraceGeom{0.0f, 0.0f, 0.0f};
        const float sc_l = (scaled && have) ? e.scale[ti_l] : 1.0f;
        OctTrace o_l{};
        if constexpr (MODEL == HSS_OCT) o_l = oct_trace<true>(g_l.h, g_l.m, e.h0);
        const int nchunk = min(kWave, e.cnt - j0);
        const unsigned long long all = nchunk == kWave ? ~0ull : (1ull << nchunk) - 1;

        // the windows of the traces in `todo` (bits of the chunk, in increasing order);
        // time(jj, t, keep) gives a trace's traveltimes and whether the lane keeps it
        auto visit = [&](unsigned long long todo, auto &&time) {
            for (; todo; todo &= todo - 1) {
                const int jj = __builtin_ctzll(todo);
                const size_t trace0 =
                    (size_t)__builtin_amdgcn_readlane(ti_l, jj) * (size_t)e.ns;
                const float sc = scaled ? bcast(sc_l, jj) : 1.0f;
                float t[CPL], f[CPL], y[CPL][W + 1];
                bool use[CPL];
                time(jj, t, use);
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    int kk;
                    const bool in = window_k<true>(t[c], dt_v, inv_v, e.ib, &kk, &f[c]);
                    use[c] = use[c] & in & active & on[c];
                    const uint32_t first = use[c] ? (uint32_t)(kk - e.tau) : 0u;
                    if constexpr (STORAGE == HSS_F32) {
                        const float *p = (const float *)at_bytes((const float *)e.samples + trace0,
                                                                 4u * first);
#pragma unroll
                        for (int j = 0; j <= W; ++j) y[c][j] = p[j];
                    } else {
                        const unsigned rpar = (unsigned)trace0 & 1u;
                        read16<STORAGE, W>(
                            (const uint32_t *)((const uint16_t *)e.samples + (trace0 - rpar)),
                            rpar, first, y[c]);
                    }
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    if (!use[c]) continue;
                    if constexpr (STORAGE != HSS_F32) {
                        // as the wave segments decode and scale (1 on a line without scales)
                        if (scaled) {
#pragma unroll
                            for (int j = 0; j <= W; ++j) y[c][j] = y[c][j] * sc;
                        }
                    }
                    acc[c].sum(y[c], f[c], c);
                    acc[c].used++;
                }
            }
        };

        if constexpr (MODEL == HSS_OCT) {
            if (!by_runs) {
                visit(all, [&](int j, float (&t)[CPL], bool (&keep)[CPL]) {
                    OctTrace ot{};
                    ot.h = bcast(o_l.h, j);
                    ot.m = bcast(o_l.m, j);
                    bcast_oct_mid_terms(ot, o_l, j);
                    bcast_oct_time_terms(ot, o_l, j);
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        bool r;
                        t[c] = 0.0f;
                        keep[c] = oct_traveltime<true>(ot, oc[c], e.m0, e.apm, &t[c], &r);
                        rej += r & active & on[c];
                    }
                });
                continue;
            }
            const uint32_t hkey_l = __float_as_uint(g_l.h);
            for (int jj = 0; jj < nchunk;) {
                // the run jj .. je-1 of traces with trace jj's half offset (its bit pattern)
                const uint32_t key = (uint32_t)__builtin_amdgcn_readlane((int)hkey_l, jj);
                const unsigned long long from = all & (~0ull << jj);
                const unsigned long long differ = __builtin_amdgcn_ballot_w64(hkey_l != key) & from;
                const unsigned long long run = from & (differ ? (differ & -differ) - 1 : ~0ull);
                OctTrace ot{};
                ot.h = bcast(o_l.h, jj);
                bcast_oct_mid_terms(ot, o_l, jj);
                OctMid om[CPL];
                unsigned long long todo = 0;
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    om[c] = oct_mid<true>(ot, oc[c], e.m0);
                    const bool ok = !om[c].bad & active & on[c];
                    if (__builtin_amdgcn_ballot_w64(ok & (om[c].mh != om[c].mh)) != 0) {
                        todo = run;  // a NaN displaced midpoint keeps every trace
                    } else if (__builtin_amdgcn_ballot_w64(ok) != 0) {
                        const float least = wave_min_f(ok ? om[c].mh : INFINITY);
                        const float most = wave_max_f(ok ? om[c].mh : -INFINITY);
                        todo |= run & __builtin_amdgcn_ballot_w64(!(g_l.m - least < -e.apm) &
                                                                  !(g_l.m - most > e.apm));
                    }
                }
                // (the traces left out are rejected by every lane)
                const unsigned skipped = (unsigned)__builtin_popcountll(run & ~todo);
                OctTime otm[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    rej += active & on[c] ? skipped : 0u;
                    otm[c] = OctTime{0.0f, 0.0f, true};
                }
                if (todo != 0) {
                    bcast_oct_time_terms(ot, o_l, jj);
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
                        otm[c] = oct_time_terms<true>(ot, oc[c], e.m0, om[c]);
                    visit(todo, [&](int j, float (&t)[CPL], bool (&keep)[CPL]) {
                        const float m = bcast(g_l.m, j);
#pragma unroll
                        for (int c = 0; c < CPL; ++c) {
                            bool r;
                            keep[c] = oct_traveltime_at(om[c], otm[c], m, e.apm, &t[c], &r);
                            rej += r & active & on[c];
                        }
                    });
                }
                jj = differ ? __builtin_ctzll(differ) : nchunk;
            }
        } else if constexpr (MODEL == HSS_ZOCRS) {
            visit(all, [&](int j, float (&t)[CPL], bool (&keep)[CPL]) {
                const float m = bcast(g_l.m, j), h2 = bcast(g_l.h2, j);
                const uint32_t key = __float_as_uint(m);
                if (!zvalid || key != zkey) {
#pragma unroll
                    for (int c = 0; c < CPL; ++c) zmid[c] = zocrs_mid_part(t0, m - e.m0, k[c]);
                    zkey = key;
                    zvalid = true;
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    t[c] = 0.0f;
                    keep[c] = zocrs_time_from<true>(zmid[c], k[c].c * h2, &t[c]);
                }
            });
        } else {
            visit(all, [&](int j, float (&t)[CPL], bool (&keep)[CPL]) {
                const float h2 = bcast(g_l.h2, j);
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    t[c] = sqrt_time<true, false>(t0sq + k[c].c * h2);
                    keep[c] = true;
                }
            });
        }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[c].reduce(e.w, &S[c], &stack[c]);
    *rejected += rej;
}

}  // namespace hss
