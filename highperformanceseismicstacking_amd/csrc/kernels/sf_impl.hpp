// Stretch-free re-stack with the best-shift pick fused in.
//
// Reference behaviour (cmp/stretch_free.cu:4-66, zocrs/stretch_free.cu:4-85,
// oct/stretch_free.cu:5-97, then common/stretch_free.cu:3-35): for every t0 sample s and
// every shift n of nArray (-10..10, StretchFreeAlgorithm.cpp:77-82) take the parameters
// picked earlier at sample s_n = s - n (velocity as v, c_n = 4/v^2), evaluate the
// traveltime at t0_n = s_n*dt and shift it by n*dt; a shift whose s_n falls outside the
// trace gives S = stack = 0.  The first strict maximum over the shifts wins and the
// result is (S, stack, n).
//
// MI355X mapping: one workgroup = (midpoint, `tile` consecutive t0 samples), whose lanes take
// the tile's (sample, shift) pairs, the shift fastest, samples and shifts rising together: lane
// pair (r, n) is sample r + n modulo the tile.  But for one jump at the wrap, the lanes of a
// row share the source sample s - n, so neighbouring lanes hold one candidate at times n*dt
// apart and read windows of the same traces one sample apart: a wave's window load touches the
// few lines around three or four source samples' windows where a lane per t0 sample, each with
// another sample's parameters, touched a line per lane (36 lines per load, 1.45 per clock and
// CU, on a 256-midpoint CMP line; 21 here).  Every pair's (S, stack) goes to LDS, and one
// thread per sample takes the first strict maximum.  Measured, 21 shifts: that line, FP32,
// w = 15, 1.90 -> 1.55 ms; ZO-CRS, 100 midpoints, BF16, 5.3 -> 5.1 ms; OCT, 2 midpoints, FP16,
// 0.69 -> 0.25 ms.  VALU issue bounds it then (77% of the cycles).
#pragma once

#include <algorithm>

#include "eval.hpp"
#include "eval_compact.hpp"
#include "eval_runs.hpp"
#include "grid_impl.hpp"
#include "launch_util.hpp"

namespace hss {

constexpr int kSfMaxShifts = 64;
constexpr int kSfWaves = 8;
constexpr int kSfThreads = kSfWaves * kWave;
// (sample, shift) pairs of a workgroup, as many as the largest shift list has in a 64-sample
// tile: 32 KB of dynamic LDS, for OCT beside 45 KB of run lists (78 of a CU's 160 KB).
constexpr int kSfPairs = 4096;
static_assert(kSfPairs * sizeof(float2) + sizeof(OctRuns) + 2 * kSfMaxShifts * sizeof(int) <=
                  160 * 1024,
              "a workgroup's LDS");
// Lanes read windows per lane (Window::add16 for 16-bit storage): they belong to several
// candidates, so a trace's windows spread over more than one wave segment.
constexpr bool kSfSegments = false;

struct SfArgs {
    EvalCtx e;
    const int *mbeg;
    const int *mcnt;
    const float *mm0;
    const int *morder;  // launch order (launch_midpoint) or NULL
    int nmid;
    const float *vparams;  // [n][np][ns]: velocity, then A,B or slope, per sample
    float nvals[kSfMaxShifts];
    int nN;
    int tile, wg_per_mid;
    float *result;  // [n][3][ns]
    float *sembl;   // [n][ns][nN] or NULL
    float *stack;
    unsigned long long *not_used;
};

// The budget of OCT's kernel, which holds both trace loops (with and without the kept
// offset terms): six waves per SIMD for windows of up to 11 samples, where both loops fit
// without spills (the C4 line's w = 11: the loop in the reference's order would otherwise
// take 81 registers, five waves); wider and generic windows at the compiler's own count.
template <int MODEL, int W, int VARIANT>
constexpr int sf_min_waves() {
    return MODEL == HSS_OCT && VARIANT != HSS_KAHAN && W > 0 && W <= 11 ? 6 : 1;
}

template <int MODEL, int W, int VARIANT, int STORAGE>
__global__ __launch_bounds__(kSfThreads)
__attribute__((amdgpu_waves_per_eu(sf_min_waves<MODEL, W, VARIANT>(), 8))) void sf_semblance_kernel(SfArgs a) {
    constexpr int NP = MODEL == HSS_CMP ? 1 : (MODEL == HSS_ZOCRS ? 3 : 2);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int blk = logical_block(blockIdx.x, gridDim.x);
    const int slot = blk / a.wg_per_mid;
    const int g = launch_midpoint(a.morder, a.nmid, slot);
    if (g < 0) return;  // (the whole workgroup)
    const int ns = a.e.ns, nN = a.nN;
    const int s0 = (blk - slot * a.wg_per_mid) * a.tile;
    const int s1 = min(s0 + a.tile, ns);
    const EvalCtx e = midpoint_ctx(a.e, a.mbeg, a.mcnt, a.mm0, g);
    const float *vp = a.vparams + (size_t)g * NP * ns;

    extern __shared__ float2 sf_pairs[];  // [tile][nN] (S, stack)
    __shared__ int shift_of[kSfMaxShifts], wrapped[kSfMaxShifts];  // n, n modulo the tile
    constexpr bool kRuns = MODEL == HSS_OCT && VARIANT != HSS_KAHAN;
    // OCT: the midpoint's offset runs, or the waves' records of a chunk of traces (eval_runs)
    union OctLists {
        OctRuns runs;
        OctTraceRec chunk[kSfWaves][kWave];
    };
    __shared__ std::conditional_t<kRuns, OctLists, int> oct_lists;
    for (int q = (int)threadIdx.x; q < nN; q += (int)blockDim.x) {
        const int n = (int)a.nvals[q];
        shift_of[q] = n;
        wrapped[q] = n % a.tile + (n % a.tile < 0 ? a.tile : 0);
    }
    bool by_runs = false;
    if constexpr (kRuns) by_runs = load_oct_runs(e, STORAGE == HSS_F32 ? 4 : 2, oct_lists.runs);
    __syncthreads();
    unsigned long long rejected = 0;
    // OCT: keep the offset-dependent traveltime terms across runs of traces with one half
    // offset when the midpoint's list is grouped by offset (wave-uniform); the kept terms are
    // per lane, as the candidates are
    bool keep = false;
    if constexpr (MODEL == HSS_OCT) keep = by_runs || oct_offset_runs_long(e);
    // a BF16 line stored without scales sums its windows as FP32 windows; both choices are
    // made outside the trace loop, one code path each
    const bool unscaled16 = STORAGE == HSS_BF16 && e.scale == nullptr;
    const int pairs = a.tile * nN;
    for (int p0 = wave * kWave; p0 < pairs; p0 += (int)blockDim.x) {
        const int p = p0 + lane;
        const int row = p / nN, q = p - row * nN;
        const int n = shift_of[q];
        const int at = row + wrapped[q];
        const int s = s0 + (at < a.tile ? at : at - a.tile);
        const int sn = s - n;  // the source sample
        const bool mine = p < pairs && s < s1;
        const bool valid = mine && sn >= 0 && sn < ns;
        if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
        const int sc = valid ? sn : 0;
        Candidate k{0.0f, 0.0f, 0.0f};
        const float v = vp[sc];
        k.c = 4.0f / (v * v);
        if constexpr (MODEL == HSS_ZOCRS) {
            k.p1 = vp[ns + sc];
            k.p2 = vp[2 * ns + sc];
        } else if constexpr (MODEL == HSS_OCT) {
            k.p1 = vp[ns + sc];
        }
        const float t0n = (float)sc * e.dt;
        const float shift = (float)n * e.dt;
        float S = 0.0f, stk = 0.0f;
        unsigned rej = 0;  // on the wave's lowest valid lane
        auto eval = [&](auto keep_c, auto factored_c) {
            evaluate<MODEL, W, VARIANT, STORAGE, true, kSfSegments, decltype(keep_c)::value,
                     decltype(factored_c)::value>(e, t0n, t0n * t0n, k, shift, valid, nullptr, &S,
                                                  &stk, &rej);
        };
        using T = std::true_type;
        using F = std::false_type;
        bool walked = false;
        if constexpr (kRuns) {
            if (keep) {
                // each lane walks only the traces its own aperture keeps (the walks of
                // differential evolution; the same sums in the same order)
                const Candidate kc[1] = {k};
                const bool on[1] = {true};
                float S1[1], T1[1];
                if (by_runs)
                    evaluate_oct_runs<W, VARIANT, STORAGE, true, 1>(
                        e, oct_lists.runs, t0n, kc, on, shift, valid, S1, T1, &rej);
                else
                    evaluate_oct_compact<W, VARIANT, STORAGE, true, 1>(
                        e, t0n, kc, on, shift, valid, oct_lists.chunk[wave], S1, T1, &rej);
                S = S1[0];
                stk = T1[0];
                walked = true;
            }
        }
        if (walked) {
        } else if (MODEL == HSS_OCT && keep) {
            if (unscaled16)
                eval(T{}, F{});
            else
                eval(T{}, T{});
        } else if (unscaled16) {
            eval(F{}, F{});
        } else {
            eval(F{}, T{});
        }
        rejected += rej;
        if (mine) {
            if (!valid) {
                S = 0.0f;
                stk = 0.0f;
            }
            sf_pairs[(s - s0) * nN + q] = float2{S, stk};
            if (a.sembl) a.sembl[((size_t)g * ns + s) * nN + q] = S;
            if (a.stack) a.stack[((size_t)g * ns + s) * nN + q] = stk;
        }
    }
    if (MODEL == HSS_OCT && a.not_used) {
        const unsigned long long tot = wave_sum_u64(rejected);
        if (lane == 0 && tot) atomicAdd(a.not_used + g, tot);
    }
    __syncthreads();
    for (int s = s0 + (int)threadIdx.x; s < s1; s += (int)blockDim.x) {
        float best = -1.0f, bstack = 0.0f;
        int bidx = -1;
        for (int q = 0; q < nN; ++q) {
            const float2 r = sf_pairs[(s - s0) * nN + q];
            if (r.x > best) {
                best = r.x;
                bstack = r.y;
                bidx = q;
            }
        }
        float *res = a.result + (size_t)g * 3 * ns;
        res[s] = best;
        res[ns + s] = bidx >= 0 ? bstack : 0.0f;
        res[2 * ns + s] = bidx >= 0 ? a.nvals[bidx] : 0.0f;
    }
}

// The launch's tile: 64 samples, fewer (down to 16) where their pairs do not fit kSfPairs or
// the launch would have fewer than kSfWorkgroups.  (CMP, 256 midpoints, FP32, w = 15: tiles of
// 32/64/128/256 1.83/1.67/1.72/1.68 ms.)
constexpr int kSfTile = 64;
constexpr long long kSfWorkgroups = 1024;
// Waves of a workgroup: four per SIMD pair up evenly, so eight, which read one tile's windows
// together, or four where the registers (the compensated sums above 9 samples, the runtime-w
// kernel) leave so few waves per SIMD that whole workgroups of eight waste them, in launches
// that fill the chip.  Five to seven, which leave fewer lanes idle in the last round over the
// pairs, load the SIMDs unevenly: 21 shifts, seven | eight | four waves, in ms, CMP, 300
// midpoints, FP16, w = 7 1.09 | 0.99 | 1.00, FP16, EXACT, w = 11 2.23 | 2.10 | 2.11, FP32, w = 15
// 1.25 | 1.24 | 1.26; compensated, BF16, w = 13 1.52 | 1.41 | 1.22; ZO-CRS, BF16, w = 11, 60
// midpoints 3.01 | 2.65 | 2.81, 400 midpoints 15.9 | 14.4 | 15.3; OCT, FP16, w = 11, 100
// midpoints 3.2 | 3.0 | 4.8 (every workgroup reads the midpoint's list).
template <int MODEL, int W, int VARIANT>
constexpr int sf_waves(long long workgroups) {
    const bool few = MODEL != HSS_OCT && (W == 0 || (VARIANT == HSS_KAHAN && W > 9));
    return few && workgroups >= kSfWorkgroups ? 4 : kSfWaves;
}
inline int sf_tile(long long n_mid, int ns, int nN) {
    int tile = kSfTile;
    while (tile > 16 &&
           (tile * nN > kSfPairs || n_mid * ((ns + tile - 1) / tile) < kSfWorkgroups))
        tile /= 2;
    return tile;
}

template <int MODEL>
int launch_sf(const SfArgs &args, int n_mid, int variant, int storage, hipStream_t stream) {
    int st = HSS_OK;
    SfArgs a = args;
    a.tile = sf_tile(n_mid, a.e.ns, a.nN);
    a.wg_per_mid = (a.e.ns + a.tile - 1) / a.tile;
    const unsigned long long blocks = (unsigned long long)n_mid * (unsigned long long)a.wg_per_mid;
    if (blocks > 0x7fffffffull) return HSS_ERR_INVALID_SIZE;
    if (blocks == 0) return HSS_OK;
    const unsigned lds = (unsigned)(a.tile * a.nN) * sizeof(float2);
    const int need = (a.tile * a.nN + kWave - 1) / kWave;
    int rc = dispatch_storage(storage, [&](auto S) {
        st = dispatch_variant(variant, [&](auto V) {
            // (dt: see sqrt_time)
            const bool fast = a.e.dt >= 0x1.0p-20f && fast_index_verified(a.e.dt, a.e.tau, stream);
            dispatch_window(a.e.w, fast, [&](auto Wc) {
                constexpr int VV = decltype(V)::value,
                              WW = window_of<decltype(Wc)::value, VV, true>();
                const int waves = std::min(sf_waves<MODEL, WW, VV>((long long)blocks), need);
                hipLaunchKernelGGL((sf_semblance_kernel<MODEL, WW, VV, decltype(S)::value>),
                                   dim3((unsigned)blocks), dim3((unsigned)(waves * kWave)), lds,
                                   stream, a);
            });
        });
    });
    if (rc != HSS_OK) return rc;
    if (st != HSS_OK) return st;
    return hip_status(hipGetLastError());
}

int launch_sf_cmp(const SfArgs &a, int n_mid, int variant, int storage, hipStream_t stream);
int launch_sf_zocrs(const SfArgs &a, int n_mid, int variant, int storage, hipStream_t stream);
int launch_sf_oct(const SfArgs &a, int n_mid, int variant, int storage, hipStream_t stream);

}  // namespace hss
