// Trace selection masks for a batch of midpoints over a whole line.
//
// Reference behaviour:
//   CMP    mask = (m0 == m)                         cmp/common.cu:3-15
//   ZO-CRS mask = |m0 - m| <= apm                   zocrs/common.cu:3-16
//   OCT    mask = some (t0 sample, candidate) has no displaced-midpoint error and
//          |m - mh| <= apm, scanning t0 then candidates with an early exit.  The
//          candidates are
//            grid:          the same (c, slope) pairs for every t0 (1024 random draws,
//                           oct/linear_search.cu:155-192);
//            stretch-free:  the (v, slope) picked at that very t0 (oct/stretch_free.cu:99-138);
//            DE:            the start population of that t0 (oct/differential_evolution.cu:130-168).
//
// CMP and ZO-CRS: each thread owns one (trace, midpoint).
//
// For OCT a trace whose midpoint distance exceeds apm + sqrt(h^2 + h0^2) cannot pass for any
// candidate: the displaced midpoint
// satisfies |mh - m0| = 2|theta||h^2-h0^2| / sqrt(theta^2 gamma^2 + 2q + 2sqrt(...))
// <= |h^2-h0^2| / sqrt(h^2+h0^2) <= sqrt(h^2+h0^2), because the denominator is at least
// |theta| gamma = 2|theta| sqrt(h^2+h0^2).  The test keeps a wide rounding margin, so it
// only skips traces whose answer is certain.
#include <algorithm>

#include "de_impl.hpp"

namespace hss {

struct SelectArgs {
    const float *mid;
    const float *hoff;
    int ntr;
    int ns;
    float dt;
    const float *m0;
    int n;
    float apm, h0;
    int model;
    hss_oct_candidates oct;
    uint32_t key0, key1;
    unsigned char *mask;
};

constexpr int kSelectThreads = 256;

// The first test of an OCT trace: a midpoint distance beyond apm + sqrt(h^2 + h0^2)
// (plus the rounding margin) cannot pass for any candidate.
__device__ __forceinline__ bool oct_within_reach(float m, float h, float m0, float h0, float apm) {
    const float reach = sqrtf(h * h + h0 * h0);
    const float margin = 1e-4f * (fabsf(m0) + fabsf(m) + reach + apm) + 1e-3f;
    return fabsf(m - m0) <= apm + reach + margin;
}

// Candidates per t0 sample of one midpoint, in each mode.
__device__ __forceinline__ int oct_candidates_per_sample(const SelectArgs &a) {
    return a.oct.mode == HSS_OCT_PER_SAMPLE ? 1
         : (a.oct.mode == HSS_OCT_DE_START ? a.oct.NP : a.oct.npairs);
}

// Candidate p of t0 sample s of midpoint g as (c, slope).
__device__ __forceinline__ void oct_candidate(const SelectArgs &a, int g, int s, int p, float *c,
                                              float *slope) {
    if (a.oct.mode == HSS_OCT_PAIRS) {
        *c = a.oct.d_pairs[2 * p];
        *slope = a.oct.d_pairs[2 * p + 1];
    } else if (a.oct.mode == HSS_OCT_PER_SAMPLE) {
        const float *vp = a.oct.d_vparams + (size_t)g * 2 * a.ns;
        const float v = vp[s];
        *c = 4.0f / (v * v);
        *slope = vp[a.ns + s];
    } else {
        // the start population of differential evolution (de_impl.hpp)
        uint32_t r[4];
        philox4x32_10((uint32_t)s, a.oct.stream_base + (uint32_t)g, (uint32_t)p, 0u, a.key0,
                      a.key1, r);
        const float v = a.oct.lower[0] + u01(r[0]) * (a.oct.upper[0] - a.oct.lower[0]);
        *c = 4.0f / (v * v);
        *slope = a.oct.lower[1] + u01(r[1]) * (a.oct.upper[1] - a.oct.lower[1]);
    }
}

// OCT.  What a candidate at a t0 does to a trace, mh = m0 + d, depends on the trace's half
// offset alone through the displacement d, and |m - mh| <= apm rounds monotonically in d: the
// displacements a trace accepts are an interval.  A workgroup takes a block of traces, a
// group of midpoints with the same candidates (pairs: many midpoints; the other modes: one)
// and a slice of the (t0, candidate) list.  It lists the block's distinct half offsets
// (rows), works out each displacement of the slice once per row, and keeps for each row
// kBins/rows bins over [-sqrt(h^2+h0^2), +sqrt(h^2+h0^2)], each with the smallest and largest
// displacement in it.  A trace then looks at the few bins its interval reaches: the exact
// test at a bin's two ends answers for the whole bin unless the interval lies strictly
// between them (an aperture narrower than a bin): the pairs of trace and midpoint left open
// so are tested against the slice's displacements one by one (select_oct_scan).
// The slices only ever set mask bytes that a first launch cleared, so they need not know of
// each other.
//
// The masks are those of testing every (trace, midpoint, t0, candidate) one by one, at one
// displacement per (t0, candidate, offset of the block) in place of one per midpoint and
// 256-trace workgroup.  What bounds it is VALU work on the displacements (three square roots
// and a division each).  Measured, 30 midpoints x 4832 traces, 1024 pairs at 1251 t0: 161 ->
// 0.31 ms; 60 midpoints with start populations of 48: 7.8 -> 0.49 ms.  About as much time
// again as the displacements take goes into the slices' looks at the traces: 256 workgroups of
// 1024 threads measured 0.31 ms, 1024 of 256 threads, which look four times as often, 0.64.
//
// A block with more than kRowsMax offsets goes through them kRowsMax at a time, and one with
// more than kOffsetsMax (offsets that hardly repeat) tests trace by trace, each candidate
// drawn once per workgroup.
constexpr int kRowsMax = 64;
constexpr int kBins = 4096;
constexpr int kOffsetsMax = 1024;
constexpr int kSlots = 2 * kOffsetsMax;  // open-addressed table of the block's offsets
constexpr int kOctThreads = 1024;
constexpr int kTracesPerThread = 4;
constexpr int kBlockTraces = kOctThreads * kTracesPerThread;
constexpr int kPairMidpoints = 64;       // midpoints of a group in pairs mode (bits of a word)

// Floats as unsigned integers of the same order.
__device__ __forceinline__ uint32_t order_key(float x) {
    const uint32_t b = __float_as_uint(x);
    return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float order_value(uint32_t k) {
    return __uint_as_float(k ^ ((k >> 31) ? 0x80000000u : 0xffffffffu));
}

struct OctRows {
    unsigned long long slot[kSlots];  // 1 << 32 | the offset's bits; 0: empty
    int number[kSlots];  // the offset's number; row = number - the pass's first
    float h[kOffsetsMax];
    float low[kRowsMax], per_unit[kRowsMax];  // the bins' start and bins per unit of d
    union {
        struct {
            uint32_t least[kBins], most[kBins];  // order keys; least > most: empty
        };
        float scan[2 * kBins];  // select_oct_scan: rows of displacements
    };
    unsigned long long filled[kBins / 64];    // bit b of word w: bin 64*w + b is not empty
    int n;
};

__device__ __forceinline__ int offset_slot(const OctRows &t, uint32_t bits) {
    int k = (int)((bits * 0x9e3779b1u) >> 16) % kSlots;
    while (t.slot[k] != ((1ull << 32) | bits)) k = (k + 1) % kSlots;
    return k;
}

__device__ __forceinline__ int bin_of(float d, float low, float per_unit, int nbins) {
    return (int)fminf(fmaxf((d - low) * per_unit, 0.0f), (float)(nbins - 1));
}

// The exact test, by the side a displacement misses on: 0 inside the aperture, +1 too far
// down (m - mh > apm), -1 too far up, 2 for a NaN.
__device__ __forceinline__ int oct_side(float m, float m0, float d, float apm) {
    const float x = m - (m0 + d);
    if (fabsf(x) <= apm) return 0;
    return x > apm ? 1 : (x < -apm ? -1 : 2);
}

// The exact test of (trace, midpoint) pairs the bins leave open: bit g of unsure[j] is midpoint
// g0 + g of trace i0 + kOctThreads*j + tid.  The slice's displacements are worked out a chunk at
// a time into LDS, once per row, and every open pair looks at every one of its row's: 30
// midpoints x 4832 traces, 1024 pairs, apertures of 2/1/0 m 10/20/57 ms.  (376/533/632 ms when
// each open pair worked the displacements out for itself, 138/161/185 ms in the kernel before
// the bins.)
__device__ void select_oct_scan(const SelectArgs &a, OctRows &t, int i0, int g0, int first,
                                int rows, int NP, long long qa, long long qb,
                                unsigned long long (&unsure)[kTracesPerThread]) {
    const int tid = (int)threadIdx.x;
    // a row of the table has an odd length: the lanes of a wave read one place of many rows
    const int stride = (2 * kBins / rows - 1) | 1, chunk = stride - 1;
    for (long long q0 = qa; q0 < qb; q0 += chunk) {
        unsigned long long open = 0;
        for (int j = 0; j < kTracesPerThread; ++j) open |= unsure[j];
        if (!__syncthreads_or(open != 0)) return;  // (also before the table is written again)
        const int n = (int)min((long long)chunk, qb - q0);
        for (int k = tid; k < n * rows; k += kOctThreads) {
            const int row = k / n, at = k - row * n;
            const int s = (int)((q0 + at) / NP), p = (int)(q0 + at - (long long)s * NP);
            float c, slope, d;
            oct_candidate(a, g0, s, p, &c, &slope);
            const int err = oct_displacement(t.h[first + row], a.h0, (float)s * a.dt, c, slope, &d);
            t.scan[row * stride + at] = err == kNoError ? d : __int_as_float(0x7fc00000);
        }
        __syncthreads();
        for (int j = 0; j < kTracesPerThread; ++j) {
            if (unsure[j] == 0) continue;
            const int i = i0 + j * kOctThreads + tid;
            const float m = a.mid[i];
            const int row = t.number[offset_slot(t, __float_as_uint(a.hoff[i]))] - first;
            const float *d = t.scan + row * stride;
            for (unsigned long long rest = unsure[j]; rest != 0; rest &= rest - 1) {
                const int g = g0 + __builtin_ctzll(rest);
                const float m0 = a.m0[g];
                bool used = false;
                for (int k = 0; k < n; ++k) used |= oct_side(m, m0, d[k], a.apm) == 0;
                if (!used) continue;
                a.mask[(size_t)g * a.ntr + i] = 1;
                unsure[j] &= ~(rest & -rest);
            }
        }
    }
}

// Every trace of the block tests the slice's candidates, kOctThreads of them at a time, which
// the workgroup's threads draw into LDS; a midpoint is done when no trace is open.
__device__ void select_oct_one_by_one(const SelectArgs &a, int i0, int g0, int g1,
                                      unsigned reached, int NP, long long qa, long long qb,
                                      uint32_t *cand_c, uint32_t *cand_s) {
    const int tid = (int)threadIdx.x;
    for (int g = g0; g < g1; ++g) {
        const float m0 = a.m0[g];
        unsigned open = 0;
        for (int j = 0; j < kTracesPerThread; ++j) {
            const int i = i0 + j * kOctThreads + tid;
            if (((reached >> j) & 1) && oct_within_reach(a.mid[i], a.hoff[i], m0, a.h0, a.apm))
                open |= 1u << j;
        }
        for (long long q0 = qa; q0 < qb; q0 += kOctThreads) {
            if (!__syncthreads_or(open != 0)) break;  // (also before LDS is written again)
            const long long q = q0 + tid;
            if (q < qb) {
                const int s = (int)(q / NP), p = (int)(q - (long long)s * NP);
                float c, slope;
                oct_candidate(a, g, s, p, &c, &slope);
                cand_c[tid] = __float_as_uint(c);
                cand_s[tid] = __float_as_uint(slope);
            }
            __syncthreads();
            const int n = (int)min((long long)kOctThreads, qb - q0);
            for (int j = 0; j < kTracesPerThread; ++j) {
                if (!((open >> j) & 1)) continue;
                const int i = i0 + j * kOctThreads + tid;
                const float m = a.mid[i], h = a.hoff[i];
                int s = (int)(q0 / NP), p = (int)(q0 - (long long)s * NP);
                for (int k = 0; k < n; ++k) {
                    float d;
                    if (oct_displacement(h, a.h0, (float)s * a.dt, __uint_as_float(cand_c[k]),
                                         __uint_as_float(cand_s[k]), &d) == kNoError &&
                        oct_side(m, m0, d, a.apm) == 0) {
                        a.mask[(size_t)g * a.ntr + i] = 1;
                        open &= ~(1u << j);
                        break;
                    }
                    if (++p == NP) {
                        p = 0;
                        ++s;
                    }
                }
            }
        }
        __syncthreads();  // before the next midpoint's candidates
    }
}

__global__ __launch_bounds__(kOctThreads) void select_oct_kernel(SelectArgs a, int group,
                                                                    int slices) {
    __shared__ OctRows t;
    __shared__ int overflow;
    const int tid = (int)threadIdx.x;
    const int i0 = (int)blockIdx.x * kBlockTraces;
    const int i1 = min(a.ntr, i0 + kBlockTraces);
    const int g0 = (int)blockIdx.y * group, g1 = min(a.n, g0 + group);
    const int NP = oct_candidates_per_sample(a);
    const long long total = (long long)a.ns * NP;
    const long long qa = total * (int)blockIdx.z / slices;
    const long long qb = total * ((int)blockIdx.z + 1) / slices;
    if (qa >= qb) return;  // (uniform)

    // the distinct offsets of the block's traces that some midpoint of the group can reach
    for (int k = tid; k < kSlots; k += kOctThreads) t.slot[k] = 0;
    if (tid == 0) overflow = 0;
    __syncthreads();
    unsigned reached = 0;  // bit j: trace i0 + kOctThreads*j + tid
    for (int j = 0; j < kTracesPerThread; ++j) {
        const int i = i0 + j * kOctThreads + tid;
        if (i >= i1) break;
        const float m = a.mid[i], h = a.hoff[i];
        bool any = false;
        for (int g = g0; g < g1 && !any; ++g) any = oct_within_reach(m, h, a.m0[g], a.h0, a.apm);
        if (!any) continue;
        reached |= 1u << j;
        const unsigned long long key = (1ull << 32) | __float_as_uint(h);
        int k = (int)((__float_as_uint(h) * 0x9e3779b1u) >> 16) % kSlots;
        int tries = 0;
        for (; tries < kSlots; ++tries, k = (k + 1) % kSlots) {
            const unsigned long long was = atomicCAS(&t.slot[k], 0ull, key);
            if (was == 0ull || was == key) break;
        }
        if (tries == kSlots) overflow = 1;
    }
    __syncthreads();
    if (tid < kWave) {  // number the used slots
        int n = 0;
        for (int k0 = 0; k0 < kSlots; k0 += kWave) {
            const unsigned long long key = t.slot[k0 + tid];
            const unsigned long long used = __builtin_amdgcn_ballot_w64(key != 0);
            const int number = n + __builtin_popcountll(used & ((1ull << tid) - 1));
            t.number[k0 + tid] = number;
            if (key != 0 && number < kOffsetsMax) t.h[number] = __uint_as_float((uint32_t)key);
            n += __builtin_popcountll(used);
        }
        if (tid == 0) {
            t.n = n;
            if (n > kOffsetsMax) overflow = 1;
        }
    }
    __syncthreads();
    const int offsets = t.n;
    if (offsets == 0) return;  // (uniform, as `overflow` is)
    if (overflow) {
        select_oct_one_by_one(a, i0, g0, g1, reached, NP, qa, qb, t.least, t.most);
        return;
    }
    const int passes = (offsets + kRowsMax - 1) / kRowsMax;
    const int per_pass = (offsets + passes - 1) / passes;
    const int nbins = per_pass <= kRowsMax / 4 ? kBins / (kRowsMax / 4) : kBins / kRowsMax;
    for (int first = 0; first < offsets; first += per_pass) {
        const int rows = min(per_pass, offsets - first);
        for (int k = tid; k < kBins; k += kOctThreads) {
            t.least[k] = 0xffffffffu;
            t.most[k] = 0;
        }
        if (tid < rows) {
            const float h = t.h[first + tid];
            const float r = sqrtf(h * h + a.h0 * a.h0);
            t.low[tid] = -r;
            t.per_unit[tid] = r > 0.0f && r < INFINITY ? (float)nbins / (2.0f * r) : 0.0f;
        }
        __syncthreads();

        // the slice's displacements, each thread its own candidates
        for (long long q = qa + tid; q < qb; q += kOctThreads) {
            const int s = (int)(q / NP), p = (int)(q - (long long)s * NP);
            float c, slope;
            oct_candidate(a, g0, s, p, &c, &slope);
            const float t0 = (float)s * a.dt;
            for (int row = 0; row < rows; ++row) {
                float d;
                if (oct_displacement(t.h[first + row], a.h0, t0, c, slope, &d) != kNoError ||
                    d != d)
                    continue;
                const int b = row * nbins + bin_of(d, t.low[row], t.per_unit[row], nbins);
                const uint32_t key = order_key(d);
                if (key < t.least[b]) atomicMin(&t.least[b], key);
                if (key > t.most[b]) atomicMax(&t.most[b], key);
            }
        }
        __syncthreads();
        for (int k = tid; k < kBins; k += kOctThreads) {
            const unsigned long long w = __builtin_amdgcn_ballot_w64(t.least[k] <= t.most[k]);
            if ((k & 63) == 0) t.filled[k / 64] = w;
        }
        __syncthreads();

        unsigned long long left[kTracesPerThread];  // bit g - g0: the bins do not answer
        for (int j = 0; j < kTracesPerThread; ++j) {
            left[j] = 0;
            if (!((reached >> j) & 1)) continue;
            const int i = i0 + j * kOctThreads + tid;
            const float m = a.mid[i], h = a.hoff[i];
            const int row = t.number[offset_slot(t, __float_as_uint(h))] - first;
            if (row < 0 || row >= rows) continue;
            const float low = t.low[row], per_unit = t.per_unit[row];
            for (int g = g0; g < g1; ++g) {
                const float m0 = a.m0[g];
                if (!oct_within_reach(m, h, m0, a.h0, a.apm)) continue;
                // the bins of the accepted displacements, m - m0 -+ apm and a margin for
                // rounding
                const float margin = 1e-4f * (fabsf(m0) + fabsf(m) - low + a.apm) + 1e-3f;
                const int ba = bin_of(m - m0 - a.apm - margin, low, per_unit, nbins);
                const int bb = bin_of(m - m0 + a.apm + margin, low, per_unit, nbins);
                bool used = false, unsure = false;
                for (int b = ba; b <= bb && !used; ++b) {
                    const int bin = row * nbins + b;
                    const unsigned long long rest = t.filled[bin / 64] >> (bin & 63);
                    if (rest == 0) {  // on to the next word
                        b += 63 - (bin & 63);
                        continue;
                    }
                    b += __builtin_ctzll(rest);
                    if (b > bb) break;
                    const int at = row * nbins + b;
                    const int lo = oct_side(m, m0, order_value(t.least[at]), a.apm);
                    const int hi = oct_side(m, m0, order_value(t.most[at]), a.apm);
                    used = lo == 0 || hi == 0;
                    unsure = unsure || lo != hi;
                }
                if (used)
                    a.mask[(size_t)g * a.ntr + i] = 1;
                else if (unsure)
                    left[j] |= 1ull << (g - g0);
            }
        }
        select_oct_scan(a, t, i0, g0, first, rows, NP, qa, qb, left);
        __syncthreads();  // the bins are cleared next
    }
}

__global__ __launch_bounds__(kSelectThreads) void clear_mask_kernel(unsigned char *mask,
                                                                    unsigned long long bytes) {
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    unsigned long long b = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    // 16 bytes at a time from the first aligned address on
    const unsigned long long head = min(bytes, (unsigned long long)(-(uintptr_t)mask & 15u));
    const unsigned long long quads = (bytes - head) / 16;
    if (b < head) mask[b] = 0;
    if (b < bytes - head - quads * 16) mask[head + quads * 16 + b] = 0;
    for (; b < quads; b += stride) ((uint4 *)(mask + head))[b] = uint4{0, 0, 0, 0};
}

__global__ __launch_bounds__(kSelectThreads) void select_traces_kernel(SelectArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int g = blockIdx.y;
    if (i >= a.ntr) return;
    const float m0 = a.m0[g];
    const float m = a.mid[i];
    unsigned char used = 0;
    if (a.model == HSS_CMP)
        used = (m0 == m);
    else  // HSS_ZOCRS
        used = fabsf(m0 - m) <= a.apm;
    a.mask[(size_t)g * a.ntr + i] = used;
}

// OCT: clear the masks, then set them.  About kSelectWorkgroups workgroups share the (t0,
// candidate) list, slices of at least kSliceLeast (a slice costs its workgroup one look at
// every trace of the block for every midpoint of the group).
constexpr long long kSelectWorkgroups = 256, kSliceLeast = 1024;

static int select_oct(const SelectArgs &a, hipStream_t stream) {
    const unsigned long long bytes = (unsigned long long)a.n * (unsigned long long)a.ntr;
    const unsigned clear = (unsigned)std::min<unsigned long long>(
        (bytes / 16 + kSelectThreads) / kSelectThreads, 4096);
    hipLaunchKernelGGL(clear_mask_kernel, dim3(clear), dim3(kSelectThreads), 0, stream, a.mask,
                       bytes);
    int rc = hip_status(hipGetLastError());
    if (rc != HSS_OK) return rc;
    const int group = a.oct.mode == HSS_OCT_PAIRS ? kPairMidpoints : 1;
    const long long per_sample = a.oct.mode == HSS_OCT_PAIRS      ? a.oct.npairs
                                 : a.oct.mode == HSS_OCT_DE_START ? a.oct.NP
                                                                  : 1;
    const long long total = (long long)a.ns * per_sample;
    if (total == 0) return HSS_OK;
    const long long x = ((long long)a.ntr + kBlockTraces - 1) / kBlockTraces;
    const long long y = (a.n + group - 1) / group;
    const long long slices =
        std::max(1ll, std::min((kSelectWorkgroups + x * y - 1) / (x * y), total / kSliceLeast));
    hipLaunchKernelGGL(select_oct_kernel, dim3((unsigned)x, (unsigned)y, (unsigned)slices),
                       dim3(kOctThreads), 0, stream, a, group, (int)slices);
    return hip_status(hipGetLastError());
}

}  // namespace hss

using namespace hss;

extern "C" int hss_select_traces(const hss_traces *traces, int model, int32_t n, const float *d_m0,
                                 float apm, float h0, const hss_oct_candidates *oct,
                                 uint8_t *d_mask, void *stream) {
    if (!traces || !traces->mid || !traces->hoff || !d_mask) return HSS_ERR_NULL_POINTER;
    if (model_param_count(model) < 0) return HSS_ERR_INVALID_MODEL;
    if (n < 0 || traces->ntr < 0 || traces->ns <= 0 || n > 65535) return HSS_ERR_INVALID_SIZE;
    if (n > 0 && !d_m0) return HSS_ERR_NULL_POINTER;
    SelectArgs a{};
    a.mid = traces->mid;
    a.hoff = traces->hoff;
    a.ntr = traces->ntr;
    a.ns = traces->ns;
    a.dt = traces->dt;
    a.m0 = d_m0;
    a.n = n;
    a.apm = apm;
    a.h0 = h0;
    a.model = model;
    a.mask = d_mask;
    if (model == HSS_OCT) {
        if (!oct) return HSS_ERR_NULL_POINTER;
        a.oct = *oct;
        if (oct->mode == HSS_OCT_PAIRS) {
            if (oct->npairs < 0) return HSS_ERR_INVALID_SIZE;
            if (oct->npairs > 0 && !oct->d_pairs) return HSS_ERR_NULL_POINTER;
        } else if (oct->mode == HSS_OCT_PER_SAMPLE) {
            if (!oct->d_vparams) return HSS_ERR_NULL_POINTER;
        } else if (oct->mode == HSS_OCT_DE_START) {
            if (oct->NP <= 0) return HSS_ERR_INVALID_SIZE;
            a.key0 = (uint32_t)oct->seed;
            a.key1 = (uint32_t)(oct->seed >> 32);
        } else {
            return HSS_ERR_INVALID_MODEL;
        }
    }
    if (n == 0 || traces->ntr == 0) return HSS_OK;
    if (model == HSS_OCT) return select_oct(a, (hipStream_t)stream);
    dim3 grid((traces->ntr + kSelectThreads - 1) / kSelectThreads, n);
    hipLaunchKernelGGL(select_traces_kernel, grid, dim3(kSelectThreads), 0, (hipStream_t)stream, a);
    return hip_status(hipGetLastError());
}
