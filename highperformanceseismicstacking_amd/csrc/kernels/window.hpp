// Window accumulation of the semblance numerator/denominator and the final reduction.
//
// Restates COMPUTE_SEMBLANCE and REDUCE_SEMBLANCE_STACK
// (common/include/gpu/interface.h:26-55) for one lane = one (t0, candidate) pair.
//   W > 0   : the window size is a compile-time constant (fully unrolled, one basic
//             block, the numerator components A_j live in VGPRs);
//   W == 0  : any w <= 32, guarded by the (wave-uniform) runtime w.
//   HSS_EXACT keeps the reference order: u = (y1 - y0)*frac + y0; A_j += u; lin += u;
//             den += u*u -- no contraction, so the sums equal an IEEE FP32 evaluation
//             of the reference text bit for bit.
//   HSS_FAST  u = fma(y1 - y0, frac, y0); A_j += u; den = fma(u, u, den); the linear sum
//             is recovered at the end as sum_j A_j (same value up to rounding).
//   HSS_KAHAN two-level compensation: the values of up to kKahanChunk consecutive
//             traces are summed as HSS_FAST sums them (A_j += u, den = fma(u, u, den)),
//             then each chunk's sums are Kahan-added into running totals (flush()), and
//             the final sums over j are compensated too.  A chunk is a sum of a few
//             terms, so its rounding stays at a few ulps whatever the number of traces,
//             and the compensation costs a few operations per chunk, not per trace.
#pragma once

#include "device_common.hpp"

namespace hss {

// base + a 32-bit byte offset: with a wave-uniform base the load takes the base in scalar
// registers and the offset as it is, no 64-bit address arithmetic per lane.
__device__ __forceinline__ const char *at_bytes(const void *base, uint32_t offset) {
    return (const char *)base + offset;
}

// All ones for p = 1, 0 for p = 0.
__device__ __forceinline__ uint32_t p_mask(unsigned p) { return 0u - p; }

// 16-bit samples read per lane without LDS (compiled window sizes only, all odd).  The
// window's first sample e0 is sample rpar + k of the wave-uniform word row `roww` (the row's
// first sample rounded down to an even sample, i.e. a 4-byte word of the aligned sample
// array; rpar = 1 when it was odd), so the loads take a scalar base and a 32-bit lane
// offset.  Words16 holds the words of samples e0 .. e0+W: for even e0 the (W+1)/2 words from
// word e0/2 on, for odd e0 one more.  What a kernel that reads windows per lane waits for is
// the vector cache, which takes every lane's line of every load by itself (an OCT
// differential evolution ran at 1.1 lines per clock and CU with four loads per window), so
// the words come in as few loads as possible, none of them past the last word needed: `a`
// from the window's first word on, and `b`, which starts at the last word of `a` for even e0
// (p = 0) and right behind it for odd e0 (p = 1).
template <int W>
struct Words16 {
    static_assert(W & 1, "covers an even number of samples");
    static constexpr int NW = (W + 1) / 2 + 1;
    static constexpr int NA = NW <= 4 ? 2 : (NW - 1) / 4 * 4;
    static constexpr int NB = NW - NA;
    uint32_t a[NA], b[NB];
    unsigned p;

    __device__ __forceinline__ void load(const uint32_t *roww, unsigned rpar, unsigned k) {
        const unsigned e0 = rpar + k;
        p = e0 & 1u;
        const uint32_t at = (e0 >> 1) << 2;
        const uint32_t *qa = (const uint32_t *)at_bytes(roww, at);
        const uint32_t *qb = (const uint32_t *)at_bytes(roww, at + 4u * p) + (NA - 1);
#pragma unroll
        for (int i = 0; i < NA; ++i) a[i] = qa[i];
#pragma unroll
        for (int i = 0; i < NB; ++i) b[i] = qb[i];
    }

    // Word i of the window shifted down to start at sample e0 (samples e0 + 2i, e0 + 2i + 1).
    // v_alignbit shifts by one sample or none; past `a` the operands move by one word with
    // p, which one v_perm_b32 does in the same step.
    __device__ __forceinline__ uint32_t shifted(int i, uint32_t sel) const {
        if (i < NA - 1) return __builtin_amdgcn_alignbit(a[i + 1], a[i], 16u * p);
        if (i == NA - 1) return __builtin_amdgcn_alignbit(b[0], a[i], 16u * p);
        return __builtin_amdgcn_perm(b[i - NA + 1], b[i - NA], sel);
    }
    // shifted()'s selector: the second word whole (p = 0), or the halves around the boundary
    __device__ __forceinline__ uint32_t selector() const { return p ? 0x05040302u : 0x07060504u; }
};

// The window's samples widened to float (not scaled).  BF16: one v_perm_b32 per sample moves
// its two bytes into the high half of a zero word (selector byte 0x0c gives 0x00), from
// either word of the pair, so the shift and the widening are one instruction.
template <int STORAGE, int W>
__device__ __forceinline__ void read16(const uint32_t *roww, unsigned rpar, unsigned k,
                                       float (&y)[W + 1]) {
    Words16<W> d;
    d.load(roww, rpar, k);
    constexpr int NA = Words16<W>::NA;
    if constexpr (STORAGE == HSS_F16) {
        const uint32_t sel = d.selector();
#pragma unroll
        for (int i = 0; i < (W + 1) / 2; ++i) {
            const uint32_t e = d.shifted(i, sel);
            y[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(e & 0xffffu));
            y[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(e >> 16));
        }
    } else {
        // samples 2i and 2i + 1: bytes {1,0} and {3,2} of words i+1:i for even e0, {3,2} and
        // {5,4} for odd e0; past `a`, where the pair b[i-NA+1]:b[i-NA] is one word lower for
        // even e0, {5,4} and {7,6}
        const uint32_t odd = p_mask(d.p) & 0x02020000u;
        const uint32_t ae = 0x01000c0cu + odd, ao = 0x03020c0cu + odd;
        const uint32_t be = 0x05040c0cu - odd, bo = 0x07060c0cu - odd;
#pragma unroll
        for (int i = 0; i < (W + 1) / 2; ++i) {
            if (i < NA) {
                const uint32_t hi = i + 1 < NA ? d.a[i + 1] : d.b[0];
                y[2 * i] = __uint_as_float(__builtin_amdgcn_perm(hi, d.a[i], ae));
                y[2 * i + 1] = __uint_as_float(__builtin_amdgcn_perm(hi, d.a[i], ao));
            } else {
                const uint32_t hi = d.b[i - NA + 1], lo = d.b[i - NA];
                y[2 * i] = __uint_as_float(__builtin_amdgcn_perm(hi, lo, be));
                y[2 * i + 1] = __uint_as_float(__builtin_amdgcn_perm(hi, lo, bo));
            }
        }
    }
}

// FP16 samples e0 .. e0+W of one window as halves (shifted by one sample for odd e0, not
// converted): arithmetic on (float)h[j] then reads each half straight from its word
// (v_fma_mix_f32) instead of converting it first.
template <int W>
__device__ __forceinline__ void read16_halves(const uint32_t *roww, unsigned rpar, unsigned k,
                                              _Float16 (&h)[W + 1]) {
    Words16<W> d;
    d.load(roww, rpar, k);
    const uint32_t sel = d.selector();
#pragma unroll
    for (int i = 0; i < (W + 1) / 2; ++i) {
        const uint32_t e = d.shifted(i, sel);
        h[2 * i] = __builtin_bit_cast(_Float16, (uint16_t)(e & 0xffffu));
        h[2 * i + 1] = __builtin_bit_cast(_Float16, (uint16_t)(e >> 16));
    }
}

// Kahan step: s + c' = s + c + x with the low part of the sum kept in c (c holds the
// negated error, as in Kahan's original form).
__device__ __forceinline__ void kahan_add(float &s, float &c, float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// Traces per compensation chunk of HSS_KAHAN (a power of two that divides the 64 traces of
// a geometry chunk).  16 measured 4% faster than 8 on the C5 line (FP16 grid); a chunk's
// plain sum then rounds at most about 8 ulps, against the ~36 of a plain 72-trace sum.
constexpr int kKahanChunk = 16;
static_assert((kKahanChunk & (kKahanChunk - 1)) == 0 && kKahanChunk <= 64,
              "the chunk must be a power of two dividing 64");

// Two neighbouring window values as HSS_FAST and HSS_KAHAN sum them: d = y1 - y0,
// u = fma(d, f, y0), A += u, den = fma(u, u, den), each the same operation the plain
// expressions give, in registers chosen by hand.
//
// What bounds the window sums is VALU issue, and on gfx950 that depends on the registers:
// an FP32 add, subtract, multiply or FMA whose sources are vector registers issues in two
// cycles per wave, but an FMA whose three sources all lie in even or all in odd registers
// takes four, as does any operation with a scalar-register source (measured with
// independent chains at 4 waves per SIMD: 2.5 against 4.9 cycles of a nominal 2.4 GHz; the
// sources of an FMA modulo 2 are all that matters).  den = fma(u, u, den) is thus fast only
// when u and den differ in parity, and the compiler, which does not know, gets a third of
// a window's FMAs wrong.  Here the differences go to even registers, f sits in an odd one
// (so fma(d, f, y0) is fast wherever y0 is), the values u go to odd ones and den sits in an
// even one: eight fast operations.  `slot` is 0 or 1 (a constant after inlining): the
// candidates of a lane that are summed in one loop keep den and f in registers of their own.
__device__ __forceinline__ void window_pair(float &A0, float &A1, float &den, float y0, float y1,
                                            float y2, float f, int slot) {
#define HSS_WINDOW_PAIR(DEN, F)                            \
    __asm__("v_sub_f32 v2, %4, %3\n\t"                     \
            "v_sub_f32 v4, %5, %4\n\t"                     \
            "v_fma_f32 v3, v2, %6, %3\n\t"                 \
            "v_fma_f32 v5, v4, %6, %4\n\t"                 \
            "v_add_f32 %0, %0, v3\n\t"                     \
            "v_fmac_f32 %2, v3, v3\n\t"                    \
            "v_add_f32 %1, %1, v5\n\t"                     \
            "v_fmac_f32 %2, v5, v5"                        \
            : "+v"(A0), "+v"(A1), "+{" DEN "}"(den)        \
            : "v"(y0), "v"(y1), "v"(y2), "{" F "}"(f)      \
            : "v2", "v3", "v4", "v5")
    if (slot == 0)
        HSS_WINDOW_PAIR("v6", "v7");
    else
        HSS_WINDOW_PAIR("v8", "v9");
#undef HSS_WINDOW_PAIR
}

// The same for one value (the last of an odd window).
__device__ __forceinline__ void window_single(float &A0, float &den, float y0, float y1, float f,
                                              int slot) {
#define HSS_WINDOW_SINGLE(DEN, F)                     \
    __asm__("v_sub_f32 v2, %3, %2\n\t"                \
            "v_fma_f32 v3, v2, %4, %2\n\t"            \
            "v_add_f32 %0, %0, v3\n\t"                \
            "v_fmac_f32 %1, v3, v3"                   \
            : "+v"(A0), "+{" DEN "}"(den)             \
            : "v"(y0), "v"(y1), "{" F "}"(f)          \
            : "v2", "v3")
    if (slot == 0)
        HSS_WINDOW_SINGLE("v6", "v7");
    else
        HSS_WINDOW_SINGLE("v8", "v9");
#undef HSS_WINDOW_SINGLE
}

// How a window's samples are summed; the same bits.  Paired: all of them in registers, the sums
// in window_pair's fixed ones.  Plain: all in registers, the rest left to the compiler.  InTurn:
// one sample after the other, for kernels whose sums take the registers.  (HSS_EXACT is never
// Paired.)
enum class Summing { Paired, Plain, InTurn };

template <int W, int VARIANT>
struct Window {
    static constexpr int N = W > 0 ? W : kMaxWindow;
    static constexpr bool KAHAN = VARIANT == HSS_KAHAN;
    static constexpr int NK = KAHAN ? N : 1;
    float A[N];            // window sums (HSS_KAHAN: of the current chunk)
    float T[NK], Tc[NK];   // HSS_KAHAN: running totals of A_j and their compensation
    float lin, den, tden, denc;
    unsigned used;

    __device__ __forceinline__ void reset() {
#pragma unroll
        for (int j = 0; j < N; ++j) A[j] = 0.0f;
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            T[j] = 0.0f;
            Tc[j] = 0.0f;
        }
        lin = 0.0f;
        den = 0.0f;
        tden = 0.0f;
        denc = 0.0f;
        used = 0;
    }

    // HSS_KAHAN: adds the chunk sums to the compensated totals and starts a new chunk
    // (a no-op for the other variants).  Callers flush every kKahanChunk traces, at
    // wave-uniform points of the trace loop.
    __device__ __forceinline__ void flush(int w) {
        if constexpr (KAHAN) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (W == 0 && j >= w) continue;
                kahan_add(T[j], Tc[j], A[j]);
                A[j] = 0.0f;
            }
            kahan_add(tden, denc, den);
            den = 0.0f;
        }
    }

    // One interpolated sample u = y + frac*d at window position j, d = y_next - y (the
    // same FP32 difference the reference forms, so HSS_EXACT keeps its bits).
    __device__ __forceinline__ void step_d(int j, float y, float d, float f) {
        if constexpr (VARIANT == HSS_EXACT) {
            float u = d * f + y;
            A[j] += u;
            lin += u;
            den += u * u;
        } else {
            // HSS_FAST, and HSS_KAHAN inside a chunk
            float u = __builtin_fmaf(d, f, y);
            A[j] += u;
            den = __builtin_fmaf(u, u, den);
        }
    }

    __device__ __forceinline__ void step(int j, float y0, float y1, float f) {
        step_d(j, y0, y1 - y0, f);
    }

    // The window whose samples are y[0..W] (compiled window sizes).
    template <Summing HOW = Summing::Paired, class Samples>
    __device__ __forceinline__ void sum(const Samples &y, float f, int slot) {
        static_assert(W > 0, "a compiled window size");
        if constexpr (VARIANT == HSS_EXACT || HOW != Summing::Paired) {
#pragma unroll
            for (int j = 0; j < W; ++j) step(j, y[j], y[j + 1], f);
        } else {
#pragma unroll
            for (int j = 0; j + 1 < W; j += 2)
                window_pair(A[j], A[j + 1], den, y[j], y[j + 1], y[j + 2], f, slot);
            if constexpr (W & 1) window_single(A[W - 1], den, y[W - 1], y[W], f, slot);
        }
    }

    // The window that starts at p[0], without counting its trace in `used`.
    template <Summing HOW, class Samples>
    __device__ __forceinline__ void sum_from(Samples p, float f, int w, int slot) {
        if constexpr (W > 0 && HOW != Summing::InTurn) {
            float y[W + 1];
#pragma unroll
            for (int j = 0; j <= W; ++j) y[j] = p[j];
            sum<HOW>(y, f, slot);
        } else {
            float y1 = p[0];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (W == 0 && j >= w) continue;
                const float y0 = y1;
                y1 = p[j + 1];
                step(j, y0, y1, f);
            }
        }
    }

    // Adds the w interpolated values starting at sample `base` of the flat sample array.
    template <class Reader>
    __device__ __forceinline__ void add(const Reader &rd, size_t base, float f, float scale,
                                        bool scaled, int w) {
        float y1 = rd(base);
        if (scaled) y1 = y1 * scale;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if (W == 0 && j >= w) continue;
            float y0 = y1;
            y1 = rd(base + j + 1);
            if (scaled) y1 = y1 * scale;
            step(j, y0, y1, f);
        }
        used++;
    }

    // FP32 samples of one trace: row[k .. k+w] with `row` wave-uniform (the trace's first
    // sample minus tau) and k the lane's sample index, so the loads take a scalar base and
    // a 32-bit lane offset.
    template <Summing HOW = Summing::Paired>
    __device__ __forceinline__ void add_row(const float *row, unsigned k, float f, int w,
                                            int slot = 0) {
        sum_from<HOW>(row + k, f, w, slot);
        used++;
    }

    // A window's values value(0) .. value(W-1) without their trace's scale: A_j += sc*u_j and
    // dn = sum_j u_j^2.  Left to the compiler: the values come from conversions or mixed FMAs
    // of four cycles each, and sums in fixed registers held their scheduling back (FP16, CMP
    // stretch-free of 1000 midpoints, w = 15, 8.49 ms fixed, 7.28 here; ZO-CRS DE, 32 midpoints,
    // 49.4 and 42.9 ms).
    template <class Value>
    __device__ __forceinline__ void sum_scaled(const Value &value, float &dn, float sc) {
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const float u = value(j);
            A[j] = __builtin_fmaf(sc, u, A[j]);
            dn = __builtin_fmaf(u, u, dn);
        }
    }

    // 16-bit samples of one window read per lane (read16), then summed.  FACTORED: the
    // non-exact variants factor the trace's scale `sc` out of the window (a line without
    // scales passes sc = 1).  !FACTORED, for a line stored without scales (BF16: FP32's
    // exponent range needs none): the FP32 steps, whose sums need an add per value where
    // the factored scale needs an FMA.  The choice is a template parameter so that a
    // kernel holds one form in its trace loop (both would add registers).
    template <int STORAGE, bool FACTORED = true>
    __device__ __forceinline__ void add16(const uint32_t *roww, unsigned rpar, unsigned k,
                                          float f, float sc, int slot = 0) {
        static_assert(W > 0, "add16 needs a compiled window size");
        // windows of other sizes than 5 to 15 samples keep the form of the runtime-w kernel
        // they came from, whose samples are scaled one by one
        constexpr bool FACTOR = FACTORED && W >= 5 && W <= 15;
        if constexpr (VARIANT != HSS_EXACT && STORAGE == HSS_F16 && FACTOR) {
            // as below, with y1 - y0 formed as fma(y1, one, -y0) = RN(y1 - y0): the same
            // bits, but an FMA reads both halves straight from the words (v_fma_mix_f32),
            // where a subtraction needs both converted first.  `one` is 1.0 hidden from the
            // optimizer (an empty asm statement), which would otherwise turn the FMA back
            // into a subtraction.
            _Float16 h[W + 1];
            read16_halves<W>(roww, rpar, k, h);
            float one = 1.0f;
            __asm__("" : "+s"(one));
            float dn = 0.0f;
            auto value = [&](int j) {
                const float d = __builtin_fmaf((float)h[j + 1], one, -(float)h[j]);
                return __builtin_fmaf(d, f, (float)h[j]);
            };
            sum_scaled(value, dn, sc);
            den = __builtin_fmaf(sc * sc, dn, den);
            used++;
            return;
        }
        float y[W + 1];
        read16<STORAGE, W>(roww, rpar, k, y);
        if constexpr (VARIANT != HSS_EXACT) {
            if constexpr (!FACTOR) {
                if constexpr (FACTORED) {
#pragma unroll
                    for (int j = 0; j <= W; ++j) y[j] = y[j] * sc;
                }
                sum(y, f, slot);
                used++;
                return;
            }
            // the trace's scale factored out of the window: u = sc * (y0 + frac*(y1 - y0))
            // on the stored values, A_j += sc*u and den += sc^2 * sum_j u^2
            float dn = 0.0f;
            sum_scaled([&](int j) { return __builtin_fmaf(y[j + 1] - y[j], f, y[j]); }, dn, sc);
            den = __builtin_fmaf(sc * sc, dn, den);
        } else {
            if constexpr (FACTORED) {
#pragma unroll
                for (int j = 0; j <= W; ++j) y[j] = y[j] * sc;
            }
#pragma unroll
            for (int j = 0; j < W; ++j) step(j, y[j], y[j + 1], f);
        }
        used++;
    }

    // A window in LDS stored as pairs, at[i] = {sample i, sample i + 1}, without counting its
    // trace in `used`: samples j and j + 1 are one aligned 8-byte read from at[j].  (8-byte
    // reads move 217 bytes per clock and CU where the 4-byte reads of a plain row, whose
    // windows start anywhere, move 120; measured.  Volatile: the compiler would merge two of
    // them into one ds_read2_b64, which is back at 122.)
    __device__ __forceinline__ void sum_pairs(LdsPair *at, float f, int w, int slot) {
        if constexpr (W > 0) {
            float y[W + 1];
#pragma unroll
            for (int j = 0; j < W; j += 2) {
                const LdsPairValue p = at[j];
                y[j] = p.x;
                y[j + 1] = p.y;
            }
            sum(y, f, slot);
        } else {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (j >= w) continue;
                const LdsPairValue p = at[j];
                step(j, p.x, p.y, f);
            }
        }
    }

    // Same as add() for a window already decoded (and scaled) into LDS: row[0..w].
    template <Summing HOW>
    __device__ __forceinline__ void add_lds(const LdsFloat *row, float f, int w, int slot) {
        sum_from<HOW>(row, f, w, slot);
        used++;
    }

    // REDUCE_SEMBLANCE_STACK: S = sum_j A_j^2 / (used * den), stack = lin / (used * w);
    // both stay 0 when no trace was used.  (HSS_KAHAN: the last chunk is flushed first.)
    __device__ __forceinline__ void reduce(int w, float *S, float *stack) {
        flush(w);
        float sem = 0.0f, stk = 0.0f;
        if (used > 0) {
            float num = 0.0f, numc = 0.0f;
            float l = lin, lc = 0.0f;
            if constexpr (VARIANT != HSS_EXACT) l = 0.0f;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (W == 0 && j >= w) continue;
                if constexpr (VARIANT == HSS_EXACT) {
                    num += A[j] * A[j];
                } else if constexpr (VARIANT == HSS_FAST) {
                    num = __builtin_fmaf(A[j], A[j], num);
                    l += A[j];
                } else {
                    // the total carries its compensation: use the corrected value; the
                    // square's rounding goes into the compensation through the FMA
                    const float a = T[j] - Tc[j];
                    const float y = __builtin_fmaf(a, a, -numc);
                    const float t = num + y;
                    numc = (t - num) - y;
                    num = t;
                    kahan_add(l, lc, a);
                }
            }
            float d = den;
            if constexpr (KAHAN) {
                num = num - numc;
                l = l - lc;
                d = tden - denc;
            }
            sem = num / ((float)used * d);
            stk = l / (float)(used * (unsigned)w);
        }
        *S = sem;
        *stack = stk;
    }
};

}  // namespace hss
