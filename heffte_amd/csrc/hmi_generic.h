// Runtime-length FFT pass (fft_generic), included by one source per precision.
//
// One block transforms a tile of lines in place in one LDS buffer (radix plan and layout: mixed_plan,
// hmi_pass.h).  The first stage takes its inputs from global memory and the last stage stores its
// outputs there, so the tile crosses LDS only between stages.  Each stage walks its butterflies over
// the block's threads with the lines of the tile fastest (lanes on consecutive lines: consecutive
// LDS elements, one twiddle for all of them, the line of a thread fixed for the whole loop), except
// the load and store of a side on which the FFT axis is the contiguous one, where lanes walk the
// axis.  Divisions are multiplications by the plan's constants (but for two in the direct stages, one a work
// unit of four outputs).
//
// Bound: HBM bytes on complex<double> (384 x 400 x 320, per pass: 305, 315 and 325 us, 4.8-5.2 TB/s;
// a device copy of such arrays runs at 4.7-5.0 TB/s), issue and latency on complex<float> (40 boxes of
// 48 x 60 x 72: 26 us per 60- or 72-point pass, 5.0 TB/s; 256 x 240 x 250: 48 us per 240-point pass).
// The pass it replaces (a ping-pong of two LDS buffers, run-time divisions per element, every stage
// through LDS) took 912-1024, 119-127 and 241 us.  Measured and not taken: two neighbouring
// complex<float> lines per lane in 16-byte values (half the index work, but as many registers as
// complex<double>: 60 points 4.35 against 4.58 TB/s, 180 points 4.48 against 4.83, 400 points 4.40
// against 4.23).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "hmi_device.h"
#include "hmi_kernels.h"

namespace hmi {

__device__ __forceinline__ unsigned fdiv(unsigned x, const fast_div &d) { return __umulhi(x << 1, d.mul) >> d.shift; }

// Offset of line L (column-fastest numbering of column x b1 x batch), and its index along one
// dimension of that numbering (0 column, 1 b1, 2 batch).
__device__ __forceinline__ long long mixed_line_offset(unsigned L, const pass_args &a, const mixed_plan &g, bool out) {
    const unsigned q = fdiv(L, g.by_ncol);
    const unsigned c = L - q * (unsigned)a.ncol;
    const unsigned b2 = fdiv(q, g.by_nb1);
    const unsigned b1 = q - b2 * (unsigned)a.nb1;
    return out ? (long long)c * a.out_sc + (long long)b1 * a.out_sb1 + (long long)b2 * a.out_sb2
               : (long long)c * a.in_sc + (long long)b1 * a.in_sb1 + (long long)b2 * a.in_sb2;
}
__device__ __forceinline__ unsigned mixed_line_index(unsigned L, const pass_args &a, const mixed_plan &g, int dim) {
    const unsigned q = fdiv(L, g.by_ncol);
    if (dim == 0) return L - q * (unsigned)a.ncol;
    const unsigned b2 = fdiv(q, g.by_nb1);
    return dim == 1 ? q - b2 * (unsigned)a.nb1 : b2;
}

// A line of the tile on one side: number, whether it exists, offset.
struct line_at {
    unsigned line;
    bool valid;
    long long base;
    __device__ __forceinline__ void locate(unsigned L, const pass_args &a, const mixed_plan &g, bool out) {
        line = L;
        valid = L < (unsigned)a.nlines;
        base = valid ? mixed_line_offset(L, a, g, out) : 0;
    }
};

// twiddles of the plan's table (after the middle stages' entries)
template <typename C> __device__ __forceinline__ const C *mixed_twiddles(const pass_args &a) {
    return reinterpret_cast<const C *>(static_cast<const char *>(a.tw) + kMixedHead);
}

// Forms of the pass: every mode and overload; plain complex lines (no product, real side, partial
// store or split twiddle); the same where both arrays lie within 4 GiB (each access is a uniform
// base plus one 32-bit offset per thread, half the address registers); chirp convolutions and plans with direct
// stages (any mode).
enum : int { kFormAny = 0, kFormPlain = 1, kFormPlain32 = 2, kFormChirp = 3, kFormDirect = 4 };

// Elements j0, j0 + step, ... (RX of them; j0 < step) of a line in the pass's input form.
template <int RX, int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_load(C (&x)[RX], const pass_args &a, const mixed_plan &g, const line_at &ln, int j0,
                                           int step) {
    constexpr bool NTL = (NTM & 2) != 0;
    const R sg = a.conj ? R(-1) : R(1);
    const int n = g.len;
    if (!ln.valid) {
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = cmk<C>(R(0), R(0));
    } else if ((FORM == kFormAny || FORM == kFormDirect) && (a.mode == kModeDCT2 || a.mode == kModeDST2)) {
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            const int jj = (j < (n + 1) / 2) ? 2 * j : 2 * (n - 1 - j) + 1;
            const R v = ldg<NTL>(&src[(long long)jj * a.in_sa]);
            x[p] = cmk<C>((a.mode == kModeDST2 && (jj & 1)) ? -v : v, R(0));
        }
    } else if ((FORM == kFormAny || FORM == kFormDirect) && (a.mode == kModeDCT3 || a.mode == kModeDST3)) {
        const bool sine = (a.mode == kModeDST3);
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
        const C *__restrict__ post = mixed_twiddles<C>(a) + g.postoff;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            const R xk = ldg<NTL>(&src[(long long)(sine ? n - 1 - j : j) * a.in_sa]);
            const R xm = j > 0 ? ldg<NTL>(&src[(long long)(sine ? j - 1 : n - j) * a.in_sa]) : R(0);
            const C w = post[j];
            x[p] = cmk<C>(w.x * xk - w.y * xm, w.x * xm + w.y * xk);  // conj of conj(w) (xk - i xm)
        }
    } else if ((FORM == kFormAny || FORM == kFormDirect) && (a.mode == kModeDCT1 || a.mode == kModeDCT1B)) {
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            x[p] = cmk<C>(ldg<NTL>(&src[(long long)(j <= n / 2 ? j : n - j) * a.in_sa]), R(0));
        }
    } else if ((FORM == kFormAny || FORM == kFormDirect) && a.in_real) {
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = cmk<C>(ldg<NTL>(&src[(long long)(j0 + p * step) * a.in_sa]), R(0));
    } else if ((FORM == kFormAny || FORM == kFormDirect) && a.herm_load) {
        const C *__restrict__ src = static_cast<const C *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            const bool mirror = j > n / 2;
            const C v = ldg<NTL>(&src[(long long)(mirror ? n - j : j) * a.in_sa]);
            x[p] = cmk<C>(v.x, (mirror ? -sg : sg) * v.y);
        }
    } else if ((FORM == kFormAny || FORM == kFormDirect) && a.mul) {
        const C *src = static_cast<const C *>(a.in) + ln.base;
        const C *mul = static_cast<const C *>(a.mul) + ln.base;
        C y[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = ldg<NTL>(&src[(long long)(j0 + p * step) * a.in_sa]);
        if (a.mul == a.in) {
#pragma unroll
            for (int p = 0; p < RX; p++) y[p] = x[p];
        } else {
#pragma unroll
            for (int p = 0; p < RX; p++) y[p] = ldg<NTL>(&mul[(long long)(j0 + p * step) * a.in_sa]);
        }
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const C v = cmul(x[p], y[p]);
            x[p] = cmk<C>(v.x, sg * v.y);
        }
    } else {
        const long long at = (ln.base + (long long)j0 * a.in_sa) * (long long)sizeof(C);
        const long long st = (long long)step * a.in_sa * (long long)sizeof(C);
        const char *__restrict__ in = static_cast<const char *>(a.in);
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const C v = ldg<NTL>(reinterpret_cast<const C *>(FORM == kFormPlain32 ? in + p * st + (unsigned)at
                                                                                  : in + p * st + at));
            x[p] = cmk<C>(v.x, sg * v.y);
        }
    }
}

// Stores frequencies k0, k0 + step, ... (RX of them) of a line.
template <int RX, int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_store(const C (&x)[RX], const pass_args &a, const mixed_plan &g, const line_at &ln,
                                            int k0, int step) {
    constexpr bool NTS = (NTM & 1) != 0;
    const R sg = a.conj ? R(-1) : R(1);
    const R sc = (R)a.scale;
    const int n = g.len;
    if ((FORM == kFormAny || FORM == kFormDirect) && (a.mode == kModeDCT2 || a.mode == kModeDST2)) {
        R *__restrict__ dst = static_cast<R *>(a.out) + ln.base;
        const C *__restrict__ post = mixed_twiddles<C>(a) + g.postoff;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int k = k0 + p * step;
            const C w = post[k];
            stg<NTS>(&dst[(long long)(a.mode == kModeDST2 ? n - 1 - k : k) * a.out_sa],
                     R(2) * (w.x * x[p].x - w.y * x[p].y) * sc);
        }
    } else if ((FORM == kFormAny || FORM == kFormDirect) && (a.mode == kModeDCT3 || a.mode == kModeDST3)) {
        R *__restrict__ dst = static_cast<R *>(a.out) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int k = k0 + p * step;
            const int j = (k < (n + 1) / 2) ? 2 * k : 2 * (n - 1 - k) + 1;
            const R y = R(2) * x[p].x;
            stg<NTS>(&dst[(long long)j * a.out_sa], ((a.mode == kModeDST3 && (j & 1)) ? -y : y) * sc);
        }
    } else if ((FORM == kFormAny || FORM == kFormDirect) && a.out_real) {
        R *__restrict__ dst = static_cast<R *>(a.out) + ln.base;
        const R f = (a.mode == kModeDCT1B) ? R(2) * sc : sc;
#pragma unroll
        for (int p = 0; p < RX; p++)
            if (k0 + p * step < a.store_len) stg<NTS>(&dst[(long long)(k0 + p * step) * a.out_sa], x[p].x * f);
    } else if ((FORM == kFormAny || FORM == kFormDirect) && (a.store_len < n || a.tw4)) {
        C *__restrict__ dst = static_cast<C *>(a.out) + ln.base;
        const C *__restrict__ w4 = static_cast<const C *>(a.tw4);
        const unsigned jl = w4 ? mixed_line_index(ln.line, a, g, a.tw4_dim) : 0;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int k = k0 + p * step;
            if (k >= a.store_len) continue;
            const C y = w4 ? cmul(x[p], w4[jl * (unsigned)k]) : x[p];
            stg<NTS>(&dst[(long long)k * a.out_sa], cmk<C>(y.x * sc, sg * y.y * sc));
        }
    } else {
        const long long at = (ln.base + (long long)k0 * a.out_sa) * (long long)sizeof(C);
        const long long st = (long long)step * a.out_sa * (long long)sizeof(C);
        char *__restrict__ out = static_cast<char *>(a.out);
        const R sy = sg * sc;
#pragma unroll
        for (int p = 0; p < RX; p++)
            stg<NTS>(reinterpret_cast<C *>(FORM == kFormPlain32 ? out + p * st + (unsigned)at : out + p * st + at),
                     cmk<C>(x[p].x * sc, x[p].y * sy));
    }
}

// Element j of a line in the pass's input form (the chirp passes; any mode).
template <int NTM, typename R, typename C>
__device__ __forceinline__ C mixed_element(const pass_args &a, const mixed_plan &g, const line_at &ln, int j) {
    C x[1];
    mixed_load<1, kFormAny, NTM, R>(x, a, g, ln, j, 0);
    return x[0];
}

// Stage 0: global memory -> LDS.
template <int RX, int SET, int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_first(const pass_args &a, const mixed_plan &g, unsigned tile, C *lds) {
    const int T = 1 << g.log2t, m = g.m0, nth = blockDim.x;
    const int stride = m * g.pitch + g.pad;
    const C *__restrict__ tw = mixed_twiddles<C>(a);
    const bool across = a.load_colfast != 0;
    line_at ln;
    if (across) ln.locate(tile * T + (threadIdx.x & (T - 1)), a, g, false);
    for (int idx = threadIdx.x; idx < m << g.log2t; idx += nth) {
        int l, j;
        if (across) {
            l = idx & (T - 1);
            j = idx >> g.log2t;
        } else {
            l = fdiv(idx, g.by_m0);
            j = idx - l * m;
            ln.locate(tile * T + l, a, g, false);
        }
        C x[RX];
        if constexpr (FORM == kFormChirp) {
            // x_j c_j for j < len, zeros behind it
            const C *__restrict__ chirp = tw + g.chirpoff;
#pragma unroll
            for (int p = 0; p < RX; p++) {
                x[p] = cmk<C>(R(0), R(0));
                if (p * m < g.len) {
                    const int at = j + p * m;
                    const int jc = at < g.len ? at : g.len - 1;
                    const C v = cmul(mixed_element<NTM, R, C>(a, g, ln, jc), chirp[jc]);
                    if (at < g.len) x[p] = v;
                }
            }
        } else {
            mixed_load<RX, FORM, NTM, R>(x, a, g, ln, j, m);
        }
        butterfly<RX, SET == kSetOdd>(x);
        if (m > 1) {
            const C *w = tw + j * (RX - 1);
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        }
        C *dp = lds + j * g.pitch + l;
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * stride] = x[q];
    }
}

// A stage between two others, in place in LDS; BACK: its transpose (twiddles before the butterfly).
template <int RX, int SET, bool BACK, typename R, typename C>
__device__ __forceinline__ void mixed_middle(const pass_args &a, const mixed_plan &g, const mixed_stage &st, C *lds) {
    const int T = 1 << g.log2t, m = st.m, nth = blockDim.x;
    const int stride = m * g.pitch;
    const unsigned nb = (unsigned)g.n / RX;
    const C *__restrict__ tw = mixed_twiddles<C>(a) + st.twoff;
    for (unsigned idx = threadIdx.x; idx < nb << g.log2t; idx += nth) {
        const int l = idx & (T - 1);
        const unsigned b = idx >> g.log2t;
        const unsigned c = fdiv(b, st.by_m);
        const int j = (int)(b - c * (unsigned)m);
        C *dp = lds + ((int)c * RX * m + j) * g.pitch + (int)fdiv(c, st.by_k0) * g.pad + l;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = dp[p * stride];
        const C *w = tw + j * (RX - 1);
        if (BACK) {
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        }
        butterfly<RX, SET == kSetOdd>(x);
        if (!BACK) {
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        }
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * stride] = x[q];
    }
}

// Chirp passes: the last stage, the product with the transformed chirp and the first transposed
// stage, which works on the same elements.
template <int RX, int SET, typename R, typename C>
__device__ __forceinline__ void mixed_center(const pass_args &a, const mixed_plan &g, const mixed_stage &st, C *lds) {
    const int T = 1 << g.log2t, nth = blockDim.x;
    const unsigned nb = (unsigned)g.n / RX;
    const C *__restrict__ hat = mixed_twiddles<C>(a) + g.chirpoff + g.len;
    for (unsigned idx = threadIdx.x; idx < nb << g.log2t; idx += nth) {
        const int l = idx & (T - 1);
        const unsigned c = idx >> g.log2t;
        C *dp = lds + (int)c * RX * g.pitch + (int)fdiv(c, st.by_k0) * g.pad + l;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = dp[p * g.pitch];
        butterfly<RX, SET == kSetOdd>(x);
#pragma unroll
        for (int q = 0; q < RX; q++) {
            const C v = cmul(x[q], hat[c * RX + q]);
            x[q] = cmk<C>(v.x, -v.y);
        }
        butterfly<RX, SET == kSetOdd>(x);
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * g.pitch] = x[q];
    }
}

// Chirp passes: the transpose of stage 0, LDS -> global memory.
template <int RX, int SET, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_chirp_last(const pass_args &a, const mixed_plan &g, unsigned tile, const C *lds) {
    const int T = 1 << g.log2t, m = g.m0, nth = blockDim.x;
    const int stride = m * g.pitch + g.pad;
    const C *__restrict__ tw = mixed_twiddles<C>(a);
    const C *__restrict__ chirp = tw + g.chirpoff;
    const bool across = a.store_colfast != 0;
    line_at ln;
    if (across) ln.locate(tile * T + (threadIdx.x & (T - 1)), a, g, true);
    for (int idx = threadIdx.x; idx < m << g.log2t; idx += nth) {
        int l, j;
        if (across) {
            l = idx & (T - 1);
            j = idx >> g.log2t;
        } else {
            l = fdiv(idx, g.by_m0);
            j = idx - l * m;
            ln.locate(tile * T + l, a, g, true);
        }
        if (!ln.valid) continue;
        const C *sp = lds + j * g.pitch + l;
        const C *w = tw + j * (RX - 1);
        C x[RX];
#pragma unroll
        for (int q = 0; q < RX; q++) x[q] = sp[q * stride];
#pragma unroll
        for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        butterfly<RX, SET == kSetOdd>(x);
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int k = j + p * m;
            if (p * m < g.len && k < g.len) {
                const C y[1] = {cmul(cmk<C>(x[p].x, -x[p].y), chirp[k])};
                mixed_store<1, kFormAny, NTM, R>(y, a, g, ln, k, 0);
            }
        }
    }
}

// The last stage: LDS -> global memory.
template <int RX, int SET, int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_last(const pass_args &a, const mixed_plan &g, unsigned tile, const C *lds) {
    const int T = 1 << g.log2t, nth = blockDim.x;
    const unsigned nb = (unsigned)g.n / RX;
    const bool across = a.store_colfast != 0;
    line_at ln;
    if (across) ln.locate(tile * T + (threadIdx.x & (T - 1)), a, g, true);
    for (unsigned idx = threadIdx.x; idx < nb << g.log2t; idx += nth) {
        unsigned l, u;
        if (across) {
            l = idx & (T - 1);
            u = idx >> g.log2t;
        } else {
            l = fdiv(idx, g.by_last);
            u = idx - l * nb;
            ln.locate(tile * T + l, a, g, true);
        }
        if (!ln.valid) continue;
        // u = k_0 + r_0 k_1 + ...: the butterfly's block number and k_0
        unsigned c = 0, k0 = 0, t = u;
#pragma unroll
        for (int s = 0; s + 2 < kMixedStages; s++) {
            if (s + 2 >= g.nst) break;
            const unsigned q = fdiv(t, g.by_r[s]);
            const unsigned d = t - q * (unsigned)g.radix[s];
            if (s == 0) k0 = d;
            c = (c + d) * (unsigned)g.radix[s + 1];
            t = q;
        }
        if (g.nst == 2) k0 = t;
        c += t;
        const C *sp = lds + (int)c * RX * g.pitch + (int)k0 * g.pad + (int)l;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = sp[p * g.pitch];
        butterfly<RX, SET == kSetOdd>(x);
        mixed_store<RX, FORM, NTM, R>(x, a, g, ln, (int)u, (int)nb);
    }
}

// Elementwise load into LDS (copy passes) and store from LDS (copy passes, one-stage lengths).
template <int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_fill(const pass_args &a, const mixed_plan &g, unsigned tile, C *lds) {
    const int T = 1 << g.log2t;
    for (int idx = threadIdx.x; idx < g.n << g.log2t; idx += blockDim.x) {
        int l, j;
        if (a.load_colfast) { l = idx & (T - 1); j = idx >> g.log2t; } else { l = fdiv(idx, g.by_n); j = idx - l * g.n; }
        line_at ln;
        ln.locate(tile * T + l, a, g, false);
        C x[1];
        mixed_load<1, FORM, NTM, R>(x, a, g, ln, j, 0);
        lds[j * g.pitch + l] = x[0];
    }
}
template <int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_drain(const pass_args &a, const mixed_plan &g, unsigned tile, const C *lds) {
    const int T = 1 << g.log2t;
    for (int idx = threadIdx.x; idx < g.n << g.log2t; idx += blockDim.x) {
        int l, k;
        if (a.store_colfast) { l = idx & (T - 1); k = idx >> g.log2t; } else { l = fdiv(idx, g.by_n); k = idx - l * g.n; }
        line_at ln;
        ln.locate(tile * T + l, a, g, true);
        if (!ln.valid) continue;
        const C x[1] = {lds[k * g.pitch + l]};
        mixed_store<1, FORM, NTM, R>(x, a, g, ln, k, 0);
    }
}

// One-stage lengths whose few lines load and store elementwise (mixed_plan::spread): their butterflies.
template <int RX, int SET, typename C> __device__ __forceinline__ void mixed_only(const mixed_plan &g, C *lds) {
    for (int l = threadIdx.x; l < 1 << g.log2t; l += blockDim.x) {
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = lds[p * g.pitch + l];
        butterfly<RX, SET == kSetOdd>(x);
#pragma unroll
        for (int p = 0; p < RX; p++) lds[p * g.pitch + l] = x[p];
    }
}

// Sums of one direct p-point butterfly at sp (elements pitch apart): outputs q and p - q for q = q0 and
// q0 + 1.  root = w_p^t, t < p.
template <typename R, typename C>
__device__ __forceinline__ void mixed_direct_sums(const C *sp, int pitch, int p, int q0, const C *__restrict__ root, C (&lo)[2],
                                                  C (&hi)[2]) {
    const C x0 = sp[0];
    C re[2] = {x0, x0}, im[2] = {cmk<C>(R(0), R(0)), cmk<C>(R(0), R(0))};
    int t[2] = {0, 0};
    const C *a = sp, *b = sp + p * pitch;
#pragma unroll 2
    for (int k = 1; k <= (p - 1) / 2; k++) {
        a += pitch;
        b -= pitch;
        const C xa = *a, xb = *b;
        const C s = cadd(xa, xb), d = csub(xa, xb);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            t[i] += q0 + i;
            t[i] -= t[i] >= p ? p : 0;
            const C w = root[t[i]];  // (cos, -sin) of 2 pi k q / p
            re[i].x += s.x * w.x;
            re[i].y += s.y * w.x;
            im[i].x += d.x * w.y;
            im[i].y += d.y * w.y;
        }
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        lo[i] = cmk<C>(re[i].x - im[i].y, re[i].y + im[i].x);
        hi[i] = cmk<C>(re[i].x + im[i].y, re[i].y - im[i].x);
    }
}

// A direct stage before the last one: from one LDS buffer to the other.
template <typename R, typename C>
__device__ __forceinline__ void mixed_direct(const pass_args &a, const mixed_plan &g, const mixed_stage &st, const C *from, C *to) {
    const int T = 1 << g.log2t, p = st.radix, m = st.m, groups = (p + 3) / 4;
    const unsigned nb = (unsigned)(g.n / p);
    const C *__restrict__ tw = mixed_twiddles<C>(a) + st.twoff, *__restrict__ root = mixed_twiddles<C>(a) + st.root;
    for (unsigned idx = threadIdx.x; idx < (nb * groups) << g.log2t; idx += blockDim.x) {
        const int l = idx & (T - 1);
        const unsigned v = idx >> g.log2t;
        const unsigned grp = v / nb, b = v - grp * nb;
        const unsigned c = fdiv(b, st.by_m);
        const int j = (int)(b - c * (unsigned)m), at = ((int)c * p * m + j) * g.pitch + l;
        C lo[2], hi[2];
        mixed_direct_sums<R>(from + at, m * g.pitch, p, 2 * (int)grp, root, lo, hi);
        C *dp = to + at;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int q = 2 * (int)grp + i;
            if (q > (p - 1) / 2) continue;
            dp[q * m * g.pitch] = q == 0 ? lo[i] : cmul(lo[i], tw[j * (p - 1) + q - 1]);
            if (q > 0) dp[(p - q) * m * g.pitch] = cmul(hi[i], tw[j * (p - 1) + p - q - 1]);
        }
    }
}

// A direct last stage: LDS -> global memory.
template <int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_direct_last(const pass_args &a, const mixed_plan &g, unsigned tile, const C *lds) {
    const int T = 1 << g.log2t, p = g.last, groups = (p + 3) / 4;
    const unsigned nb = (unsigned)(g.n / p), per_line = nb * groups;
    const C *__restrict__ root = mixed_twiddles<C>(a) + g.root_last;
    for (unsigned idx = threadIdx.x; idx < per_line << g.log2t; idx += blockDim.x) {
        unsigned l, v;
        if (a.store_colfast) {
            l = idx & (T - 1);
            v = idx >> g.log2t;
        } else {
            l = idx / per_line;
            v = idx - l * per_line;
        }
        const unsigned grp = fdiv(v, g.by_last), u = v - grp * nb;
        line_at ln;
        ln.locate(tile * T + l, a, g, true);
        if (!ln.valid) continue;
        unsigned c = 0, t = u;
#pragma unroll
        for (int s = 0; s + 2 < kMixedStages; s++) {
            if (s + 2 >= g.nst) break;
            const unsigned q = fdiv(t, g.by_r[s]);
            c = (c + t - q * (unsigned)g.radix[s]) * (unsigned)g.radix[s + 1];
            t = q;
        }
        c += t;
        C lo[2], hi[2];
        mixed_direct_sums<R>(lds + (int)c * p * g.pitch + (int)l, g.pitch, p, 2 * (int)grp, root, lo, hi);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int q = 2 * (int)grp + i;
            if (q > (p - 1) / 2) continue;
            const C x[1] = {lo[i]}, y[1] = {hi[i]};
            mixed_store<1, kFormAny, NTM, R>(x, a, g, ln, (int)(u + nb * q), 0);
            if (q > 0) mixed_store<1, kFormAny, NTM, R>(y, a, g, ln, (int)(u + nb * (p - q)), 0);
        }
    }
}

// Radices of the light build (every thread holds at most kLightRadix values), what the full one adds, and
// those of the odd one.
#define HMI_MIXED_LIGHT(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10)
#define HMI_MIXED_HEAVY(X) X(11) X(12) X(13) X(14) X(15) X(16)
#define HMI_MIXED_ODD(X) X(3) X(5) X(7) X(9)

template <typename R, int SET, int FORM, int NTM>
__global__ void __launch_bounds__(kMixedThreads) fft_generic(pass_args a, mixed_plan g) {
    using C = typename cvec<R>::type;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    unsigned tile = blockIdx.x;
    if (a.load_colfast || a.store_colfast) {
        // the numbering of fft_uniform's tiles, by the width of a column chunk
        const int chunk = (int)sizeof(C) << g.log2t;
        if (chunk >= 128 && chunk < 1024) {
            tile = chunk >= 512 ? xcd_grouped_tile<2>(tile, gridDim.x)
                 : chunk >= 256 ? xcd_grouped_tile<4>(tile, gridDim.x) : xcd_grouped_tile<8>(tile, gridDim.x);
        } else if (chunk <= 32) {
            tile = chunk == 32 ? xcd_grouped_tile<4>(tile, gridDim.x)
                 : chunk == 16 ? xcd_grouped_tile<8>(tile, gridDim.x) : xcd_grouped_tile<16>(tile, gridDim.x);
        }
    }
#define HMI_MIXED_FIRST(RX) case RX: mixed_first<RX, SET, FORM, NTM, R>(a, g, tile, lds); break;
#define HMI_MIXED_ONLY(RX) case RX: mixed_only<RX, SET>(g, lds); break;
#define HMI_MIXED_MID(RX) case RX: mixed_middle<RX, SET, false, R>(a, g, st, lds); break;
#define HMI_MIXED_BACK(RX) case RX: mixed_middle<RX, SET, true, R>(a, g, st, lds); break;
#define HMI_MIXED_CENTER(RX) case RX: mixed_center<RX, SET, R>(a, g, st, lds); break;
#define HMI_MIXED_LAST(RX) case RX: mixed_last<RX, SET, FORM, NTM, R>(a, g, tile, lds); break;
#define HMI_MIXED_CHIRP_LAST(RX) case RX: mixed_chirp_last<RX, SET, NTM, R>(a, g, tile, lds); break;
#define HMI_MIXED_SWITCH(R, CASE)                                                     \
    if constexpr (SET == kSetFull) {                                                  \
        switch (R) { HMI_MIXED_LIGHT(CASE) HMI_MIXED_HEAVY(CASE) }                    \
    } else if constexpr (SET == kSetOdd) {                                            \
        switch (R) { HMI_MIXED_ODD(CASE) }                                            \
    } else {                                                                          \
        switch (R) { HMI_MIXED_LIGHT(CASE) }                                          \
    }
    const mixed_stage *stages = static_cast<const mixed_stage *>(a.tw);
    [[maybe_unused]] C *other = lds + g.n * g.pitch;  // plans with two direct stages or more
    if (FORM != kFormChirp && (g.nst == 0 || g.radix[0] > 16 || (FORM == kFormAny && g.spread))) {
        if constexpr (FORM != kFormChirp) mixed_fill<FORM, NTM, R>(a, g, tile, lds);
        if constexpr (FORM == kFormAny && SET != kSetOdd) {
            if (g.spread) {
                __syncthreads();
                switch (g.radix[0]) {
                    HMI_MIXED_ONLY(10)
                    default: if constexpr (SET == kSetFull) { switch (g.radix[0]) { HMI_MIXED_HEAVY(HMI_MIXED_ONLY) } }
                }
            }
        }
        if (FORM == kFormDirect && g.nst > 1) {
            __syncthreads();
            const mixed_stage st{g.radix[0], g.m0, 0, g.by_m0, fast_div{}, g.root0};
            mixed_direct<R>(a, g, st, lds, other);
            C *t = lds; lds = other; other = t;
        }
    } else {
        HMI_MIXED_SWITCH(g.radix[0], HMI_MIXED_FIRST)
    }
    __syncthreads();
    for (int s = 1; s + 1 < g.nst; s++) {
        const mixed_stage st = stages[s - 1];
        if (FORM == kFormDirect && st.radix > 16) {
            mixed_direct<R>(a, g, st, lds, other);
            C *t = lds; lds = other; other = t;
        } else {
            HMI_MIXED_SWITCH(st.radix, HMI_MIXED_MID)
        }
        __syncthreads();
    }
    if constexpr (FORM == kFormChirp) {
        for (int s = g.nst - 1; s > 0; s--) {
            const mixed_stage st = stages[s - 1];
            if (s == g.nst - 1) {
                HMI_MIXED_SWITCH(st.radix, HMI_MIXED_CENTER)
            } else {
                HMI_MIXED_SWITCH(st.radix, HMI_MIXED_BACK)
            }
            __syncthreads();
        }
        HMI_MIXED_SWITCH(g.radix[0], HMI_MIXED_CHIRP_LAST)
    } else if (FORM == kFormDirect) {
        mixed_direct_last<NTM, R>(a, g, tile, lds);
    } else if (g.nst < 2) {
        mixed_drain<FORM, NTM, R>(a, g, tile, lds);
    } else {
        HMI_MIXED_SWITCH(g.last, HMI_MIXED_LAST)
    }
}

template <typename R> struct generic_builds {
    using fn = void (*)(pass_args, mixed_plan);
    // [radix set][kFormAny, kFormPlain, kFormPlain32, kFormChirp, kFormDirect][non-temporal: none, stores, both]
    static fn pick(int set, int form, int stream) {
#ifdef HMI_EMULATE  // the CPU tests run the kernels without the non-temporal hints
#define HMI_MIXED_BUILDS(S, F) {&fft_generic<R, S, F, 0>, nullptr, nullptr}
#else
#define HMI_MIXED_BUILDS(S, F) \
    {&fft_generic<R, S, F, 0>, &fft_generic<R, S, F, kStreamStores>, &fft_generic<R, S, F, kStreamLoadsStores>}
#endif
        static const fn f[2][5][3] = {
            {HMI_MIXED_BUILDS(kSetLight, 0), HMI_MIXED_BUILDS(kSetLight, 1), HMI_MIXED_BUILDS(kSetLight, 2), HMI_MIXED_BUILDS(kSetLight, 3), HMI_MIXED_BUILDS(kSetLight, 4)},
            {HMI_MIXED_BUILDS(kSetFull, 0), HMI_MIXED_BUILDS(kSetFull, 1), HMI_MIXED_BUILDS(kSetFull, 2), HMI_MIXED_BUILDS(kSetFull, 3), HMI_MIXED_BUILDS(kSetFull, 4)}};
        // (a plan of the odd set has neither a chirp nor direct stages)
        static const fn odd[3][3] = {HMI_MIXED_BUILDS(kSetOdd, 0), HMI_MIXED_BUILDS(kSetOdd, 1), HMI_MIXED_BUILDS(kSetOdd, 2)};
        const int at = stream == 0 ? 0 : (stream == kStreamStores ? 1 : 2);
        return set == kSetOdd ? odd[form][at] : f[set][form][at];
    }
    static int form(const pass_args &a, const mixed_plan &g) {
        if (g.chirp || g.direct) return g.chirp ? kFormChirp : kFormDirect;
        if (a.mode != kModeC2C || a.in_real || a.out_real || a.herm_load || a.mul || a.tw4 || a.store_len != g.len) return kFormAny;
        // elements up to the furthest one of either side (no stride is negative)
        auto span = [&](long long sa, long long sc, long long sb1, long long sb2) {
            return (g.n - 1) * sa + (a.ncol - 1) * sc + (a.nb1 - 1) * sb1 + (a.nbatch - 1) * sb2 + 1;
        };
        const long long most = std::max(span(a.in_sa, a.in_sc, a.in_sb1, a.in_sb2),
                                        span(a.out_sa, a.out_sc, a.out_sb1, a.out_sb2));
        return most * (long long)sizeof(typename cvec<R>::type) <= (1LL << 32) ? kFormPlain32 : kFormPlain;
    }
    static fn choose(const pass_args &a, const mixed_plan &g) { return pick(g.set, form(a, g), a.stream); }
    // Few lines of one stage of 10 to 16 points in any form: a wave that loads, transforms and stores whole
    // lines alone on its CU waits for itself.  Elements are spread over four times the threads instead, with
    // the butterflies in between (us a call, whole lines / spread: sine 14 x 15 x 4 float 14.0 / 11.8, cosine 10 x
    // (14, 14, 16) double 19.2 / 17.3, sine (12, 1, 14) double 14.3 / 12.0; with more lines it loses, r2c 4 x (32, 13,
    // 32) double 13.6 / 15.0, 64 x (64, 14, 32) 36.9 / 50.1, 36 x (33, 12, 10) 21.2 / 25.8, and so do shorter ones, r2c
    // 4 x (64, 5, 64) 13.1 / 14.7).
    static int spread(const pass_args &a, mixed_plan &g, int threads) {
        g.spread = g.nst == 1 && g.n >= 10 && a.nlines <= 3072 && form(a, g) == kFormAny;
        return g.spread ? std::max(threads, (int)std::min<long long>(256, ((long long)g.n << g.log2t) / 256 * 64)) : threads;
    }
#ifndef HMI_EMULATE
    static hipError_t launch(const pass_args &a, mixed_plan g, int threads, long long nblocks, size_t lds, hipStream_t s) {
        // once per process, thread-safe (static initialisation)
        static const bool configured = [] {
            for (int set : {kSetLight, kSetFull, kSetOdd})
                for (int form = 0; form < (set == kSetOdd ? 3 : 5); form++)
                    for (int st : {0, (int)kStreamStores, (int)kStreamLoadsStores})
                        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(pick(set, form, st)),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, kGenericMaxLds);
            return true;
        }();
        (void)configured;
        threads = spread(a, g, threads);
        choose(a, g)<<<dim3((unsigned)nblocks), dim3(threads), lds, s>>>(a, g);
        return hipGetLastError();
    }
#endif
};

}  // namespace hmi
