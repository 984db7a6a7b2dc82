// Runtime-length FFT pass (fft_generic), included by one source per precision.
//
// One block transforms a tile of lines in place in one LDS buffer (radix plan and layout: mixed_plan,
// hmi_pass.h).  The first stage takes its inputs from global memory and the last stage stores its
// outputs there, so the tile crosses LDS only between stages.  Each stage walks its butterflies over
// the block's threads with the lines of the tile fastest (lanes on consecutive lines: consecutive
// LDS elements, one twiddle for all of them, the line of a thread fixed for the whole loop), except
// the load and store of a side on which the FFT axis is the contiguous one, where lanes walk the
// axis.  All divisions are multiplications by the plan's constants.
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
// base plus one 32-bit offset per thread, half the address registers).
enum : int { kFormAny = 0, kFormPlain = 1, kFormPlain32 = 2 };

// Elements j0, j0 + step, ... (RX of them) of a line in the pass's input form.
template <int RX, int FORM, int NTM, typename R, typename C>
__device__ __forceinline__ void mixed_load(C (&x)[RX], const pass_args &a, const mixed_plan &g, const line_at &ln, int j0,
                                           int step) {
    constexpr bool NTL = (NTM & 2) != 0;
    const R sg = a.conj ? R(-1) : R(1);
    const int n = g.n;
    if (!ln.valid) {
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = cmk<C>(R(0), R(0));
    } else if (FORM == kFormAny && (a.mode == kModeDCT2 || a.mode == kModeDST2)) {
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            const int jj = (j < (n + 1) / 2) ? 2 * j : 2 * (n - 1 - j) + 1;
            const R v = ldg<NTL>(&src[(long long)jj * a.in_sa]);
            x[p] = cmk<C>((a.mode == kModeDST2 && (jj & 1)) ? -v : v, R(0));
        }
    } else if (FORM == kFormAny && (a.mode == kModeDCT3 || a.mode == kModeDST3)) {
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
    } else if (FORM == kFormAny && (a.mode == kModeDCT1 || a.mode == kModeDCT1B)) {
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            x[p] = cmk<C>(ldg<NTL>(&src[(long long)(j <= n / 2 ? j : n - j) * a.in_sa]), R(0));
        }
    } else if (FORM == kFormAny && a.in_real) {
        const R *__restrict__ src = static_cast<const R *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = cmk<C>(ldg<NTL>(&src[(long long)(j0 + p * step) * a.in_sa]), R(0));
    } else if (FORM == kFormAny && a.herm_load) {
        const C *__restrict__ src = static_cast<const C *>(a.in) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int j = j0 + p * step;
            const bool mirror = j > n / 2;
            const C v = ldg<NTL>(&src[(long long)(mirror ? n - j : j) * a.in_sa]);
            x[p] = cmk<C>(v.x, (mirror ? -sg : sg) * v.y);
        }
    } else if (FORM == kFormAny && a.mul) {
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
    const int n = g.n;
    if (FORM == kFormAny && (a.mode == kModeDCT2 || a.mode == kModeDST2)) {
        R *__restrict__ dst = static_cast<R *>(a.out) + ln.base;
        const C *__restrict__ post = mixed_twiddles<C>(a) + g.postoff;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int k = k0 + p * step;
            const C w = post[k];
            stg<NTS>(&dst[(long long)(a.mode == kModeDST2 ? n - 1 - k : k) * a.out_sa],
                     R(2) * (w.x * x[p].x - w.y * x[p].y) * sc);
        }
    } else if (FORM == kFormAny && (a.mode == kModeDCT3 || a.mode == kModeDST3)) {
        R *__restrict__ dst = static_cast<R *>(a.out) + ln.base;
#pragma unroll
        for (int p = 0; p < RX; p++) {
            const int k = k0 + p * step;
            const int j = (k < (n + 1) / 2) ? 2 * k : 2 * (n - 1 - k) + 1;
            const R y = R(2) * x[p].x;
            stg<NTS>(&dst[(long long)j * a.out_sa], ((a.mode == kModeDST3 && (j & 1)) ? -y : y) * sc);
        }
    } else if (FORM == kFormAny && a.out_real) {
        R *__restrict__ dst = static_cast<R *>(a.out) + ln.base;
        const R f = (a.mode == kModeDCT1B) ? R(2) * sc : sc;
#pragma unroll
        for (int p = 0; p < RX; p++)
            if (k0 + p * step < a.store_len) stg<NTS>(&dst[(long long)(k0 + p * step) * a.out_sa], x[p].x * f);
    } else if (FORM == kFormAny && (a.store_len < n || a.tw4)) {
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

// Stage 0: global memory -> LDS.
template <int RX, int FORM, int NTM, typename R, typename C>
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
        mixed_load<RX, FORM, NTM, R>(x, a, g, ln, j, m);
        dft<RX>::run(x);
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

// A stage between two others, in place in LDS.
template <int RX, typename R, typename C>
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
        dft<RX>::run(x);
        const C *w = tw + j * (RX - 1);
#pragma unroll
        for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * stride] = x[q];
    }
}

// The last stage: LDS -> global memory.
template <int RX, int FORM, int NTM, typename R, typename C>
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
        dft<RX>::run(x);
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

// Radices of the light build (every thread holds at most kLightRadix values) and of the full one.
#define HMI_MIXED_LIGHT(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10)
#define HMI_MIXED_HEAVY(X) X(11) X(12) X(13) X(14) X(15) X(16)

template <typename R, bool HEAVY, int FORM, int NTM>
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
#define HMI_MIXED_FIRST(RX) case RX: mixed_first<RX, FORM, NTM, R>(a, g, tile, lds); break;
#define HMI_MIXED_MID(RX) case RX: mixed_middle<RX, R>(a, g, st, lds); break;
#define HMI_MIXED_LAST(RX) case RX: mixed_last<RX, FORM, NTM, R>(a, g, tile, lds); break;
    if (g.nst == 0) {
        mixed_fill<FORM, NTM, R>(a, g, tile, lds);
    } else if constexpr (HEAVY) {
        switch (g.radix[0]) { HMI_MIXED_LIGHT(HMI_MIXED_FIRST) HMI_MIXED_HEAVY(HMI_MIXED_FIRST) }
    } else {
        switch (g.radix[0]) { HMI_MIXED_LIGHT(HMI_MIXED_FIRST) }
    }
    __syncthreads();
    for (int s = 1; s + 1 < g.nst; s++) {
        const mixed_stage st = static_cast<const mixed_stage *>(a.tw)[s - 1];
        if constexpr (HEAVY) {
            switch (st.radix) { HMI_MIXED_LIGHT(HMI_MIXED_MID) HMI_MIXED_HEAVY(HMI_MIXED_MID) }
        } else {
            switch (st.radix) { HMI_MIXED_LIGHT(HMI_MIXED_MID) }
        }
        __syncthreads();
    }
    if (g.nst < 2) {
        mixed_drain<FORM, NTM, R>(a, g, tile, lds);
    } else if constexpr (HEAVY) {
        switch (g.last) { HMI_MIXED_LIGHT(HMI_MIXED_LAST) HMI_MIXED_HEAVY(HMI_MIXED_LAST) }
    } else {
        switch (g.last) { HMI_MIXED_LIGHT(HMI_MIXED_LAST) }
    }
}

template <typename R> struct generic_builds {
    using fn = void (*)(pass_args, mixed_plan);
    // [full radix set][kFormAny, kFormPlain, kFormPlain32][non-temporal: none, stores, loads and stores]
    static fn pick(bool heavy, int form, int stream) {
#ifdef HMI_EMULATE  // the CPU tests run the kernels without the non-temporal hints
#define HMI_MIXED_BUILDS(H, F) {&fft_generic<R, H, F, 0>, nullptr, nullptr}
#else
#define HMI_MIXED_BUILDS(H, F) \
    {&fft_generic<R, H, F, 0>, &fft_generic<R, H, F, kStreamStores>, &fft_generic<R, H, F, kStreamLoadsStores>}
#endif
        static const fn f[2][3][3] = {
            {HMI_MIXED_BUILDS(false, 0), HMI_MIXED_BUILDS(false, 1), HMI_MIXED_BUILDS(false, 2)},
            {HMI_MIXED_BUILDS(true, 0), HMI_MIXED_BUILDS(true, 1), HMI_MIXED_BUILDS(true, 2)}};
        return f[heavy ? 1 : 0][form][stream == 0 ? 0 : (stream == kStreamStores ? 1 : 2)];
    }
    static fn choose(const pass_args &a, const mixed_plan &g) {
        int top = 0;
        for (int i = 0; i < g.nst; i++) top = std::max(top, g.radix[i]);
        const bool plain = a.mode == kModeC2C && !a.in_real && !a.out_real && !a.herm_load && !a.mul && !a.tw4 &&
                           a.store_len == g.n;
        // elements up to the furthest one of either side (no stride is negative)
        auto span = [&](long long sa, long long sc, long long sb1, long long sb2) {
            return (g.n - 1) * sa + (a.ncol - 1) * sc + (a.nb1 - 1) * sb1 + (a.nbatch - 1) * sb2 + 1;
        };
        const long long most = std::max(span(a.in_sa, a.in_sc, a.in_sb1, a.in_sb2),
                                        span(a.out_sa, a.out_sc, a.out_sb1, a.out_sb2));
        const bool near = most * (long long)sizeof(typename cvec<R>::type) <= (1LL << 32);
        return pick(top > kLightRadix, !plain ? kFormAny : (near ? kFormPlain32 : kFormPlain), a.stream);
    }
#ifndef HMI_EMULATE
    static hipError_t launch(const pass_args &a, const mixed_plan &g, int threads, long long nblocks, size_t lds,
                             hipStream_t s) {
        // once per process, thread-safe (static initialisation)
        static const bool configured = [] {
            for (bool heavy : {false, true})
                for (int form = 0; form < 3; form++)
                    for (int st : {0, (int)kStreamStores, (int)kStreamLoadsStores})
                        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(pick(heavy, form, st)),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, kGenericMaxLds);
            return true;
        }();
        (void)configured;
        choose(a, g)<<<dim3((unsigned)nblocks), dim3(threads), lds, s>>>(a, g);
        return hipGetLastError();
    }
#endif
};

}  // namespace hmi
