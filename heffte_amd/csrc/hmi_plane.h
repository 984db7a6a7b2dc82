// Fused pass over the two fastest axes of a box (fft_plane), included by one source per precision.
//
// One block takes whole planes (n0 x n1, contiguous in memory) of one layout: the n0-point transforms
// of the rows and the n1-point ones of the columns run in place in one LDS buffer with the radix plans
// and tables of the runtime-length pass; the first row stage loads from and the last column stage
// stores to global memory.  Rows end with frequency k0 at position pos(k0) of their plan, columns work
// on positions, and the final store walks k0 so that lanes write consecutive elements.  Two axes thus
// cost one read and one write of the array and one launch.
//
// Bound: LDS and issue latency inside the block (2.7-3.8 TB/s of its own read + write), still less than
// the pass over the array and the launch it saves.  Two passes against three, us a transform: 32^3
// complex<float> 12.0 -> 9.1, 64^3 13.2 -> 10.0, 256 x 64^3 596 -> 379, 16 x 100^3 133 -> 96, 40 x
// (48, 60, 72) 73 -> 58; complex<double> 256 x 64^3 1095 -> 731, 8 x (70, 70, 256) 204 -> 123.
#pragma once
#include "hmi_generic.h"

namespace hmi {

// Position of frequency k after all stages of a plan (natural LDS stride), and the block of its last
// stage that holds the frequencies u + q n / r_last.
__device__ __forceinline__ unsigned plane_block(unsigned u, const mixed_plan &g) {
    unsigned c = 0;
#pragma unroll
    for (int s = 0; s + 2 < kMixedStages; s++) {
        if (s + 2 >= g.nst) break;
        const unsigned q = fdiv(u, g.by_r[s]);
        c = (c + u - q * (unsigned)g.radix[s]) * (unsigned)g.radix[s + 1];
        u = q;
    }
    return c + u;
}
__device__ __forceinline__ int plane_position(unsigned k, const mixed_plan &g) {
    unsigned c = 0;
#pragma unroll
    for (int s = 0; s + 1 < kMixedStages; s++) {
        if (s + 1 >= g.nst) break;
        const unsigned q = fdiv(k, g.by_r[s]);
        c = (c + k - q * (unsigned)g.radix[s]) * (unsigned)g.radix[s + 1];
        k = q;
    }
    return (int)(c + k);
}

// One axis of the plane: stage s of every line of the block in place in LDS.  A line is a row (stride
// rp between rows, elements 1 apart) or a column (columns 1 apart, planes ps apart, elements rp apart).
template <int RX, bool COLS, typename C>
__device__ __forceinline__ void plane_stage(const plane_args &a, const mixed_plan &g, const C *__restrict__ tw, int m,
                                            const fast_div &by_m, C *lds) {
    const unsigned nb = (unsigned)(g.n / RX), nlines = COLS ? a.cols : a.rows;
    const fast_div by_lines = COLS ? a.by_cols : a.by_rows;
    const int es = COLS ? a.rp : 1, stride = m * es;
    for (unsigned idx = threadIdx.x; idx < nb * nlines; idx += blockDim.x) {
        const unsigned b = fdiv(idx, by_lines), l = idx - b * nlines;
        const unsigned c = fdiv(b, by_m);
        const int j = (int)(b - c * (unsigned)m);
        int at = ((int)c * RX * m + j) * es;
        if (COLS) {
            const unsigned pl = fdiv(l, a.by_n0);
            at += (int)pl * a.ps + (int)(l - pl * (unsigned)a.n0);
        } else {
            at += (int)l * a.rp;
        }
        C *dp = lds + at;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = dp[p * stride];
        dft<RX>::run(x);
        if (m > 1) {
            const C *w = tw + j * (RX - 1);
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        }
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * stride] = x[q];
    }
}

// First row stage, global memory -> LDS (lanes walk the rows).
template <int RX, int NTM, typename R, typename C>
__device__ __forceinline__ void plane_load(const plane_args &a, const C *__restrict__ tw, long long base, unsigned rows, C *lds) {
    constexpr bool NTL = (NTM & 2) != 0;
    const int m = a.g0.m0;
    const R sg = a.conj ? R(-1) : R(1);
    const C *in = static_cast<const C *>(a.in) + base;
    const C *mul = a.mul ? static_cast<const C *>(a.mul) + base : nullptr;
    for (unsigned idx = threadIdx.x; idx < rows * (unsigned)m; idx += blockDim.x) {
        const unsigned row = fdiv(idx, a.g0.by_m0);
        const int j = (int)(idx - row * (unsigned)m);
        const unsigned off = row * (unsigned)a.n0 + (unsigned)j;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = ldg<NTL>(in + p * m + off);
        if (mul) {
            C y[RX];
#pragma unroll
            for (int p = 0; p < RX; p++) y[p] = a.mul == a.in ? x[p] : ldg<NTL>(mul + p * m + off);
#pragma unroll
            for (int p = 0; p < RX; p++) x[p] = cmul(x[p], y[p]);
        }
#pragma unroll
        for (int p = 0; p < RX; p++) x[p].y *= sg;
        dft<RX>::run(x);
        if (m > 1) {
            const C *w = tw + j * (RX - 1);
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        }
        C *dp = lds + (int)row * a.rp + j;
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * m] = x[q];
    }
}

// Last column stage, LDS -> global memory (lanes walk the columns in frequency order).
template <int RX, int NTM, typename R, typename C>
__device__ __forceinline__ void plane_store(const plane_args &a, long long base, unsigned cols, const C *lds) {
    constexpr bool NTS = (NTM & 1) != 0;
    const unsigned nb = (unsigned)(a.g1.n / RX);
    const R sc = (R)a.scale, sy = a.conj ? -sc : sc;
    C *__restrict__ out = static_cast<C *>(a.out) + base;
    for (unsigned idx = threadIdx.x; idx < nb * cols; idx += blockDim.x) {
        unsigned u, l;
        if (cols == a.cols) u = fdiv(idx, a.by_cols);
        else u = idx / cols;  // the last, partial group of planes
        l = idx - u * cols;
        const unsigned pl = fdiv(l, a.by_n0), k0 = l - pl * (unsigned)a.n0;
        const C *sp = lds + (int)pl * a.ps + plane_position(k0, a.g0) + (int)plane_block(u, a.g1) * RX * a.rp;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = sp[p * a.rp];
        dft<RX>::run(x);
        const unsigned off = (pl * (unsigned)a.n1 + u) * (unsigned)a.n0 + k0;
        const unsigned st = nb * (unsigned)a.n0;
#pragma unroll
        for (int q = 0; q < RX; q++) stg<NTS>(out + q * st + off, cmk<C>(x[q].x * sc, x[q].y * sy));
    }
}

template <typename R, bool HEAVY, int NTM> __global__ void __launch_bounds__(kMixedThreads) fft_plane(plane_args a) {
    using C = typename cvec<R>::type;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    const unsigned p0 = blockIdx.x * (unsigned)a.planes;
    const unsigned planes = p0 + a.planes <= (unsigned)a.nplanes ? (unsigned)a.planes : (unsigned)a.nplanes - p0;
    const long long base = (long long)p0 * a.n0 * a.n1;
    const C *__restrict__ tw0 = reinterpret_cast<const C *>(static_cast<const char *>(a.tw0) + kMixedHead);
    const C *__restrict__ tw1 = reinterpret_cast<const C *>(static_cast<const char *>(a.tw1) + kMixedHead);
    const mixed_stage *st0 = static_cast<const mixed_stage *>(a.tw0), *st1 = static_cast<const mixed_stage *>(a.tw1);
#define HMI_PLANE_LOAD(RX) case RX: plane_load<RX, NTM, R>(a, tw0, base, planes * (unsigned)a.n1, lds); break;
#define HMI_PLANE_ROW(RX) case RX: plane_stage<RX, false>(a, a.g0, tw0 + st.twoff, st.m, st.by_m, lds); break;
#define HMI_PLANE_COL0(RX) case RX: plane_stage<RX, true>(a, a.g1, tw1, a.g1.m0, a.g1.by_m0, lds); break;
#define HMI_PLANE_COL(RX) case RX: plane_stage<RX, true>(a, a.g1, tw1 + st.twoff, st.m, st.by_m, lds); break;
#define HMI_PLANE_STORE(RX) case RX: plane_store<RX, NTM, R>(a, base, planes * (unsigned)a.n0, lds); break;
    // (a partial group leaves the rows and columns of the missing planes untransformed garbage in LDS)
    HMI_MIXED_SWITCH(a.g0.radix[0], HMI_PLANE_LOAD)
    __syncthreads();
    for (int s = 1; s < a.g0.nst; s++) {
        const mixed_stage st = st0[s - 1];
        HMI_MIXED_SWITCH(st.radix, HMI_PLANE_ROW)
        __syncthreads();
    }
    if (a.g1.nst > 1) {
        HMI_MIXED_SWITCH(a.g1.radix[0], HMI_PLANE_COL0)
        __syncthreads();
    }
    for (int s = 1; s + 1 < a.g1.nst; s++) {
        const mixed_stage st = st1[s - 1];
        HMI_MIXED_SWITCH(st.radix, HMI_PLANE_COL)
        __syncthreads();
    }
    HMI_MIXED_SWITCH(a.g1.last, HMI_PLANE_STORE)
}

template <typename R> struct plane_builds {
    using fn = void (*)(plane_args);
    static fn choose(const plane_args &a) {
        int top = 0;
        for (int i = 0; i < a.g0.nst; i++) top = std::max(top, a.g0.radix[i]);
        for (int i = 0; i < a.g1.nst; i++) top = std::max(top, a.g1.radix[i]);
#ifdef HMI_EMULATE
        return top > kLightRadix ? &fft_plane<R, true, 0> : &fft_plane<R, false, 0>;
#else
        static const fn f[2][2] = {{&fft_plane<R, false, 0>, &fft_plane<R, false, kStreamLoadsStores>},
                                   {&fft_plane<R, true, 0>, &fft_plane<R, true, kStreamLoadsStores>}};
        return f[top > kLightRadix ? 1 : 0][a.stream ? 1 : 0];
#endif
    }
#ifndef HMI_EMULATE
    static hipError_t launch(const plane_args &a, int threads, long long nblocks, size_t lds, hipStream_t s) {
        // once per process, thread-safe (static initialisation)
        static const bool configured = [] {
            for (int stream : {0, (int)kStreamLoadsStores})
                for (int r : {2, 16}) {
                    plane_args p{};
                    p.g0.nst = 1;
                    p.g0.radix[0] = r;
                    p.stream = stream;
                    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(choose(p)),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, kGenericMaxLds);
                }
            return true;
        }();
        (void)configured;
        choose(a)<<<dim3((unsigned)nblocks), dim3(threads), lds, s>>>(a);
        return hipGetLastError();
    }
#endif
};

}  // namespace hmi
