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
// (48, 60, 72) 73 -> 58; complex<double> 256 x 64^3 1095 -> 731, 8 x (70, 70, 256) 204 -> 123.  Its accesses take
// the caches' default policy at any size: outputs above the Infinity Cache, default / non-temporal stores /
// non-temporal loads and stores, us of a whole transform, complex<float> 512 x 64^3 729 / 742 / 759, 400 x
// (48, 60, 72) 507 / 520 / 603, 32768 x 16^3 825 / 814 / 1582, 262144 x 8^3 686 / 717 / 1018, complex<double>
// 40 x 100^3 511 / 520 / 534.
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
template <int RX, int SET, bool COLS, typename C>
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
        butterfly<RX, SET == kSetOdd>(x);
        if (m > 1) {
            const C *w = tw + j * (RX - 1);
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], w[q - 1]);
        }
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * stride] = x[q];
    }
}

// First row stage, global memory -> LDS (lanes walk the rows).  (Values through ldg: where the choice below is
// one between addresses, the compiler turns every access into flat and scratch ones, 745 -> 1077 us for
// 512 x 64^3 complex<float>.)
template <int RX, int SET, typename R, typename C>
__device__ __forceinline__ void plane_load(const plane_args &a, const C *__restrict__ tw, long long base, unsigned rows, C *lds) {
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
        for (int p = 0; p < RX; p++) x[p] = ldg<false>(in + p * m + off);
        if (mul) {
            C y[RX];
#pragma unroll
            for (int p = 0; p < RX; p++) y[p] = a.mul == a.in ? x[p] : ldg<false>(mul + p * m + off);
#pragma unroll
            for (int p = 0; p < RX; p++) x[p] = cmul(x[p], y[p]);
        }
#pragma unroll
        for (int p = 0; p < RX; p++) x[p].y *= sg;
        butterfly<RX, SET == kSetOdd>(x);
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
template <int RX, int SET, typename R, typename C>
__device__ __forceinline__ void plane_store(const plane_args &a, long long base, unsigned cols, const C *lds) {
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
        butterfly<RX, SET == kSetOdd>(x);
        const unsigned off = (pl * (unsigned)a.n1 + u) * (unsigned)a.n0 + k0;
        const unsigned st = nb * (unsigned)a.n0;
#pragma unroll
        for (int q = 0; q < RX; q++) stg<false>(out + q * st + off, cmk<C>(x[q].x * sc, x[q].y * sy));
    }
}

template <typename R, int SET> __global__ void __launch_bounds__(kMixedThreads) fft_plane(plane_args a) {
    using C = typename cvec<R>::type;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    const unsigned p0 = blockIdx.x * (unsigned)a.planes;
    const unsigned planes = p0 + a.planes <= (unsigned)a.nplanes ? (unsigned)a.planes : (unsigned)a.nplanes - p0;
    const long long base = (long long)p0 * a.n0 * a.n1;
    const C *__restrict__ tw0 = reinterpret_cast<const C *>(static_cast<const char *>(a.tw0) + kMixedHead);
    const C *__restrict__ tw1 = reinterpret_cast<const C *>(static_cast<const char *>(a.tw1) + kMixedHead);
    const mixed_stage *st0 = static_cast<const mixed_stage *>(a.tw0), *st1 = static_cast<const mixed_stage *>(a.tw1);
#define HMI_PLANE_LOAD(RX) case RX: plane_load<RX, SET, R>(a, tw0, base, planes * (unsigned)a.n1, lds); break;
#define HMI_PLANE_ROW(RX) case RX: plane_stage<RX, SET, false>(a, a.g0, tw0 + st.twoff, st.m, st.by_m, lds); break;
#define HMI_PLANE_COL0(RX) case RX: plane_stage<RX, SET, true>(a, a.g1, tw1, a.g1.m0, a.g1.by_m0, lds); break;
#define HMI_PLANE_COL(RX) case RX: plane_stage<RX, SET, true>(a, a.g1, tw1 + st.twoff, st.m, st.by_m, lds); break;
#define HMI_PLANE_STORE(RX) case RX: plane_store<RX, SET, R>(a, base, planes * (unsigned)a.n0, lds); break;
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

// ---- batches: the same stages over work lists of transforms of different sizes

// Copy of a device-resident radix plan (uniform over the block: scalar loads)
__device__ __forceinline__ mixed_plan load_plan(const mixed_plan *p) {
#ifdef HMI_EMULATE
    return *p;
#else
    mixed_plan g;
    const auto *src = (const __attribute__((address_space(4))) int *)(uintptr_t)p;
    int *dst = reinterpret_cast<int *>(&g);
#pragma unroll
    for (unsigned i = 0; i < sizeof(mixed_plan) / 4; i++) dst[i] = src[i];
    return g;
#endif
}

// First stage of a column block, global memory -> LDS: position i of column l at src + i row + l.
template <int RX, int SET, typename R, typename C>
__device__ __forceinline__ void cols_load(const plane_args &a, const C *__restrict__ tw, const C *src, long long row, unsigned w,
                                          C *lds) {
    const int m = a.g1.m0;
    const R sg = a.conj ? R(-1) : R(1);
    for (unsigned idx = threadIdx.x; idx < a.cols * (unsigned)m; idx += blockDim.x) {
        const unsigned j = fdiv(idx, a.by_cols), l = idx - j * a.cols;
        if (l >= w) continue;
        const C *sp = src + (long long)j * row + l;
        const long long st = (long long)m * row;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = sp[p * st];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p].y *= sg;
        butterfly<RX, SET == kSetOdd>(x);
        if (m > 1) {
            const C *wt = tw + j * (RX - 1);
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], wt[q - 1]);
        }
        C *dp = lds + (int)j * a.rp + (int)l;
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * m * a.rp] = x[q];
    }
}

// Last stage of a column block, LDS -> global memory.
template <int RX, int SET, typename R, typename C>
__device__ __forceinline__ void cols_store(const plane_args &a, C *dst, long long row, unsigned w, const C *lds) {
    const unsigned nb = (unsigned)(a.g1.n / RX);
    const R sc = (R)a.scale, sy = a.conj ? -sc : sc;
    for (unsigned idx = threadIdx.x; idx < nb * a.cols; idx += blockDim.x) {
        const unsigned u = fdiv(idx, a.by_cols), l = idx - u * a.cols;
        if (l >= w) continue;
        const C *sp = lds + (int)plane_block(u, a.g1) * RX * a.rp + (int)l;
        C x[RX];
#pragma unroll
        for (int p = 0; p < RX; p++) x[p] = sp[p * a.rp];
        butterfly<RX, SET == kSetOdd>(x);
        C *dp = dst + (long long)u * row + l;
        const long long st = (long long)nb * row;
#pragma unroll
        for (int q = 0; q < RX; q++) dp[q * st] = cmk<C>(x[q].x * sc, x[q].y * sy);
    }
}

// One-stage lengths: the transformed columns back to global memory.
template <typename R, typename C>
__device__ __forceinline__ void cols_copy(const plane_args &a, C *dst, long long row, unsigned w, const C *lds) {
    const R sc = (R)a.scale, sy = a.conj ? -sc : sc;
    for (unsigned idx = threadIdx.x; idx < a.cols * (unsigned)a.g1.n; idx += blockDim.x) {
        const unsigned k = fdiv(idx, a.by_cols), l = idx - k * a.cols;
        if (l >= w) continue;
        const C v = lds[(int)k * a.rp + (int)l];
        dst[(long long)k * row + l] = cmk<C>(v.x * sc, v.y * sy);
    }
}

// Fused phases of a batch.  XY: item = (transform, group of consecutive z-planes), both axes of the
// planes in LDS, input to output arrays, no scale.  Otherwise: item = (transform, block of consecutive
// (x, y) positions), their z lines, in place in the output arrays, with the scale.
//
// Bound: HBM bytes in the z phase, LDS and issue inside the blocks in the x-y phase.  1000 transforms of
// sides 16 ... 128, complex<float>, 1.5 GB: x-y 0.79 ms (3.8 TB/s, in three launches by block size),
// z 0.62 ms (4.8 TB/s) a direction, pair 3.69 -> 2.83 ms against compile-time tiles that held whole
// butterfly chains per line in registers (two 256-thread blocks per CU; x-y 1.2 ms, z 0.75 ms).  Measured
// around it: radices up to 10 only 3.10 ms; first block size 32, 24 or 52 KB 2.84-2.88; 512 threads in it
// 3.00, 256 in the second 2.92; z blocks of 20 KB 2.94, of 80 KB with 512 threads 2.79.
template <typename R, bool XY> __global__ void __launch_bounds__(kMixedThreads) fft_batch_fused(batch_args b) {
    using C = typename cvec<R>::type;
    constexpr int SET = kSetFull;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    for (int i = blockIdx.x; i < b.nitems; i += gridDim.x) {
        const batch_item it = b.items[i];
        const batch_xform x = b.xforms[it.xform];
        const batch_fused f = b.fused[it.xform];
        const int n0 = x.n[0], n1 = x.n[1], n2 = x.n[2];
        plane_args a;
        a.mul = nullptr;
        a.conj = b.conj;
        const C *in = b.from_in ? static_cast<const C *>(b.in) + x.in_off : static_cast<const C *>(b.out) + x.out_off;
        C *out = static_cast<C *>(b.out) + x.out_off;
        a.in = in;
        a.out = out;
        const int id1 = x.size_id[XY ? 1 : 2];
        a.g1 = load_plan(b.mplans + id1);
        const unsigned char *t1 = b.mtab + b.mtoff[id1];
        const C *__restrict__ tw1 = reinterpret_cast<const C *>(t1 + kMixedHead);
        const mixed_stage *st1 = reinterpret_cast<const mixed_stage *>(t1);
        unsigned planes = 0, w = 0;
        long long base = 0;
        const long long row = (long long)n0 * n1;
        if constexpr (XY) {
            const int id0 = x.size_id[0];
            a.g0 = load_plan(b.mplans + id0);
            const unsigned char *t0 = b.mtab + b.mtoff[id0];
            const C *__restrict__ tw0 = reinterpret_cast<const C *>(t0 + kMixedHead);
            const mixed_stage *st0 = reinterpret_cast<const mixed_stage *>(t0);
            const unsigned z0 = (unsigned)(it.tile * f.planes);
            planes = (unsigned)(n2 - (int)z0 < f.planes ? n2 - (int)z0 : f.planes);
            base = z0 * row;
            a.n0 = n0;
            a.n1 = n1;
            a.rp = n0 | 1;
            a.ps = n1 * a.rp;
            a.rows = (unsigned)(f.planes * n1);
            a.cols = (unsigned)(f.planes * n0);
            a.by_rows = f.by_rows;
            a.by_cols = f.by_cols;
            a.by_n0 = f.by_n0;
            a.scale = 1.0;
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
        } else {
            const long long c0 = (long long)it.tile * f.width;
            w = (unsigned)(row - c0 < f.width ? row - c0 : f.width);
            a.n0 = f.width;
            a.rp = f.width;
            a.ps = 0;
            a.cols = (unsigned)f.width;
            a.by_cols = f.by_width;
            a.by_n0 = f.by_width;
            const double ntot = (double)row * (double)n2;
            a.scale = (b.scaling == 0) ? 1.0 : (b.scaling == 1 ? 1.0 / ntot : sqrt(1.0 / ntot));
            in += c0;
            out += c0;
#define HMI_COLS_LOAD(RX) case RX: cols_load<RX, SET, R>(a, tw1, in, row, w, lds); break;
            HMI_MIXED_SWITCH(a.g1.radix[0], HMI_COLS_LOAD)
            __syncthreads();
        }
        for (int s = 1; s + 1 < a.g1.nst; s++) {
            const mixed_stage st = st1[s - 1];
            HMI_MIXED_SWITCH(st.radix, HMI_PLANE_COL)
            __syncthreads();
        }
        if constexpr (XY) {
            HMI_MIXED_SWITCH(a.g1.last, HMI_PLANE_STORE)
        } else {
#define HMI_COLS_STORE(RX) case RX: cols_store<RX, SET, R>(a, out, row, w, lds); break;
            if (a.g1.nst == 1) cols_copy<R>(a, out, row, w, lds);
            else { HMI_MIXED_SWITCH(a.g1.last, HMI_COLS_STORE) }
        }
        __syncthreads();
    }
}

template <typename R> struct plane_builds {
    using fn = void (*)(plane_args);
    static fn choose(const plane_args &a) {
        // both axes in one set: the odd one only for two plans of it (its radices are light ones too)
        const int set = a.g0.set == kSetFull || a.g1.set == kSetFull ? kSetFull : a.g0.set == a.g1.set ? a.g0.set : kSetLight;
        static const fn f[3] = {&fft_plane<R, kSetLight>, &fft_plane<R, kSetFull>, &fft_plane<R, kSetOdd>};
        return f[set];
    }
#ifndef HMI_EMULATE
    static hipError_t launch(const plane_args &a, int threads, long long nblocks, size_t lds, hipStream_t s) {
        // once per process, thread-safe (static initialisation)
        static const bool configured = [] {
            for (int set : {kSetLight, kSetFull, kSetOdd}) {
                plane_args p{};
                p.g0.set = p.g1.set = set;
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

#ifndef HMI_EMULATE
template <typename R> hipError_t launch_batch_builds(bool xy, const batch_args &b, int threads, int nblocks, size_t lds, hipStream_t s) {
    static const bool configured = [] {
        for (const void *f : {reinterpret_cast<const void *>(&fft_batch_fused<R, true>),
                              reinterpret_cast<const void *>(&fft_batch_fused<R, false>)})
            (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kGenericMaxLds);
        return true;
    }();
    (void)configured;
    if (threads > kMixedThreads || lds > (size_t)kGenericMaxLds) return hipErrorInvalidValue;
    (xy ? &fft_batch_fused<R, true> : &fft_batch_fused<R, false>)
        <<<dim3((unsigned)nblocks), dim3(threads), lds, s>>>(b);
    return hipGetLastError();
}
#endif

}  // namespace hmi
