// Runs the fused phases of a batch (fft_batch_fused, csrc/hmi_plane.h) on the CPU over the work lists a
// batch plan builds, against a direct transform in long double: boxes of many lengths without a prime factor above
// 13 (the compile-time tiles' and others, planes of every block size, z lines down to one column a block),
// arrays, tables and LDS that end where the phases may last touch them.
#include <algorithm>
#include <array>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#define HMI_EMULATE 1
#include "emulate/emulate.h"
#include "hmi_plane.h"
#include "hmi_plan.h"

namespace hmi {
alignas(16) unsigned char smem_raw[kGenericMaxLds + 64];
}

using cld = std::complex<long double>;
using size3 = std::array<int, 3>;

// exact copy of a vector on the heap
template <typename T> T *copy_of(const std::vector<T> &v) {
    T *p = new T[v.size()];
    std::copy(v.begin(), v.end(), p);
    return p;
}

void direct_axis(std::vector<cld> &x, const size3 &n, int axis, bool inverse) {
    const int len = n[axis];
    const size_t stride = axis == 0 ? 1 : axis == 1 ? n[0] : (size_t)n[0] * n[1];
    const long double pi = 3.141592653589793238462643383279502884L;
    std::vector<cld> w(len), line(len);
    for (int t = 0; t < len; t++) w[t] = cld(cosl(2 * pi * t / len), (inverse ? 1 : -1) * sinl(2 * pi * t / len));
    for (size_t at = 0; at < x.size(); at++) {
        if (at / stride % len) continue;
        for (int k = 0; k < len; k++) {
            cld s = 0;
            for (int j = 0; j < len; j++) s += x[at + j * stride] * w[(long long)j * k % len];
            line[k] = s;
        }
        for (int k = 0; k < len; k++) x[at + k * stride] = line[k];
    }
}

template <typename R> int run_batch(const std::vector<size3> &sizes, bool inverse, int scaling, bool in_place) {
    const bool dbl = sizeof(R) == 8;
    std::vector<hmi::batch_xform> xf;
    std::vector<int> lengths;
    long long nin = 0, nout = in_place ? 0 : 3;  // outputs begin at another offset and leave gaps
    for (const size3 &n : sizes) {
        hmi::batch_xform x{};
        for (int d = 0; d < 3; d++) {
            x.n[d] = n[d];
            auto it = std::find(lengths.begin(), lengths.end(), n[d]);
            x.size_id[d] = (int)(it - lengths.begin());
            if (it == lengths.end()) lengths.push_back(n[d]);
        }
        x.in_off = nin;
        x.out_off = nout;
        nin += (long long)n[0] * n[1] * n[2];
        nout += (long long)n[0] * n[1] * n[2] + (in_place ? 0 : 1);
        xf.push_back(x);
    }
    const hmi::fused_lists f = hmi::make_fused_lists(xf, lengths, dbl);
    std::mt19937 rng((unsigned)sizes.size() + scaling);
    std::uniform_real_distribution<double> d(-1, 1);
    R *in = new R[2 * nin], *out = in_place ? in : new R[2 * nout];
    if (!in_place) std::fill(out, out + 2 * nout, (R)77);
    for (long long i = 0; i < 2 * nin; i++) in[i] = (R)d(rng);
    const std::vector<R> input(in, in + 2 * nin);

    hmi::batch_args b{};
    b.in = in;
    b.out = out;
    b.xforms = copy_of(xf);
    b.fused = copy_of(f.fused);
    b.mplans = copy_of(f.plans);
    b.mtab = copy_of(f.table);
    b.mtoff = copy_of(f.offset);
    b.conj = inverse;
    int fails = 0;
    for (size_t i = 0; i < sizes.size(); i++)
        if (!f.in_xy[i] || !f.in_zc[i]) std::printf("FAIL transform %zu is not fused\n", i), fails++;
    b.from_in = 1;
    for (int k = hmi::kFusedSizes - 1; k >= 0 && !fails; k--) {
        if (f.xy[k].empty()) continue;
        b.items = copy_of(f.xy[k]);
        b.nitems = (int)f.xy[k].size();
        // (some blocks take several items)
        emulate::run_blocks((b.nitems + 1) / 2, hmi::kFusedThreads[k], hmi::smem_raw, sizeof(hmi::smem_raw), f.xy_lds[k],
                            [&] { hmi::fft_batch_fused<R, true>(b); });
        delete[] b.items;
    }
    b.from_in = 0;
    b.scaling = scaling;
    b.items = copy_of(f.zc);
    b.nitems = (int)f.zc.size();
    if (!fails)
        emulate::run_blocks((b.nitems + 1) / 2, hmi::kFusedThreads[0], hmi::smem_raw, sizeof(hmi::smem_raw), f.zc_lds,
                            [&] { hmi::fft_batch_fused<R, false>(b); });
    delete[] b.items;
    const long double tol = dbl ? 2e-15L : 1e-6L;
    std::vector<bool> written(nout, false);
    for (size_t i = 0; i < sizes.size() && !fails; i++) {
        const size3 &n = sizes[i];
        std::vector<cld> x((size_t)n[0] * n[1] * n[2]);
        for (size_t k = 0; k < x.size(); k++) x[k] = cld(input[2 * (xf[i].in_off + k)], input[2 * (xf[i].in_off + k) + 1]);
        for (int axis = 0; axis < 3; axis++) direct_axis(x, n, axis, inverse);
        const long double scale = scaling == 0 ? 1.0L : scaling == 1 ? 1.0L / x.size() : sqrtl(1.0L / x.size());
        long double num = 0, den = 0;
        for (size_t k = 0; k < x.size(); k++) {
            const size_t at = xf[i].out_off + k;
            written[at] = true;
            num += std::norm(cld(out[2 * at], out[2 * at + 1]) - x[k] * scale);
            den += std::norm(x[k] * scale);
        }
        if (!(sqrtl(num / den) <= tol)) {
            std::printf("FAIL %d x %d x %d %s: %g of the tolerance\n", n[0], n[1], n[2], dbl ? "f64" : "f32", (double)(sqrtl(num / den) / tol));
            fails++;
        }
    }
    for (long long k = 0; k < nout && !in_place; k++)
        if (!written[k] && (out[2 * k] != (R)77 || out[2 * k + 1] != (R)77)) std::printf("FAIL gap %lld was written\n", k), fails++;
    delete[] in;
    if (!in_place) delete[] out;
    delete[] b.xforms; delete[] b.fused; delete[] b.mplans; delete[] b.mtab; delete[] b.mtoff;
    return fails;
}

int main(int argc, char **argv) {
    const int share = argc > 1 ? std::atoi(argv[1]) : 0, shares = argc > 2 ? std::atoi(argv[2]) : 1;
    std::mt19937 rng(11);
    int cases = 0, fails = 0, at = 0;
    auto one = [&](bool dbl, const std::vector<size3> &sizes) {
        const bool inverse = rng() & 1, in_place = rng() % 3 == 0;
        const int scaling = (int)(rng() % 3);
        if (at++ % shares != share) return;
        cases += (int)sizes.size();
        fails += dbl ? run_batch<double>(sizes, inverse, scaling, in_place) : run_batch<float>(sizes, inverse, scaling, in_place);
    };
    const int sides[] = {2, 3, 7, 10, 13, 14, 16, 20, 27, 30, 36, 45, 50, 60, 63, 72, 77, 90, 100, 105, 128, 150};
    for (bool dbl : {false, true}) {
        for (int k = 0; k < 12; k++) {
            std::vector<size3> sizes;
            while (sizes.size() < 6) {
                const size3 n = {sides[rng() % 22], sides[rng() % 22], sides[rng() % 22]};
                if ((n[0] | 1) * n[1] * (dbl ? 16 : 8) <= hmi::kGenericMaxLds && n[0] * n[1] * n[2] <= 40000) sizes.push_back(n);
            }
            one(dbl, sizes);
        }
        // planes of every block size, one plane a block, groups with a remainder
        one(dbl, {size3{50, 60, 3}, size3{72, 60, 2}, size3{dbl ? 100 : 200, 100, 2}, size3{16, 9, 40}});
        // z lines of two columns and of one
        one(dbl, {size3{3, 2, dbl ? 1001 : 2002}, size3{2, 2, dbl ? 1300 : 2600}});
    }
    std::printf("%s %d\n", fails ? "failed" : "ok", cases);
    return fails ? 1 : 0;
}
