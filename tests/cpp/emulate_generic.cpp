// Runs the runtime-length pass kernel (csrc/hmi_generic.h) on the CPU, block by block, over many
// lengths, layouts and forms, against a direct DFT in long double.  Every array ends at the last
// element the pass may touch and the LDS ends at the size the launch would ask for, so
// AddressSanitizer sees any access past them.  Prints one line per failure, "ok <cases>" at the end.
#include <algorithm>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#define HMI_EMULATE 1
#include "emulate/emulate.h"
#include "hmi_generic.h"
#include "hmi_plan.h"

namespace hmi {
alignas(16) unsigned char smem_raw[kGenericMaxLds + 64];
}

using hmi::pass_args;
using cld = std::complex<long double>;

// exp(2 pi i t / m) from a table
struct roots {
    long long m;
    std::vector<cld> w;
    explicit roots(long long m_) : m(m_), w(m_) {
        const long double pi = 3.141592653589793238462643383279502884L;
        for (long long t = 0; t < m; t++) w[t] = cld(cosl(2 * pi * t / m), sinl(2 * pi * t / m));
    }
    cld operator()(long long t) const { return w[t % m]; }
};

struct sides { long long sa, sc, sb1, sb2, span; };

// strides of a (n, ncol, nb1) box in one of the six orders, batches behind each other
sides layout_of(int order, long long n, long long ncol, long long nb1) {
    const int o[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
    const long long ext[3] = {n, ncol, nb1};
    long long st[3], s = 1;
    for (int i = 0; i < 3; i++) { st[o[order][i]] = s; s *= ext[o[order][i]]; }
    return {st[0], st[1], st[2], s, s};
}

template <typename R> int run_case(int n, int mode, int flags, int oi, int oo, int ncol, int nb1, int batch, unsigned seed,
                                   std::string &what, double limit = 0) {
    using C = typename hmi::cvec<R>::type;
    const bool dbl = sizeof(R) == 8;
    const bool copy = flags & 1, in_real = flags & 2, out_real = flags & 4, half = flags & 8, herm = flags & 16,
               product = flags & 32, inverse = flags & 64, square = flags & 128, split = flags & 256;
    const bool r2r = mode >= hmi::kModeDCT2;
    // points of the line in memory on either side (n: length of the kernel's transform)
    long long nin = n, nout = n;
    if (mode == hmi::kModeDCT1 || mode == hmi::kModeDCT1B) nin = nout = n / 2 + 1;
    if (half) nout = n / 2 + 1;
    if (herm) nin = n / 2 + 1;
    const sides si = layout_of(oi, nin, ncol, nb1), so = layout_of(oo, nout, ncol, nb1);
    const bool load_across = si.sa != 1 && nin > 1, store_across = so.sa != 1 && nout > 1;
    const int tail = (mode >= hmi::kModeDCT2 && mode <= hmi::kModeDST3) ? n : 0;
    // the full tile, or the one a launch of these lines takes
    hmi::mixed_tiles tiles(n, dbl, copy, load_across, store_across, tail);
    const hmi::mixed_config &c = (flags & 1024) || !tiles.full().ok ? tiles.full() : tiles.of((long long)ncol * nb1 * batch);
    what = "n=" + std::to_string(n) + (dbl ? " f64" : " f32") + " mode=" + std::to_string(mode) + " flags=" +
           std::to_string(flags) + " orders=" + std::to_string(oi) + std::to_string(oo) + " ncol=" + std::to_string(ncol) +
           " nb1=" + std::to_string(nb1) + " batch=" + std::to_string(batch);
    if (!c.ok) { what += ": no plan"; return 1; }
    const bool rin = r2r || in_real, rout = r2r || out_real;
    std::mt19937 rng(seed);
    std::uniform_real_distribution<double> d(-1, 1);
    const size_t cin = (size_t)batch * si.span, cout = (size_t)batch * so.span;
    R *in = new R[cin * (rin ? 1 : 2)], *mul = product ? new R[cin * 2] : nullptr, *out = new R[cout * (rout ? 1 : 2)];
    for (size_t i = 0; i < cin * (rin ? 1 : 2); i++) in[i] = (R)d(rng);
    if (mul) for (size_t i = 0; i < cin * 2; i++) mul[i] = (R)d(rng);
    for (size_t i = 0; i < cout * (rout ? 1 : 2); i++) out[i] = (R)77;
    const std::vector<unsigned char> tab = hmi::mixed_table(c.plan, dbl, 4LL * n);
    unsigned char *table = new unsigned char[tab.size()];
    std::copy(tab.begin(), tab.end(), table);
    // w_{n ncol}^m of a split axis whose interleaved index is the column
    const long long n4 = (long long)n * ncol;
    C *tw4 = split ? new C[n4] : nullptr;
    const long double pi = 3.141592653589793238462643383279502884L;
    if (split)
        for (long long m = 0; m < n4; m++)
            tw4[m] = hmi::cmk<C>((R)cosl(2 * pi * m / n4), (R)-sinl(2 * pi * m / n4));
    pass_args a{};
    a.in = in; a.out = out; a.tw = table;
    a.in_sa = si.sa; a.in_sc = si.sc; a.in_sb1 = si.sb1; a.in_sb2 = si.sb2;
    a.out_sa = so.sa; a.out_sc = so.sc; a.out_sb1 = so.sb1; a.out_sb2 = so.sb2;
    a.ncol = ncol; a.nb1 = nb1; a.nbatch = batch; a.nlines = ncol * nb1 * batch;
    a.load_colfast = load_across; a.store_colfast = store_across;
    a.conj = (inverse && !r2r) ? 1 : 0;
    a.in_real = rin; a.out_real = rout;
    a.store_len = (half || mode == hmi::kModeDCT1 || mode == hmi::kModeDCT1B) ? (int)nout : n;
    a.herm_load = herm; a.mode = mode;
    a.mul = square ? (const void *)in : mul; a.tw4 = tw4; a.tw4_dim = 0;
    a.scale = 0.5;
    hmi::mixed_plan g = c.plan;
    hmi::mixed_launch_divs(g, a);
    const long long nblocks = (a.nlines + (1LL << g.log2t) - 1) >> g.log2t;
    const int threads = hmi::generic_builds<R>::spread(a, g, c.threads);
    auto kernel = hmi::generic_builds<R>::choose(a, g);
    emulate::run_blocks(nblocks, threads, hmi::smem_raw, sizeof(hmi::smem_raw), c.lds, [&] { kernel(a, g); });
    // direct transform of each line
    const roots wn(n), w4n(4 * nin), wd(2 * std::max<long long>(1, nin - 1)), ws(split ? n4 : 1);
    long double num = 0, den = 0;
    for (int b2 = 0; b2 < batch; b2++)
        for (int b1 = 0; b1 < nb1; b1++)
            for (int col = 0; col < ncol; col++) {
                const long long ib = col * si.sc + b1 * si.sb1 + b2 * si.sb2, ob = col * so.sc + b1 * so.sb1 + b2 * so.sb2;
                auto xr = [&](long long j) { return (long double)in[ib + j * si.sa]; };
                std::vector<cld> ref(nout);
                if (r2r) {
                    const long long N = nin;
                    for (long long k = 0; k < N; k++) {
                        long double y = 0;
                        for (long long j = 0; j < N; j++) {
                            switch (mode) {
                                case hmi::kModeDCT2: y += 2 * xr(j) * w4n((2 * j + 1) * k).real(); break;
                                case hmi::kModeDST2: y += 2 * xr(j) * w4n((2 * j + 1) * (k + 1)).imag(); break;
                                case hmi::kModeDCT3: y += (j == 0 ? 2 : 4) * xr(j) * w4n(j * (2 * k + 1)).real(); break;
                                case hmi::kModeDST3: y += (j == N - 1 ? 2 : 4) * xr(j) * w4n((j + 1) * (2 * k + 1)).imag(); break;
                                default: {
                                    const long double t = (j == 0 || j == N - 1) ? xr(j) : 2 * xr(j);
                                    y += (mode == hmi::kModeDCT1B ? 2 : 1) * t * wd(j * k).real();
                                }
                            }
                        }
                        ref[k] = y;
                    }
                } else {
                    std::vector<cld> x(n);
                    for (long long j = 0; j < n; j++) {
                        const long long p = (herm && j > n / 2) ? n - j : j;
                        const long long at = ib + p * si.sa;
                        x[j] = in_real ? cld(in[at], 0) : cld(in[2 * at], in[2 * at + 1]);
                        if (herm && j > n / 2) x[j] = std::conj(x[j]);
                        if (product) x[j] *= cld(mul[2 * at], mul[2 * at + 1]);
                        if (square) x[j] *= x[j];
                    }
                    for (long long k = 0; k < nout; k++) {
                        cld y = 0;
                        if (copy) y = x[k];
                        else
                            for (long long j = 0; j < n; j++) {
                                const cld w = wn(j * k);
                                y += x[j] * (inverse ? w : std::conj(w));
                            }
                        if (split) {
                            const cld w = ws(k * col);
                            y *= inverse ? w : std::conj(w);
                        }
                        ref[k] = y;
                    }
                }
                for (long long k = 0; k < nout; k++) {
                    const long long at = ob + k * so.sa;
                    const cld want = ref[k] * 0.5L;
                    const cld got = rout ? cld(out[at], 0) : cld(out[2 * at], out[2 * at + 1]);
                    const cld diff = rout ? cld(got.real() - want.real(), 0) : got - want;
                    num += std::norm(diff);
                    den += rout ? want.real() * want.real() : std::norm(want);
                }
            }
    const long double err = den > 0 ? sqrtl(num / den) : sqrtl(num);
    delete[] in; delete[] mul; delete[] out; delete[] table; delete[] tw4;
    const long double tol = limit > 0 ? (long double)limit : dbl ? 2e-15L : 1e-6L;
    if (!(err <= tol)) {
        what += ": relative error " + std::to_string((double)(err / tol)) + " of the tolerance";
        return 1;
    }
    return 0;
}

// The tile of a launch goes by all its lines: the full one from kFewBlocks blocks on, otherwise the
// largest that makes as many, or the smallest there is.
int check_tiles() {
    int fails = 0;
    for (bool dbl : {false, true})
        for (int n : {1, 7, 14, 60, 127, 240, 1000})
            for (int sides = 0; sides < 4; sides++) {
                hmi::mixed_tiles tiles(n, dbl, false, sides & 1, sides & 2, 0);
                const int full = tiles.full().plan.log2t, least = std::min(full, sides ? (dbl ? 2 : 3) : 0);
                for (long long lines : {1LL, 100LL, 330LL, 1000LL, 11880LL, 13184LL, 100000LL, 1LL << 30}) {
                    const hmi::mixed_config &c = tiles.of(lines);
                    const int l2 = c.plan.log2t;
                    const bool enough = (lines >> l2) >= hmi::kFewBlocks;
                    const bool good = l2 == full ? enough || l2 == least : (lines >> (l2 + 1)) < hmi::kFewBlocks && (enough || l2 == least);
                    if (!c.ok || !good || &tiles.of(lines) != &c) std::printf("FAIL tile n=%d sides %d lines %lld: %d\n", n, sides, lines, l2), fails++;
                }
            }
    return fails;
}

int main(int argc, char **argv) {
    const int share = argc > 1 ? std::atoi(argv[1]) : 0, shares = argc > 2 ? std::atoi(argv[2]) : 1;
    std::mt19937 rng(5);
    auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    int fails = share == 0 ? check_tiles() : 0, cases = 0, at = 0;
    auto one = [&](bool dbl, int n, int mode, int flags, int oi, int oo, int ncol, int nb1, int batch, double limit = 0) {
        if (at++ % shares != share) return;
        std::string what;
        flags |= (at & 1) * 1024;  // both tiles of a plan
        const int bad = dbl ? run_case<double>(n, mode, flags, oi, oo, ncol, nb1, batch, at, what, limit)
                            : run_case<float>(n, mode, flags, oi, oo, ncol, nb1, batch, at, what, limit);
        cases++;
        if (bad) { fails++; std::printf("FAIL %s\n", what.c_str()); std::fflush(stdout); }
    };
    // every radix alone and in each place of two- to five-stage plans, every order pair
    const int lengths[] = {1, 2, 3, 4, 5, 6, 7, 9, 10, 11, 12, 13, 14, 15, 16, 18, 21, 22, 25, 26, 30, 33, 36, 39, 44,
                           49, 50, 55, 60, 65, 72, 75, 77, 81, 84, 88, 90, 91, 98, 99, 100, 104, 110, 117, 120, 121,
                           125, 130, 140, 143, 144, 150, 169, 180, 196, 225, 240, 250, 275, 320, 343, 384, 400, 625};
    for (bool dbl : {false, true})
        for (int n : lengths)
            for (int k = 0; k < 3; k++)
                one(dbl, n, hmi::kModeC2C, pick(0, 1) * 64, k == 0 ? 0 : pick(0, 5), k == 0 ? 2 : pick(0, 5), pick(1, 21),
                    pick(1, 3), pick(1, 2));
    // direct stages, one to three of them, and chirp convolutions of two to four stages
    for (bool dbl : {false, true})
        for (int n : {17, 19, 23, 34, 37, 51, 61, 67, 68, 97, 127, 158, 186, 199, 254, 257, 289, 323, 509, 578})
            for (int k = 0; k < 3; k++)
                one(dbl, n, hmi::kModeC2C, pick(0, 1) * 64, k == 0 ? 0 : pick(0, 5), k == 0 ? 2 : pick(0, 5), pick(1, 21),
                    pick(1, 3), pick(1, 2));
    const int few[] = {1, 2, 6, 10, 12, 13, 15, 16, 17, 22, 38, 134, 289, 45, 60, 77, 105, 127, 180, 216};
    for (bool dbl : {false, true})
        for (int n : few) {
            for (int flags : {1, 2, 2 | 8, 4 | 64, 4 | 16 | 64, 16 | 64, 32, 32 | 64, 128, 256, 256 | 64, 8}) {
                if ((flags & 256) && n == 1) continue;
                one(dbl, n, hmi::kModeC2C, flags, pick(0, 5), pick(0, 5), pick(2, 19), pick(1, 3), 1);
            }
            for (int mode : {3, 4, 5, 6}) one(dbl, n, mode, 0, pick(0, 5), pick(0, 5), pick(1, 19), pick(1, 3), pick(1, 2));
            if (n % 2 == 0)
                for (int mode : {7, 8}) one(dbl, n, mode, 0, pick(0, 5), pick(0, 5), pick(1, 19), pick(1, 3), pick(1, 2));
        }
    // few lines per tile and the largest tile
    for (bool dbl : {false, true})
        for (int n : {1000, 1021, 1331, 2187, 2400, 4913, 4999, 5000}) one(dbl, n, hmi::kModeC2C, 0, 0, pick(2, 5), 3, 1, 1);
    // a large prime beside other factors: no less exact than smooth stages and one plain direct sum of the
    // prime's terms (its relative error on random lines, measured on the GPU)
    const struct { bool dbl; int n; double plain; } exact[] = {
        {true, 213, 3.13e-16}, {true, 268, 3.01e-16}, {true, 402, 3.16e-16}, {true, 404, 3.60e-16}, {true, 536, 3.11e-16},
        {false, 268, 1.63e-7}, {false, 670, 1.70e-7}, {false, 2010, 1.78e-7}, {false, 4984, 1.97e-07}};
    // odd lengths with several stages of radix 9: no less exact than with stages of radix 3
    const struct { bool dbl; int n; double plain; } nines[] = {
        {false, 81, 1.010e-7}, {false, 729, 1.282e-7}, {true, 81, 2.032e-16}};
    for (const auto &e : nines) one(e.dbl, e.n, hmi::kModeC2C, 0, 0, 2, 80000 / e.n, 1, 1, e.plain);
    for (const auto &e : exact) one(e.dbl, e.n, hmi::kModeC2C, 0, 0, 2, e.n < 1000 ? 40 : 5, 1, 1, e.plain);
    std::printf("%s %d\n", fails ? "failed" : "ok", cases);
    return fails ? 1 : 0;
}
