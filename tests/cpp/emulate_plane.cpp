// Runs the fused two-axis pass (csrc/hmi_plane.h) on the CPU over many plane shapes against a direct
// transform in long double; arrays and LDS end where the pass may last touch them.
#include <algorithm>
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

template <typename R> bool run_case(int n0, int n1, int nplanes, bool inverse, int product, unsigned seed) {
    const bool dbl = sizeof(R) == 8;
    // as a launch does: planned for the planes of one transform, grouped for those of the batch
    hmi::plane_config c = hmi::make_plane(n0, n1, 1 + nplanes / 8, dbl);
    if (c.ok) hmi::group_planes(c, nplanes, dbl);
    const std::string what = std::to_string(n0) + " x " + std::to_string(n1) + " planes " + std::to_string(nplanes) +
                             (dbl ? " f64" : " f32") + (inverse ? " inverse" : "") + " product " + std::to_string(product);
    if (!c.ok) { std::printf("FAIL %s: no plan\n", what.c_str()); return false; }
    const size_t count = (size_t)n0 * n1 * nplanes;
    std::mt19937 rng(seed);
    std::uniform_real_distribution<double> d(-1, 1);
    R *in = new R[2 * count], *out = new R[2 * count], *mul = new R[2 * count];
    for (size_t i = 0; i < 2 * count; i++) { in[i] = (R)d(rng); mul[i] = (R)d(rng); out[i] = 77; }
    const auto t0 = hmi::mixed_table(c.args.g0, dbl, 1), t1 = hmi::mixed_table(c.args.g1, dbl, 1);
    unsigned char *d0 = new unsigned char[t0.size()], *d1 = new unsigned char[t1.size()];
    std::copy(t0.begin(), t0.end(), d0);
    std::copy(t1.begin(), t1.end(), d1);
    hmi::plane_args a = c.args;
    a.in = in; a.out = out; a.tw0 = d0; a.tw1 = d1;
    a.mul = product == 0 ? nullptr : product == 1 ? (const void *)mul : in;
    a.conj = inverse; a.scale = 0.5;
    auto kernel = hmi::plane_builds<R>::choose(a);
    emulate::run_blocks(c.nblocks, c.threads, hmi::smem_raw, sizeof(hmi::smem_raw), c.lds,
                        [&] { kernel(a); });
    const long double pi = 3.141592653589793238462643383279502884L;
    auto root = [&](long long t, long long n) {
        const long double x = 2 * pi * (t % n) / n;
        return cld(cosl(x), inverse ? sinl(x) : -sinl(x));
    };
    std::vector<cld> w0(n0), w1(n1);
    for (int t = 0; t < n0; t++) w0[t] = root(t, n0);
    for (int t = 0; t < n1; t++) w1[t] = root(t, n1);
    long double num = 0, den = 0;
    for (int pl = 0; pl < nplanes; pl++) {
        std::vector<cld> x((size_t)n0 * n1), y(x.size());
        for (size_t i = 0; i < x.size(); i++) {
            const size_t at = (size_t)pl * n0 * n1 + i;
            x[i] = cld(in[2 * at], in[2 * at + 1]);
            if (product) x[i] *= product == 1 ? cld(mul[2 * at], mul[2 * at + 1]) : x[i];
        }
        for (int r = 0; r < n1; r++)
            for (int k = 0; k < n0; k++) {
                cld s = 0;
                for (int j = 0; j < n0; j++) s += x[(size_t)r * n0 + j] * w0[(long long)j * k % n0];
                y[(size_t)r * n0 + k] = s;
            }
        for (int k = 0; k < n1; k++)
            for (int col = 0; col < n0; col++) {
                cld s = 0;
                for (int j = 0; j < n1; j++) s += y[(size_t)j * n0 + col] * w1[(long long)j * k % n1];
                s *= 0.5L;
                const size_t at = ((size_t)pl * n1 + k) * n0 + col;
                num += std::norm(cld(out[2 * at], out[2 * at + 1]) - s);
                den += std::norm(s);
            }
    }
    delete[] in; delete[] out; delete[] mul; delete[] d0; delete[] d1;
    const long double err = sqrtl(num / den), tol = dbl ? 2e-15L : 1e-6L;
    if (!(err <= tol)) { std::printf("FAIL %s: %g of the tolerance\n", what.c_str(), (double)(err / tol)); return false; }
    return true;
}

// The grid of any launch stays below 2^32 threads, and many small planes share blocks: nplanes as
// many as the limit on lines of a pass, or the memory of one GPU, allows.
int check_grids() {
    int fails = 0;
    for (bool dbl : {false, true})
        for (int n0 = 2; n0 <= hmi::kPlaneMaxSide; n0++)
            for (int n1 : {2, 3, 4, 5, 8, 10, 16, 24, 27, 45, 64, 77, 100, 128, 200, 256}) {
                hmi::plane_config c = hmi::make_plane(n0, n1, 1, dbl);
                if (!c.ok) continue;
                const long long elem = dbl ? 16 : 8, most = std::min(0x7fffffffLL / std::max(n0, n1), (288LL << 30) / (elem * n0 * n1));
                for (long long nplanes : {1LL, 255LL, 4096LL * n0, most}) {
                    if (nplanes > most) continue;
                    hmi::group_planes(c, nplanes, dbl);
                    const long long bytes = (long long)c.args.ps * elem;
                    const bool bad = c.nblocks * c.threads > 0xffffffffLL || c.threads < 64 || c.threads % 64 ||
                                     c.nblocks * c.args.planes < nplanes || (c.nblocks - 1) * c.args.planes >= nplanes ||
                                     c.lds != (size_t)(c.args.planes * bytes) ||
                                     (nplanes >= 1LL << 20 && 2 * (c.args.planes + 1) * bytes <= hmi::kPlaneTile);
                    if (bad) std::printf("FAIL grid %d x %d planes %lld\n", n0, n1, nplanes), fails++;
                }
            }
    for (int threads : {64, 128, 320, 512})
        for (long long nblocks : {1LL, 1LL << 22, 1LL << 23, (1LL << 26) - 1}) {
            const int t = hmi::launch_threads(threads, nblocks);
            const bool most = t == threads || nblocks * (t + 64) > 0xffffffffLL;
            if (t < 64 || t % 64 || t > threads || nblocks * t > 0xffffffffLL || !most)
                std::printf("FAIL threads %d blocks %lld\n", threads, nblocks), fails++;
        }
    return fails;
}

int main(int argc, char **argv) {
    const int share = argc > 1 ? std::atoi(argv[1]) : 0, shares = argc > 2 ? std::atoi(argv[2]) : 1;
    std::mt19937 rng(3);
    int cases = 0, fails = share == 0 ? check_grids() : 0, at = 0;
    auto one = [&](bool dbl, int n0, int n1, int nplanes) {
        const bool inverse = rng() & 1;
        const int product = (int)(rng() % 4) % 3;
        if (at++ % shares != share) return;
        cases++;
        fails += (dbl ? run_case<double>(n0, n1, nplanes, inverse, product, at) : run_case<float>(n0, n1, nplanes, inverse, product, at)) ? 0 : 1;
    };
    const int sides[] = {2, 3, 5, 8, 11, 12, 15, 16, 22, 27, 32, 36, 45, 49, 60, 64, 77, 90, 96, 100, 128, 169, 200, 225, 256};
    for (bool dbl : {false, true})
        for (int k = 0; k < 120; k++) {
            const int n0 = sides[rng() % 25], n1 = sides[rng() % 25];
            if ((n0 | 1) * n1 * (dbl ? 16 : 8) > hmi::kPlaneBytes) continue;
            one(dbl, n0, n1, 1 + (int)(rng() % 4));
        }
    // several planes per block and a partial last group
    for (bool dbl : {false, true})
        for (int n : {4, 7, 12, 20}) one(dbl, n, n + 1, 1030 + n);
    std::printf("%s %d\n", fails ? "failed" : "ok", cases);
    return fails ? 1 : 0;
}
