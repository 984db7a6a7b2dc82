// Radix plans, tile shapes and twiddle tables of the runtime-length pass (fft_generic).
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <limits>
#include <stdexcept>

#include "hmi_plan.h"

namespace hmi {

namespace {

constexpr int kRadices[] = {16, 15, 14, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// Real operations of the radix-r butterfly (additions and multiply-adds).
double butterfly_ops(int r) {
    switch (r) {
        case 2: return 4;
        case 3: return 16;
        case 4: return 16;
        case 5: return 40;
        case 6: return 44;
        case 7: return 72;
        case 8: return 64;
        case 9: return 120;
        case 10: return 100;
        case 11: return 150;
        case 12: return 112;
        case 13: return 210;
        case 14: return 172;
        case 15: return 200;
        default: return 170;
    }
}

// Cost per element of one stage: its butterfly and twiddles, and a fixed part for the LDS exchange
// and the index work.
double stage_cost(int r, bool dbl) {
    // radices past the light build's cost resident waves
    return 14.0 + (butterfly_ops(r) + 6.0 * (r - 1)) / r + (r > kLightRadix ? (dbl ? 4.0 : 2.0) : 0.0);
}

void search(int n, int top, bool dbl, std::vector<int> &cur, double cost, std::vector<int> &best, double &best_cost) {
    if (cost >= best_cost) return;
    if (n == 1) {
        best = cur;
        best_cost = cost;
        return;
    }
    if ((int)cur.size() == kMixedStages) return;
    for (int r : kRadices)
        if (r <= top && n % r == 0) {
            cur.push_back(r);
            search(n / r, r, dbl, cur, cost + stage_cost(r, dbl), best, best_cost);
            cur.pop_back();
        }
}

bool is_prime(int p) {
    for (int d = 3; d * d <= p; d += 2)
        if (p % d == 0) return false;
    return true;
}

// Largest prime factor that runs as a direct stage in a length of `cofactor` times that prime.  The error
// of a direct stage grows with its prime alone, that of a chirp convolution with the whole length, whose
// transforms it needs twice.  Relative errors against long double, direct stage / chirp / one direct sum
// without shared pairs:
//   complex<double>  67 points 2.11e-16 / 2.56e-16 / 2.88e-16, 4 x 67 2.32 / 3.45 / 3.01, 6 x 67 2.42 / 3.80 / 3.16
//   complex<float>   30 x 67 1.41e-7 / 1.91e-7 / 1.78e-7, 4 x 101 1.45 / 1.62 / 1.93
// A prime alone is direct up to 61 (67 points 1.0 to 1.2 times the chirp's time, 127 points 1.5 to 2.6), and
// with a cofactor up to where the chirp would be less exact than that plain direct sum (complex<double>
// 3 x 71 ... 30 x 107, complex<float> 4 x 67, 60 x 83, 56 x 89; of all lengths of one tile): there the direct
// stage takes 0.5 to 1.4 times the chirp's time.
int max_direct(int cofactor, bool dbl) {
    if (dbl) return cofactor < 3 ? 61 : 107;
    return cofactor < 4 ? 61 : cofactor < 24 ? 73 : cofactor < 48 ? 83 : 107;
}

fast_div make_div(unsigned d) {
    unsigned s = 0;
    while ((1ull << s) < d) s++;
    const unsigned long long p = 1ull << (31 + s);
    return {(unsigned)((p + d - 1) / d), s};
}

// LDS cycles of the last stage's reads when lanes walk the FFT axis: lane u reads position u's block,
// k_0 m_0 pitch + k_0 pad + (rest); the LDS serves `group` lanes at once from
// `group` element slots (32 of 8 bytes over its 64 banks, 16 of 16 bytes).
int read_conflicts(const mixed_plan &g, int pad, int group) {
    const int nb = g.n / g.last, lanes = std::min(nb, 2 * group);
    int total = 0;
    for (int u0 = 0; u0 < lanes; u0 += group) {
        int used[32] = {}, worst = 0;
        for (int u = u0; u < std::min(u0 + group, nb); u++) {
            int t = u, pos = 0, k0 = 0, span = g.n;
            for (int s = 0; s + 1 < g.nst; s++) {
                span /= g.radix[s];
                const int d = t % g.radix[s];
                t /= g.radix[s];
                if (s == 0) k0 = d;
                pos += d * span;
            }
            worst = std::max(worst, ++used[(pos * g.pitch + k0 * pad) % group]);
        }
        total += worst;
    }
    return total;
}

}  // namespace

std::vector<int> mixed_radices(int n, bool dbl) {
    int largest = n;  // prime factor
    for (int p = 2; p * p <= largest; p++)
        while (largest % p == 0 && largest > p) largest /= p;
    const int top = max_direct(n / largest, dbl);
    std::vector<int> direct;
    for (int p = 17; p <= top; p += 2)
        while (is_prime(p) && n % p == 0) {
            direct.push_back(p);
            n /= p;
        }
    std::vector<int> cur, best;
    double cost = std::numeric_limits<double>::infinity();
    search(n, 16, dbl, cur, 0.0, best, cost);
    if (best.size() > 2) {
        // the largest radix first and the next one last: the stages on global memory keep the most
        // accesses in flight
        std::rotate(best.begin() + 1, best.begin() + 2, best.end());
    }
    if (n > 1 && best.empty()) return best;
    best.insert(best.end(), direct.begin(), direct.end());
    return best;
}

int chirp_length(int n, bool dbl) {
    // the cheapest transform of at least 2 n - 1 points that fits the LDS
    const int most = kGenericMaxLds / (dbl ? 16 : 8);
    int best = 0;
    double cost = std::numeric_limits<double>::infinity();
    for (int m = 2 * n - 1; m <= std::min(most, 3 * n + 64); m++) {
        int rest = m;
        for (int p : {2, 3, 5, 7, 11, 13})
            while (rest % p == 0) rest /= p;
        if (rest != 1) continue;
        double c = 0.0;
        const std::vector<int> rad = mixed_radices(m, dbl);
        for (int r : rad) c += stage_cost(r, dbl);
        if (rad.size() > 1 && c * m < cost) {
            cost = c * m;
            best = m;
        }
    }
    return best;
}

namespace {
// Lines per tile (log2) of a launch of nlines lines, l2 the full tile's: few lines take smaller tiles on more
// CUs, down to 64-byte chunks of a side that walks the column axis.
int tile_lines(const mixed_plan &g, int l2, bool across, bool dbl, long long nlines) {
    const int least = across ? (dbl ? 2 : 3) : 0;
    while (l2 > least && (nlines >> l2) < kFewBlocks) l2--;
    return l2;
}
}  // namespace

mixed_tiles::mixed_tiles(int n, bool dbl, bool copy, bool load_across, bool store_across, int tail)
    : n_(n), tail_(tail), dbl_(dbl), copy_(copy), load_(load_across), store_(store_across) {
    full_ = make_mixed(n, dbl, copy, load_across, store_across, 0, tail);
}

const mixed_config &mixed_tiles::of(long long nlines) {
    const int l2 = tile_lines(full_.plan, full_.plan.log2t, load_ || store_, dbl_, nlines);
    if (l2 == full_.plan.log2t) return full_;
    std::lock_guard<std::mutex> lock(mtx_);
    std::unique_ptr<mixed_config> &c = smaller_[l2];
    if (!c) c = std::make_unique<mixed_config>(make_mixed(n_, dbl_, copy_, load_, store_, nlines, tail_));
    return *c;
}

mixed_config make_mixed(int n, bool dbl, bool copy, bool load_across, bool store_across, long long nlines,
                        int tail) {
    mixed_config c{};
    mixed_plan &g = c.plan;
    std::vector<int> rad = (copy || n == 1) ? std::vector<int>{} : mixed_radices(n, dbl);
    const long long elem = dbl ? 16 : 8;
    g.len = n;
    g.chirp = (copy || n == 1 || !rad.empty()) ? 0 : 1;
    if (g.chirp) {
        n = chirp_length(n, dbl);
        if (n) rad = mixed_radices(n, dbl);
    }
    c.ok = n > 0 && (int)rad.size() <= kMixedStages;
    if (!c.ok) return c;
    g.n = n;
    for (int r : rad) g.direct += r > 16 ? 1 : 0;
    // Odd lengths with several stages of radix 9 and 3 meet the rounding errors of w9 in each of them:
    // relative error on random lines, stages of radix 3 / of radix 9 / of radix 9 with exact constants,
    // complex<float> 81 points 1.010e-7 / 1.027e-7 / 0.978e-7, 729 1.282 / 1.312 / 1.240, complex<double> 567
    // points 2.371e-16 / 2.416 / 2.332.  (A build of its own: the same choice inside the others' stages costs
    // up to 3 % of any pass.  Even lengths are more exact than stages of radix 3 and 8 as it is, 72 points 0.93.)
    g.set = kSetLight;
    for (int r : rad)
        if (r > kLightRadix && r <= 16) g.set = kSetFull;
    if (n % 2 == 1 && n % 9 == 0 && n >= 81 && g.set == kSetLight && !g.direct && !g.chirp) g.set = kSetOdd;
    const int bufs = g.direct > 1 ? 2 : 1;
    g.nst = (int)rad.size();
    for (int s = 0; s < kMixedStages; s++) {
        g.radix[s] = s < g.nst ? rad[s] : 1;
        g.by_r[s] = make_div(g.radix[s]);
        if (s == 0) g.m0 = n / g.radix[0];

    }
    g.last = g.nst ? rad.back() : 1;
    g.by_m0 = make_div(g.m0);
    g.by_last = make_div(n / g.last);
    g.by_n = make_div(n);
    g.postoff = mixed_post_offset(rad);
    g.chirpoff = g.postoff + tail;
    int at = g.chirpoff;  // (a plan has direct stages or a chirp)
    for (int s = 0; s < g.nst; s++)
        if (rad[s] > 16) {
            if (s == 0) g.root0 = at;
            if (s + 1 == g.nst) g.root_last = at;
            at += rad[s];
        }
    // Lines per tile: about kMixedTile bytes, and in any case the 128-byte column chunk where a side
    // walks the column axis or where that keeps two blocks per CU.
    const bool across = load_across || store_across;
    const bool walk = !load_across || !store_across;  // a side on which lanes walk the FFT axis
    auto bytes = [&](int t) {
        const long long pitch = walk && t > 1 ? t + 1 : t;
        return bufs * ((long long)n * pitch + (g.direct ? 0 : 32LL * g.radix[0])) * elem;
    };
    int l2 = 0;
    while (l2 < 6 && (n * elem << (l2 + 1)) <= kMixedTile) l2++;
    while ((elem << l2) < 128 && bytes(2 << l2) <= (across ? kGenericMaxLds : kGenericMaxLds / 2)) l2++;
    if (nlines > 0) l2 = tile_lines(g, l2, across, dbl, nlines);
    g.log2t = l2;
    const int T = 1 << l2;
    g.pitch = walk && T > 1 ? T + 1 : T;
    g.pad = 0;
    if (g.nst > 1 && !g.chirp && !g.direct && !store_across) {
        int best = std::numeric_limits<int>::max();
        for (int pad = 0; pad < (dbl ? 16 : 32); pad++) {
            const int k = read_conflicts(g, pad, dbl ? 16 : 32);
            if (k < best && ((long long)n * g.pitch + (long long)(g.radix[0] - 1) * pad) * elem <= kGenericMaxLds) {
                best = k;
                g.pad = pad;
            }
        }
    }
    c.lds = (size_t)(bufs * ((long long)n * g.pitch + (long long)(g.radix[0] - 1) * g.pad) * elem);
    // Threads: the rounds a block spends in each stage (the ones on global memory weigh more) over
    // the blocks a CU holds, and the idle lanes of the last rounds.  Blocks of more than four waves
    // count as whole sets of four, one for each SIMD: 320 points complex<double>, 8 lines, contiguous:
    // 256 threads 5.36 TB/s, 320 4.54, 512 5.22; 400 points: 256 4.62, 320 4.73, 512 5.25.
    bool light = true;
    for (int r : rad) light = light && (r <= kLightRadix || r > 16);
    const int by_lds = (int)(kGenericMaxLds / std::max<long long>(1, (long long)c.lds));
    const int waves = 4 * (dbl ? (light ? 4 : 3) : (light ? 8 : 5));
    double best = std::numeric_limits<double>::infinity();
    for (int th = 64; th <= kMixedThreads; th += 64) {
        if (th % T) continue;
        const int held = th <= 256 ? th : (th + 255) / 256 * 256;
        double rounds = 0.0, lanes = 0.0, ideal = 0.0;
        const int stages = std::max(1, g.nst);
        for (int s = 0; s < stages; s++) {
            const int r = g.nst ? rad[s] : 1;
            // (a direct stage: four outputs per unit)
            const long long units = r > 16 ? (long long)T * (n / r) * ((r + 3) / 4) : (long long)T * n / r;
            const double w = r > 16 ? 12.0 * r : r * stage_cost(r, dbl);
            const double k = (double)((units + th - 1) / th);
            // (a chirp pass runs each stage forth and back)
            rounds += k * (g.chirp ? (s == 0 ? 5.0 : 2.0) : (s == 0 ? 3.0 : s + 1 == stages ? 2.0 : 1.0));
            lanes += w * k * held;
            ideal += w * (double)units;
        }
        const int resident = std::max(1, std::min({by_lds, waves * 64 / held, 16}));
        const double cost = rounds / resident * (0.5 + 0.5 * lanes / ideal);
        if (cost < best - 1e-9) {
            best = cost;
            c.threads = th;
        }
    }
    return c;
}

plane_config make_plane(int n0, int n1, long long nplanes, bool dbl) {
    plane_config c{};
    if (n0 < 2 || n1 < 2 || n0 > kPlaneMaxSide || n1 > kPlaneMaxSide) return c;
    const long long elem = dbl ? 16 : 8, rp = n0 | 1, ps = rp * n1;
    if (ps * elem > kPlaneBytes) return c;
    // (only the radix plans are used: the orientation with the least work)
    const mixed_config c0 = make_mixed(n0, dbl, false, true, true, 0, 0), c1 = make_mixed(n1, dbl, false, true, true, 0, 0);
    if (!c0.ok || !c1.ok) return c;
    plane_args &a = c.args;
    a.g0 = c0.plan;
    a.g1 = c1.plan;
    if (a.g0.chirp || a.g0.direct || a.g1.chirp || a.g1.direct) return c;
    a.n0 = n0;
    a.n1 = n1;
    a.rp = (int)rp;
    a.ps = (int)ps;
    a.by_n0 = make_div((unsigned)n0);
    c.ok = true;
    group_planes(c, nplanes, dbl);
    return c;
}

void group_planes(plane_config &c, long long nplanes, bool dbl) {
    plane_args &a = c.args;
    const long long elem = dbl ? 16 : 8;
    // planes per block: up to kPlaneTile bytes, as long as the launch keeps kFewBlocks blocks
    int planes = 1;
    while (2 * planes * a.ps * elem <= kPlaneTile && nplanes / (2 * planes) >= kFewBlocks) planes *= 2;
    a.planes = planes;
    a.rows = (unsigned)(planes * a.n1);
    a.cols = (unsigned)(planes * a.n0);
    a.by_rows = make_div(a.rows);
    a.by_cols = make_div(a.cols);
    a.nplanes = (int)nplanes;
    c.lds = (size_t)(planes * a.ps * elem);
    c.nblocks = (nplanes + planes - 1) / planes;
    // threads: about one round of the smallest stage, whole sets of four waves above 256
    int top = 2;
    for (const mixed_plan *g : {&a.g0, &a.g1})
        for (int s = 0; s < g->nst; s++) top = std::max(top, g->radix[s]);
    const long long units = (long long)planes * a.n0 * a.n1 / top;
    c.threads = 64;
    while (c.threads < 256 && c.threads < units) c.threads += 64;
    if (units > 256 + 64) c.threads = kMixedThreads;
    c.threads = launch_threads(c.threads, c.nblocks);
}

// A plane of about 64 KiB or more has a CU to itself, and a launch of few of them leaves most CUs idle
// while one pass per axis spreads their lines, the sooner the faster those passes are: the tiles of powers of
// two against the others.  One pass for both axes / one pass for each, us of a whole transform:
//   complex<float>   128 x 128 x 1 12.7 / 8.8, x 64 22.3 / 21.3, x 128 25.2 / 27.5; 256 x 64 x 8 16.6 / 12.4
//                    200 x 100 x 1 17.5 / 8.7, x 32 24.4 / 18.8, x 128 32.9 / 34.4; 100 x 100 x 8 12.1 / 11.5, x 32 13.7 /
//                    13.8; 96 x 196 x 105 26.8 / 30.6; 112 x 112 x 3 13.5 / 18.2; 80 x 80 (51 KiB) x 1 7.1 / 9.6
//   complex<double>  64 x 64 (65 KiB) x 4 10.5 / 10.4, x 8 10.6 / 10.9; 128 x 32 x 4 13.5 / 12.2; 32 x 32 x 1 5.7 / 7.1
//                    100 x 100 x 8 16.4 / 12.7, x 32 19.5 / 18.8, x 64 23.3 / 25.0; 80 x 80 x 2 13.3 / 11.6, x 32 15.1 / 15.7
long long min_planes(int n0, int n1, bool dbl) {
    const long long above = (long long)(n0 | 1) * n1 - (dbl ? 3072 : 8192);  // 48 and 64 KiB
    const bool powers = (n0 & (n0 - 1)) == 0 && (n1 & (n1 - 1)) == 0;
    return above <= 0 ? 1 : 1 + above / ((dbl ? 128 : 96) * (powers ? 1 : 4));
}

int launch_threads(int threads, long long nblocks) {
    while (threads > 64 && nblocks * threads > 0xffffffffLL) threads -= 64;
    return threads;
}

fused_lists make_fused_lists(const std::vector<batch_xform> &xf, const std::vector<int> &lengths, bool dbl) {
    fused_lists f;
    const long long elem = dbl ? 16 : 8;
    // radix plans and tables (no plan: one point, or a prime factor above 13)
    for (int n : lengths) {
        mixed_plan g{};
        f.offset.push_back((int)f.table.size());
        if (n > 1 && 2 * n * elem <= kGenericMaxLds) g = make_mixed(n, dbl, false, true, true, 0, 0).plan;
        if (g.chirp || g.direct) g = mixed_plan{};
        if (g.n > 1) {
            const std::vector<unsigned char> t = mixed_table(g, dbl, 1);
            f.table.insert(f.table.end(), t.begin(), t.end());
        }
        f.plans.push_back(g);
    }
    const size_t count = xf.size();
    f.fused.resize(count);
    f.in_xy.resize(count);
    f.in_zc.resize(count);
    std::vector<long long> xy_elems(count, 0), zc_elems(count, 0);
    for (int i = 0; i < (int)count; i++) {
        const batch_xform &x = xf[i];
        const long long plane = (long long)xy_row_stride(x.n[0]) * x.n[1];  // LDS elements
        batch_fused &e = f.fused[i];
        if (f.plans[x.size_id[0]].n > 1 && f.plans[x.size_id[1]].n > 1 && plane * elem <= kGenericMaxLds) {
            int b = 0;
            while (plane * elem > kFusedLds[b]) b++;
            e.planes = (int)std::min<long long>(x.n[2], kFusedLds[b] / (plane * elem));
            e.by_rows = make_div((unsigned)(e.planes * x.n[1]));
            e.by_cols = make_div((unsigned)(e.planes * x.n[0]));
            e.by_n0 = make_div((unsigned)x.n[0]);
            f.in_xy[i] = true;
            xy_elems[i] = e.planes * plane;
            f.xy_lds[b] = std::max(f.xy_lds[b], (size_t)(xy_elems[i] * elem));
            for (long long t = 0; t * e.planes < x.n[2]; t++) f.xy[b].push_back({i, (int)t});
        }
        const long long cols = (long long)x.n[0] * x.n[1];
        if (f.plans[x.size_id[2]].n > 1 && elem * x.n[2] <= kFusedLds[0] && cols <= 0x7fffffffLL / 2) {
            e.width = (int)std::min<long long>(cols, kFusedLds[0] / (elem * x.n[2]));
            e.by_width = make_div((unsigned)e.width);
            f.in_zc[i] = true;
            zc_elems[i] = (long long)e.width * x.n[2];
            f.zc_lds = std::max(f.zc_lds, (size_t)(zc_elems[i] * elem));
            for (long long t = 0; t * e.width < cols; t++) f.zc.push_back({i, (int)t});
        }
    }
    // largest items first (the blocks take them in list order, so a launch ends on small ones)
    auto by_size = [](std::vector<batch_item> &v, const std::vector<long long> &e) {
        std::stable_sort(v.begin(), v.end(), [&](const batch_item &a, const batch_item &b) { return e[a.xform] > e[b.xform]; });
        if (v.size() > 0x7fffffffULL) throw std::runtime_error("batch work list too long");
    };
    for (std::vector<batch_item> &v : f.xy) by_size(v, xy_elems);
    by_size(f.zc, zc_elems);
    return f;
}

void mixed_launch_divs(mixed_plan &g, const pass_args &a) {
    g.by_ncol = make_div((unsigned)a.ncol);
    g.by_nb1 = make_div((unsigned)a.nb1);
}

int mixed_post_offset(const std::vector<int> &rad) {
    int off = 0;
    long long m = 1;
    for (int r : rad) m *= r;
    for (size_t s = 0; s + 1 < rad.size(); s++) {
        m /= rad[s];
        off += (int)m * (rad[s] - 1);
    }
    return off;
}

std::vector<unsigned char> mixed_table(const mixed_plan &g, bool dbl, long long tail_mod) {
    std::vector<unsigned char> out(kMixedHead, 0);
    using cld = std::complex<long double>;
    const long double pi = 3.141592653589793238462643383279502884L;
    auto root = [&](long long e, long long mod) {  // exp(-2 pi i e / mod)
        const long double ang = 2.0L * pi * (long double)(e % mod) / (long double)mod;
        return cld(cosl(ang), -sinl(ang));
    };
    auto push = [&](cld w) {
        const size_t at = out.size();
        if (dbl) {
            const double v[2] = {(double)w.real(), (double)w.imag()};
            out.resize(at + sizeof(v));
            std::memcpy(&out[at], v, sizeof(v));
        } else {
            const float v[2] = {(float)w.real(), (float)w.imag()};
            out.resize(at + sizeof(v));
            std::memcpy(&out[at], v, sizeof(v));
        }
    };
    // w_n^t, the upper half and (n even) the second quarter by symmetry
    std::vector<cld> wn(g.nst > 1 ? g.n : 0);
    for (int t = 0; t < (int)wn.size(); t++) {
        if (2 * t > g.n) wn[t] = std::conj(wn[g.n - t]);
        else if (g.n % 2 == 0 && 4 * t > g.n) wn[t] = -std::conj(wn[g.n / 2 - t]);
        else wn[t] = root(t, g.n);
    }
    long long len = g.n, off = 0, blocks = 1;
    for (int s = 0; s < g.nst; s++) {
        const int r = g.radix[s];
        const long long m = len / r;
        if (s > 0) {
            int root = g.chirpoff;
            for (int i = 0; i < s; i++) root += g.radix[i] > 16 ? g.radix[i] : 0;
            const mixed_stage st{r, (int)m, (int)off, make_div((unsigned)m), make_div((unsigned)blocks), root};
            std::memcpy(&out[(s - 1) * sizeof(mixed_stage)], &st, sizeof(st));
            blocks *= r;
        }
        if (m > 1) {
            for (long long j = 0; j < m; j++)
                for (int q = 1; q < r; q++) push(wn[j * q * (g.n / len)]);
            off += m * (r - 1);
        }
        len = m;
    }
    for (int k = 0; k < g.chirpoff - g.postoff; k++) push(root(k, tail_mod));
    for (int s = 0; s < g.nst; s++)
        for (int t = 0; g.radix[s] > 16 && t < g.radix[s]; t++) push(root(t, g.radix[s]));
    if (!g.chirp) return out;
    // c_j = exp(-i pi j^2 / len), and the transform of conj(c_{|j|}) / n by the stages of the plan
    std::vector<cld> b(g.n, cld(0, 0));
    for (long long j = 0; j < g.len; j++) {
        const cld c = root(j * j % (2LL * g.len), 2LL * g.len);
        push(c);
        b[j] = std::conj(c) / (long double)g.n;
        if (j > 0) b[g.n - j] = b[j];
    }
    len = g.n;
    for (int s = 0; s < g.nst; s++) {
        const int r = g.radix[s];
        const long long m = len / r;
        std::vector<cld> x(r);
        for (long long at = 0; at < g.n; at += len)
            for (long long j = 0; j < m; j++) {
                for (int p = 0; p < r; p++) x[p] = b[at + j + p * m];
                for (int q = 0; q < r; q++) {
                    cld y = 0;
                    for (int p = 0; p < r; p++) y += x[p] * wn[(long long)(p * q % r) * (g.n / r)];
                    b[at + j + q * m] = y * wn[j * q * (g.n / len)];
                }
            }
        len = m;
    }
    for (const cld &v : b) push(v);
    return out;
}

}  // namespace hmi
