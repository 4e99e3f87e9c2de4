// Host check of the window order's index arithmetic (win_device.cuh): for points
// on and around every kind of place (random, exact cells, the ends of [-1, nf + 1],
// NaN), each point's window, shifts and offset must describe exactly the ns taps
// of the per-point kernels: the same grid cells after the wrap, the same distances,
// all inside the window; keys inside [0, nkeys), every window cell inside the grid.
// The ranges of a weighted order must tile it.  Built with AddressSanitizer and
// UndefinedBehaviorSanitizer.
//
// usage: win_check type dim ns nf0 nf1 nf2
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>
#include <vector>

#include "../../cufinufft_amd/csrc/win_device.cuh"

static int g_fail = 0;
#define CHECK(c, ...)                                   \
    do {                                                \
        if (!(c)) {                                     \
            if (g_fail < 20) std::printf(__VA_ARGS__);  \
            ++g_fail;                                   \
        }                                               \
    } while (0)

template <typename T, int DIM>
static void check_points(const cfa::WinGeom &w, int type, int ns, const int *nf)
{
    std::mt19937_64 rng(5);
    const int F = cfa::win_first(ns);
    // cells a window reads or writes along each axis
    int cells[3] = {16, 16, 1};
    if (DIM == 3) {
        cells[2] = type == 1 ? ns : 2 * cfa::win_interp_half(ns);
        if (type == 2) cells[1] = cells[2];
    }
    for (int it = 0; it < 200000; ++it) {
        int kw[3] = {0, 0, 0};
        for (int d = 0; d < DIM; ++d) {
            const int n = nf[d];
            std::uniform_real_distribution<double> u(-1.0, n + 1.0);
            double v = u(rng);
            switch (it % 8) {
            case 1: v = std::floor(v); break;
            case 2: v = std::nextafter(std::floor(v), 1e9); break;
            case 3: v = std::nextafter(std::floor(v), -1e9); break;
            case 4: v = (it / 8) % 2 ? -1.0 : n + 1.0; break;
            case 5: v = std::floor(v) + 0.5; break;
            case 6: v = (it / 8) % 2 ? 0.0 : (double)n; break;
            case 7:
                if (it % 64 == 7) v = std::numeric_limits<double>::quiet_NaN();
                break;
            }
            v = cfa::tap_pos(v, n);
            T f;
            const int uu = cfa::win_place<T>(v, ns, f);
            const int k = uu / w.S[d], sh = uu - k * w.S[d];
            kw[d] = k;
            CHECK(uu >= 0 && k >= 0 && k < w.nw[d], "axis %d v %.17g: window %d of %d\n", d, v, k,
                  w.nw[d]);
            CHECK(sh + ns <= cells[d], "axis %d v %.17g: taps end at %d of %d\n", d, v, sh + ns,
                  cells[d]);
            CHECK(f >= T(0) && f <= T(1), "axis %d v %.17g: offset %g\n", d, v, (double)f);
            const int start = (int)std::ceil(v - 0.5 * ns);
            for (int i = 0; i < ns; ++i) {
                const int cell = cfa::win_wrap(k * w.S[d] - F + sh + i, n);
                CHECK(cell == cfa::wrapmod(start + i, n), "axis %d v %.17g tap %d: cell %d\n", d, v,
                      i, cell);
                const double x = (double)f + (i - 0.5 * ns), want = (double)(start + i) - v;
                CHECK(std::fabs(x - want) <= (sizeof(T) == 4 ? 3.1e-8 : 3e-13),
                      "axis %d v %.17g tap %d: distance %.17g, not %.17g\n", d, v, i, x, want);
            }
            for (int i = 0; i < cells[d]; ++i) {
                const int cell = cfa::win_wrap(k * w.S[d] - F + i, n);
                CHECK(cell >= 0 && cell < n, "axis %d window %d cell %d: %d of %d\n", d, k, i, cell,
                      n);
            }
        }
        const int key = cfa::win_key<DIM>(w, kw);
        CHECK(key >= 0 && key < w.nkeys, "key %d of %d\n", key, w.nkeys);
    }
}

// Ranges over random counts: ascending, from 0 to M, none far above its share.
static void check_ranges(unsigned seed)
{
    std::mt19937_64 rng(seed);
    const int nkeys = 1 + (int)(rng() % 3000), ranges = 1 + (int)(rng() % 700);
    std::vector<int> start(nkeys + 1), used(nkeys + 1);
    long long M = 0;
    int ne = 0;
    for (int k = 0; k < nkeys; ++k) {
        const int kind = (int)(rng() % 4);
        const int n = kind == 0 ? 0 : (kind == 1 ? (int)(rng() % 5) : (int)(rng() % 400));
        start[k] = (int)M;
        used[k] = ne;
        M += n;
        ne += n > 0;
    }
    start[nkeys] = (int)M;
    used[nkeys] = ne;
    if (M == 0) return;
    const long long total = M + (long long)cfa::kWinKeyWeight * ne;
    int prev = 0;
    for (int r = 0; r <= ranges; ++r) {
        const int p = cfa::win_range_start(start.data(), used.data(), nkeys, (int)M, r, ranges);
        CHECK(p >= prev && p <= M, "range %d starts at %d after %d\n", r, p, prev);
        CHECK(r > 0 || p == 0, "first range starts at %d\n", p);
        CHECK(r < ranges || p == M, "last range ends at %d of %lld\n", p, M);
        CHECK(r == 0 || p - prev <= total / ranges + 1, "range %d holds %d points\n", r, p - prev);
        prev = p;
    }
}

int main(int argc, char **argv)
{
    if (argc != 7) return 2;
    const int type = std::atoi(argv[1]), dim = std::atoi(argv[2]), ns = std::atoi(argv[3]);
    const int nf[3] = {std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6])};
    cfa::WinGeom w;
    CHECK(cfa::win_windows(type, dim, ns, nf, w), "no windows for this grid\n");
    if (!g_fail) {
        if (dim == 2) {
            check_points<float, 2>(w, type, ns, nf);
            check_points<double, 2>(w, type, ns, nf);
        } else {
            check_points<float, 3>(w, type, ns, nf);
            check_points<double, 3>(w, type, ns, nf);
        }
        for (unsigned s = 1; s <= 200; ++s) check_ranges(s);
    }
    std::printf(g_fail ? "FAILED: %d checks\n" : "OK: %d failed checks\n", g_fail);
    return g_fail ? 1 : 0;
}
