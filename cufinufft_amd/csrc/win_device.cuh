// Window kernels: spreading and interpolation in 2D and 3D as small matrix
// products on the matrix cores (v_mfma_{f32_16x16x4f32, f64_16x16x4f64}).
//
// The ns^DIM taps of a point are an outer product of its axis weights, so the
// taps of many points that share a small window of the fine grid form a
// matrix product over the points:
//   spread:  win[(y, z), x] += sum_p (ky_p[y] kz_p[z]) * (c_p kx_p[x])
//   interp:  g[p, x] = sum_(y, z) (ky_p[y] kz_p[z]) * win[(y, z), x],
//            c_p = sum_x kx_p[x] g[p, x]
// with weights that are 0 outside a point's own taps.  A window is 16 cells
// wide in x, so it holds every point whose first tap lies in its first 17 - ns
// cells, and likewise along the other axes.  setpts orders the points by window
// (win_sort.hip); a wave then takes a range of that order and keeps a whole
// window in registers, so a tap costs neither an LDS operation nor a VALU
// instruction of its own.  No wave waits for another.
//
// What this replaces was bound by exactly those: the per-point spread issued
// two LDS atomics and six VALU instructions per tap (14 / 10 / 7 lanes per
// clock and CU for 32-bit, 64-bit integer and FP64 LDS adds), the per-point
// interp one LDS or L1 read and two FMAs per tap.
// Spread or interp alone, per-point -> window kernel: 3D FP32 type 1, ns 6, 1e8
// points on 512^3: 20.7 -> 6.9 ms; 3D FP64 type 2, ns 10, 1e7: 17.7 -> 2.5 ms;
// 2D FP64 type 2: 0.90 -> 0.30 ms (the rule of win_sort.hip has both sides at
// the edges of its range).
#pragma once
#include <utility>

#include "nufft_device.cuh"

namespace cfa {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<float> {
    using Acc = v4f;
    __device__ static __forceinline__ Acc mac(float a, float b, Acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<double> {
    using Acc = v4d;
    __device__ static __forceinline__ Acc mac(double a, double b, Acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};

// Row of the 16 x 16 result held by register r of the lanes of quarter q
// (the column is the lane within the quarter).
template <typename T>
__device__ __forceinline__ int mfma_row(int q, int r)
{
    return sizeof(T) == 4 ? 4 * q + r : q + 4 * r;
}

// Lane movement inside rows of 16 lanes (DPP); CTRL as in the ISA's dpp_ctrl:
// broadcast of lane n of each row (0x150 + n), rotation by n (0x120 + n), lane i from
// lane 7 - i of each 8, from lane i ^ 1 and i ^ 2.
constexpr int kDppBcast = 0x150, kDppRor = 0x120, kDppHalfMirror = 0x141, kDppQuadXor1 = 0xb1,
              kDppQuadXor2 = 0x4e;
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v)
{
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}

// f(0), ..., f(N - 1) with the index as a compile-time constant.
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// Square root of a in [2^-60, 1], within an ulp: the hardware reciprocal square
// root and Newton (Goldschmidt) steps with fused residuals.  The library's
// sqrt spends most of its instructions on ranges that cannot occur here.
__device__ __forceinline__ double win_sqrt(double a)
{
    const double y = __builtin_amdgcn_rsq(a);
    double s = a * y, h = 0.5 * y;
    const double r = fma(-h, s, 0.5);
    s = fma(s, r, s);
    h = fma(h, r, h);
    return fma(fma(-s, s, a), h, s);
}

// e^x in FP64 for |x| < 700: x = n ln 2 + r with |r| <= ln 2 / 2 (ln 2 in two
// parts), the Taylor polynomial of e^r to r^13 (its remainder is 4e-18), and a
// scaling by 2^n.
__device__ __forceinline__ double win_exp(double x)
{
    const double n = __builtin_rint(x * 1.4426950408889634);
    double r = fma(n, -0x1.62e42fefa3800p-1, x);
    r = fma(n, -0x1.ef35793c76730p-45, r);
    double p = 1.0 / 6227020800.0;
    p = fma(p, r, 1.0 / 479001600.0);
    p = fma(p, r, 1.0 / 39916800.0);
    p = fma(p, r, 1.0 / 3628800.0);
    p = fma(p, r, 1.0 / 362880.0);
    p = fma(p, r, 1.0 / 40320.0);
    p = fma(p, r, 1.0 / 5040.0);
    p = fma(p, r, 1.0 / 720.0);
    p = fma(p, r, 1.0 / 120.0);
    p = fma(p, r, 1.0 / 24.0);
    p = fma(p, r, 1.0 / 6.0);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return __builtin_ldexp(p, (int)n);
}

// Kernel value at offset x from the point, over its peak: phi(x) / e^beta; the
// callers put e^(DIM beta) back in FP64.  Outside the support the exponent is
// replaced by one that underflows to 0, so the code has no branch: many
// evaluations overlap.
//
// FP32 forms the exponent beta (sqrt(1 - t) - 1), t = c x^2, as -beta t /
// (1 + sqrt(1 - t)): its rounding is then relative to the exponent, which is
// small where the kernel is large, and the hardware square root and reciprocal
// (1 ulp) do.  The difference sqrt(..) - 1 itself carries half an ulp of 1, times
// beta (14 - 20) a relative error of ~3e-7 in every weight.
__device__ __forceinline__ float win_phi(float x, const KerParams<float> &k)
{
    const float t = k.c * x * x;
    const float s = __builtin_amdgcn_sqrtf(fmaxf(1.0f - t, 0.0f));
    const float w = t * __builtin_amdgcn_rcpf(1.0f + s);
    const float e = fmaf(-k.bl2e, w, -k.bl2e_lo * w);
    return __builtin_amdgcn_exp2f(fabsf(x) < k.hw ? e : -1000.0f);
}
__device__ __forceinline__ double win_phi(double x, const KerParams<double> &k)
{
    const double v = win_exp(k.beta * (win_sqrt(fmax(1.0 - k.c * x * x, 0x1p-60)) - 1.0));
    return fabs(x) < k.hw ? v : 0.0;
}

// Place of a point (position v, in [-1, nf + 1]) along one axis: its first tap
// is cell u - P - 1, u >= 0; f = first tap - position + ns/2 in [0, 1).  The weight
// of tap i is evaluated at f + (i - ns/2): i - ns/2 is exact, so a point keeps the
// precision of f, 2^-25 in FP32 (first tap - position itself would round at 2^-23).
// Window k of S first taps starts at cell k S - P - 1.
CFA_HD int win_first(int ns) { return (ns + 1) / 2 + 1; }
template <typename T>
CFA_HD int win_place(double v, int ns, T &f)
{
    const double s = ceil(v - 0.5 * ns);
    f = (T)((s - v) + 0.5 * ns);
    return (int)s + win_first(ns);
}
// Grid index of a cell in [-nf, 2 nf).
CFA_HD int win_wrap(int c, int n)
{
    c += c < 0 ? n : 0;
    return c - (c >= n ? n : 0);
}

// Key of a window.  3D: along z fastest, so a strip of windows along z is a run of
// the order; 2D spread: along y for the same reason; 2D interp: along x, as the bins
// (the window order of 3e6 FP64 points then takes 20 us less).
template <int DIM>
CFA_HD int win_key(const WinGeom &w, const int *k)
{
    if (DIM == 3) return (k[1] * w.nw[0] + k[0]) * w.nw[2] + k[2];
    return w.ystrips ? k[0] * w.nw[1] + k[1] : k[1] * w.nw[0] + k[0];
}

// Windows of a grid nf for transforms of the given type and width: S, nw, nkeys,
// ns.  false: a grid so small that a window's cells could wrap twice, or too
// many windows to count in ints.
inline bool win_windows(int type, int dim, int ns, const int *nf, WinGeom &w)
{
    w.ns = ns;
    w.ystrips = type == 1;
    w.S[0] = w.S[1] = 17 - ns;
    w.S[2] = 1;
    if (dim == 3 && type == 2) w.S[1] = w.S[2] = 2 * win_interp_half(ns) - ns + 1;
    double keys = 1;
    for (int d = 0; d < dim; ++d) {
        if (nf[d] < 24) return false;
        w.nw[d] = (nf[d] + 3) / w.S[d] + 1;
        keys *= w.nw[d];
    }
    if (keys > 1 << 27) return false;
    w.nkeys = (int)keys;
    return true;
}

// First point of range r of `ranges` ranges of equal weight, a point counting 1
// and a window that has points kWinKeyWeight (before its points).  start and used:
// points and windows with points before each key (used[nkeys]: all).
CFA_HD int win_range_start(const int *start, const int *used, int nkeys, int M, int r, int ranges)
{
    if (r >= ranges) return M;
    const long long total = M + (long long)kWinKeyWeight * used[nkeys];
    const long long w = total * r / ranges;
    int lo = 0, hi = nkeys - 1;  // last key whose weight starts at or before w
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] + (long long)kWinKeyWeight * used[mid] <= w) lo = mid; else hi = mid - 1;
    }
    const long long off = w - start[lo] - (long long)kWinKeyWeight * (used[lo] + 1);
    const int n = (lo + 1 < nkeys ? start[lo + 1] : M) - start[lo];
    return start[lo] + (int)(off > 0 ? (off < n ? off : n) : 0);
}

// Last key k with start[k] <= p (n keys): the key of point p.
__device__ __forceinline__ int win_key_of(const int *__restrict__ start, int n, int p)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= p) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// The keys of a wave's range, in order: 64 of their ends in the lanes.
struct WinKeys {
    int base, end;  // lane j: start[base + 1 + j]
    __device__ __forceinline__ void load(const WinPts &wp, int nkeys, int key)
    {
        base = key;
        end = wp.start[min(key + 1 + (int)(threadIdx.x & 63), nkeys)];
    }
    // Key of point p (>= the points asked for before).
    __device__ __forceinline__ int key_of(const WinPts &wp, int nkeys, int p)
    {
        unsigned long long m = __ballot(end > p);
        if (!m) {  // past these 64: a run of empty keys, or the next ones
            int k = base + 64;
            if (wp.start[min(k + 64, nkeys)] <= p) k = win_key_of(wp.start, nkeys, p);
            load(wp, nkeys, k);
            m = __ballot(end > p);
        }
        return base + __builtin_ctzll(m);
    }
    __device__ __forceinline__ int key_end(int key) const
    {
        return __builtin_amdgcn_readlane(end, key - base);
    }
};

// The weights of a point in LDS: its NS weights along x, a zero, those along y, a
// zero, and (3D) those along z.  A wave's lanes are points when the weights are
// evaluated, so each is evaluated once, and window cells when they are used: a
// cell reads the weight of tap (cell - first tap), or the zero behind the taps.
// The pitch is odd: the lanes' rows start in different banks.
template <typename T, int DIM, int NS>
struct WinRow {
    static constexpr int Y = NS + 1, Z = 2 * NS + 2;
    static constexpr int pitch = (DIM == 3 ? 3 * NS + 2 : 2 * NS + 2) | 1;
    // Index of tap i of an axis, of its zero where i is none of the NS taps.
    __device__ static __forceinline__ int tap(int i) { return (int)min((unsigned)i, (unsigned)NS); }
    __device__ static __forceinline__ void clear(T *rows, int n, int lane)
    {
        for (int k = lane; k < 2 * n; k += 64) rows[(k >> 1) * pitch + (k & 1 ? Y : 0) + NS] = T(0);
    }
    // Weights of an axis at f (see win_place), and the half h of the z weights.
    __device__ static __forceinline__ void axis(T *w, T f, const KerParams<T> &kp)
    {
#pragma unroll
        for (int i = 0; i < NS; ++i) w[i] = win_phi(f + ((T)i - T(0.5) * NS), kp);
    }
    __device__ static __forceinline__ void half(T *w, int h, T f, const KerParams<T> &kp)
    {
        constexpr int N = (NS + 1) / 2;
        w += h * N;
        f += (T)(h * N) - T(0.5) * NS;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const T v = win_phi(f + (T)i, kp);
            if (i + 1 < N || NS % 2 == 0 || h == 0) w[i] = v;
        }
    }
};

// ---------------------------------------------------------------------------
// Spread.  Windows of 16 x 16 cells in (x, y).  In 3D the points of a strip
// of windows come in order of their first z plane; the registers hold the ns
// planes that the current first plane reaches, plane z in slot z mod ns, and
// when the first plane moves on, the planes left behind go to the fine grid
// with global atomics.  So a strip writes every cell of its 16 x 16 column
// once: 256 / (17 - ns)^2 cells per grid cell (2.1 at ns 6), and no LDS tile, no
// common scale and no barrier is needed.  In 2D a window is one such plane, the
// strips run along y, row y is held in row slot y mod 16, and a window that follows
// its neighbour takes over the ns - 1 rows they share (17 - ns rows are written
// instead of 16); NT transforms share the weights.  Points come in window order, so strengths
// are gathered, 8 or 16 bytes of each 64-byte piece: batches are first packed point
// after point (k_win_pack; 32 coils of
// 2e6 points on 1024^2, ns 7, in batches of 8: 1.56 -> 1.27 ms with the shared rows).
//
// Bounds per 4 points and SIMD: 64 ns (FP32) or 128 ns clocks of the matrix cores
// in 3D, about 110 for the operands and 120 for the weights (which took 240 when
// each lane evaluated those of its own cell, zeros included: ns 6, 1e8 points on
// 512^3, 7.87 -> 6.85 ms), and the atomics, 1.9e10 64-byte pieces a second on the
// whole device (ns 7, 2e7 points on 384^3, 2.28 -> 1.93 ms by place()'s order).
template <typename T, int DIM, int NS, int NT>
struct WinSpread {
    using Acc = typename Mfma<T>::Acc;
    static constexpr int RB = DIM == 3 ? NS : 1;
    static constexpr int kBlock = 32;  // points staged at a time
    Acc ar[NT][RB], ai[NT][RB];
    unsigned row[4], col[2], src[2];  // see place()

    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int m = 0; m < RB; ++m) ar[t][m] = ai[t][m] = Acc{0, 0, 0, 0};
    }
    // The window's place (kx, ky): where in a plane the components go that
    // flush() hands this lane (row, col), and their index in a row (src).  Of a
    // row's 32 components lane i takes two, 16 apart, so that a 16-lane group
    // covers whole 64-byte pieces of memory but for the row's two ends: 3 pieces a
    // row in FP32 instead of 4, which is what the memory counts.  Quarter q takes
    // rows q + 4 r: grid rows have an even length, so 4 of them shift a row by whole
    // pieces.
    __device__ __forceinline__ void place(int kx, int ky, const BinGeom &g)
    {
        constexpr int S = 17 - NS, F = (NS + 1) / 2 + 1;
        const int lane = threadIdx.x & 63, q = lane >> 4, i16 = lane & 15;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = DIM == 2 ? (q + 4 * r - ky * S) & 15 : q + 4 * r;
            row[r] = 2u * (unsigned)(win_wrap(ky * S - F + j, g.nf[1]) * g.nf[0]);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            constexpr int cells = 32 / sizeof(T);  // cells of 64 bytes
            const int at = kx * S - F + (DIM == 2 ? q - F : ky * S - F + q) * g.nf[0];
            src[b] = (unsigned)(16 * b + i16 - 2 * (at & (cells - 1))) & 31;
            col[b] = 2u * (unsigned)win_wrap(kx * S - F + (int)(src[b] >> 1), g.nf[0]) + (src[b] & 1);
        }
    }
    // Points s .. e - 1 of the staged block (of one window); slot: that of their
    // first plane (3D) or of the window's first row (2D).
    __device__ __forceinline__ void accumulate(int s, int e, int slot, const T *rows,
                                               const unsigned *sh, const cpx<T> *cs)
    {
        using Row = WinRow<T, DIM, NS>;
        const int lane = threadIdx.x & 63, q = lane >> 4, i16 = lane & 15;
        // lane i of a row takes the x and y weights of cell i and the z weight
        // of slot i (any weight for i >= ns)
        const int zt = i16 - slot, z = Row::Z + min(zt < 0 ? zt + NS : zt, NS - 1);
        const int y = DIM == 2 ? zt & 15 : i16;
        // quarter q of the wave holds point b + q; groups of 4 start at multiples
        // of 4 of the block, so only a window's first and last are not full
        for (int b = s & ~3; b < e; b += 4) {
            const bool ok = b + q >= s && b + q < e;
            const int p = ok ? b + q : s;
            const T *row = rows + __umul24(p, Row::pitch);
            const unsigned u = sh[p];
            const T kx = row[ok ? Row::tap(i16 - (int)(u & 255)) : NS];
            const T ky = row[Row::Y + Row::tap(y - (int)(u >> 8 & 255))];
            T kz = T(0);
            if (DIM == 3) kz = row[z];
            T br[NT], bi[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const cpx<T> v = cs[NT * p + t];
                br[t] = v.x * kx;
                bi[t] = v.y * kx;
            }
            static_for<RB>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                const T a = DIM == 3 ? ky * dpp_mov<kDppBcast + m>(kz) : ky;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    ar[t][m] = Mfma<T>::mac(a, br[t], ar[t][m]);
                    ai[t][m] = Mfma<T>::mac(a, bi[t], ai[t][m]);
                }
            });
        }
    }
    // Adds plane slot m (2D: the first `rows` rows, from slot `slot` on) of every
    // transform to the grid and clears it; plane: the plane's first cell in transform
    // 0.  The lanes first trade places through
    // LDS (sc, 256 complex values of the wave), so that 16 lanes add the 16
    // components of 8 neighbouring cells: 1.9e11 adds per second against 1.2e11
    // for a lane per cell that adds its two components in turn (16 x 16 windows
    // every 10 cells of a 1024^2 FP32 grid).
    template <int m>
    __device__ __forceinline__ void flush(T *plane, long long tstride, int nt, cpx<T> *sc, int slot,
                                          int rows)
    {
        const int lane = threadIdx.x & 63, q = lane >> 4;
        // row q + 4 r: register r of quarter q in FP64, register q of quarter r in FP32
        const T *from = reinterpret_cast<const T *>(sc) + (lane >> 4) * (sizeof(T) == 4 ? 128 : 32);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (NT == 1 || t < nt) {
                T *p = plane + t * tstride;
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    cpx<T> v;
                    v.x = ar[t][m][r];
                    v.y = ai[t][m][r];
                    sc[64 * r + lane] = v;
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (DIM == 2 && ((q + 4 * r - slot) & 15) >= rows) continue;
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const T v = from[(sizeof(T) == 4 ? 32 : 128) * r + src[b]];
                        if (v != T(0)) gadd(p + (row[r] + col[b]), v);
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (DIM == 3 || ((mfma_row<T>(q, r) - slot) & 15) < rows)
                    ar[t][m][r] = ai[t][m][r] = T(0);
        }
    }
};

// Strengths of NT transforms, point after point: out[NT i + t] = c[t M + i].
template <typename T, int NT>
__global__ void __launch_bounds__(256)
k_win_pack(int M, int nt, const cpx<T> *__restrict__ c, cpx<T> *__restrict__ out)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= M) return;
    cpx<T> v[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        v[t].x = v[t].y = T(0);
        if (t < nt) v[t] = c[(long long)t * M + i];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) out[(long long)NT * i + t] = v[t];
}

// LDS of a wave.
template <typename T, int DIM, int NS, int NT>
struct WinSpreadLds {
    static constexpr int B = WinSpread<T, DIM, NS, NT>::kBlock;
    alignas(16) cpx<T> cs[B * NT];
    cpx<T> sc[256];
    unsigned sh[B];
    T rows[B * WinRow<T, DIM, NS>::pitch];
};

// One wave spreads range rng of a window order: nt <= NT transforms; point id's
// strength of transform t is c[t ct + id ci].
template <typename T, int DIM, int NS, int NT>
__device__ __forceinline__ void
win_spread_range(int rng, const WinPts &wp, const cpx<T> *__restrict__ c, long long ct, int ci,
                 T *__restrict__ ft, const BinGeom &g, const WinGeom &wg, const KerParams<T> &kp,
                 int nt, long long nftot, WinSpreadLds<T, DIM, NS, NT> &lds)
{
    constexpr int F = (NS + 1) / 2 + 1, S = 17 - NS;
    using Acc = WinSpread<T, DIM, NS, NT>;
    using Row = WinRow<T, DIM, NS>;
    constexpr int B = Acc::kBlock;
    const int lane = threadIdx.x & 63, h = lane >> 5, pl = lane & 31;
    T *rows = lds.rows;
    unsigned *sh = lds.sh;
    cpx<T> *cs = lds.cs, *sc = lds.sc;
    const T *x1 = static_cast<const T *>(wp.x);
    const int2 r0 = wp.range[rng];
    int p = r0.x;
    const int pe = wp.range[rng + 1].x;
    if (p >= pe) return;
    const double back = exp((double)DIM * (double)kp.beta);
    Acc acc;
    acc.clear();
    Row::clear(rows, B, lane);
    WinKeys keys;
    keys.load(wp, wg.nkeys, r0.y);
    // blocks of 32 points: lane l has point l % 32 and, half h of the wave, axis h
    // (and a half of the z weights), and a half of the transforms.  The next
    // block's strengths and the records of the one after are in flight while one
    // is worked on
    constexpr int NC = (NT + 1) / 2;
    T xa, za = T(0), xb, zb = T(0);
    unsigned sa, sb;
    int ib;
    cpx<T> ca[NC];
    const T *xh = x1 + h * wp.stride;
    auto load = [&](int i, T &x, T &z, unsigned &s, int &id) {
        const int k = min(i, pe - 1);
        x = xh[k];
        if (DIM == 3) z = x1[2 * wp.stride + k];
        s = wp.sh[k];
        id = wp.idx[k];
    };
    auto gather = [&](int id) {
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int t = NC * h + j;
            ca[j].x = ca[j].y = T(0);
            if (t < nt) ca[j] = c[t * ct + (long long)id * ci];
        }
    };
    load(p + pl, xa, za, sa, ib);
    gather(ib);
    load(p + B + pl, xb, zb, sb, ib);
    int b0 = p;
    bool staged = false;
    int strip = -1, z = 0;  // strip of the points held and the window's place in it
    const int nz = wg.nw[DIM - 1];
    const long long pstride = 2ll * g.nf[0] * g.nf[1];
    for (;;) {
        const bool last = p >= pe;
        int key = 0, ke = 0, st = -1, zk = 0;
        if (!last) {
            key = keys.key_of(wp, wg.nkeys, p);
            ke = min(pe, keys.key_end(key));
            st = key / nz;
            zk = key - st * nz;
        }
        // the planes (2D: rows) no later point of the strip reaches go to the grid
        if (DIM == 3) {
            const int nf = strip < 0 ? 0 : (st != strip ? NS : min(zk - z, NS));
            for (int k = z; k < z + nf; ++k) {
                T *plane = ft + win_wrap(k - F, g.nf[2]) * pstride;
                const int m = k % NS;
                static_for<Acc::RB>([&](auto mc) {
                    if (m == decltype(mc)::value)
                        acc.template flush<decltype(mc)::value>(plane, 2 * nftot, nt, sc, 0, 16);
                });
            }
            if (st != strip && !last) acc.place(st % wg.nw[0], st / wg.nw[0], g);
        } else {
            if (strip >= 0)
                acc.template flush<0>(ft, 2 * nftot, nt, sc, z * S & 15,
                                      st != strip ? 16 : min((zk - z) * S, 16));
            if (!last) acc.place(st, zk, g);
        }
        if (last) break;
        strip = st;
        z = zk;
        while (p < ke) {
            if (!staged || p >= b0 + B) {
                if (staged) b0 += B;
                staged = true;
                __builtin_amdgcn_wave_barrier();
                T *row = rows + pl * Row::pitch;
                Row::axis(row + h * Row::Y, xa, kp);
                if (DIM == 3) Row::half(row + Row::Z, h, za, kp);
                sh[pl] = sa;
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    ca[j].x = (T)((double)ca[j].x * back);
                    ca[j].y = (T)((double)ca[j].y * back);
                    if (NC * h + j < NT) cs[NT * pl + NC * h + j] = ca[j];
                }
                gather(ib);
                xa = xb;
                za = zb;
                sa = sb;
                load(b0 + 2 * B + pl, xb, zb, sb, ib);
                __builtin_amdgcn_wave_barrier();
            }
            const int e = min(ke, b0 + B);
            acc.accumulate(p - b0, e - b0, DIM == 3 ? z % NS : z * S & 15, rows, sh, cs);
            p = e;
        }
    }
}

template <typename T, int DIM, int NS, int NT>
__global__ void __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2)
k_win_spread(WinPts wp, const cpx<T> *__restrict__ c, long long ct, int ci, cpx<T> *__restrict__ fw,
             BinGeom g, WinGeom wg, KerParams<T> kp, int ntr, long long nftot)
{
    __shared__ WinSpreadLds<T, DIM, NS, NT> lds[4];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const JobRange jr = xcd_jobs(gridDim.x);  // one range per wave, contiguous per XCD
    const int rng = (int)jr.begin * 4 + wave;
    if (rng >= wg.ranges) return;
    const int t0 = blockIdx.y * NT;
    win_spread_range<T, DIM, NS, NT>(rng, wp, c + t0 * ct, ct, ci,
                                     reinterpret_cast<T *>(fw + (long long)t0 * nftot), g, wg, kp,
                                     min(NT, ntr - t0), nftot, lds[wave]);
}

// The ranges of all members of a plan group: wave w takes range map[w].y of item
// map[w].x (a member's transform).
template <typename T, int NS>
__global__ void __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2)
k_win_spread_group(const WinItem<T> *__restrict__ items, const int2 *__restrict__ map, int waves,
                   KerParams<T> kp)
{
    __shared__ WinSpreadLds<T, 2, NS, 1> lds[4];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // neighbouring windows on one XCD
    const int w = (int)xcd_jobs(gridDim.x).begin * 4 + wave;
    if (w >= waves) return;
    const int2 m = map[w];
    const WinItem<T> &it = items[m.x];
    const WinPts wp = it.wp;
    const BinGeom g = it.g;
    const WinGeom wg = it.wg;
    win_spread_range<T, 2, NS, 1>(m.y, wp, it.c, 0, 1, reinterpret_cast<T *>(it.fw), g, wg, kp, 1,
                                  0, lds[wave]);
}

// ---------------------------------------------------------------------------
// Interp (the product's inner dimension = (y, z) cells, 4 per instruction,
// one for each quarter of the wave).  3D: quarter (a, b) holds the y cells
// a HY .. and z cells b HZ ..; 2D: quarter q holds y = 4 i + q.  A wave takes
// up to NB batches of 16 points of one window: it takes their weights from LDS
// in the operand layout of the product (each lane only those of its own
// cells), reads the window's cells straight from the fine grid (a window is
// read once per run; neighbouring windows share lines in L1 and L2) and
// finishes with the x weights and a sum over 16 lanes.
template <typename T, int DIM, int NS>
struct InterpWin {
    static constexpr int NB = DIM == 3 ? 2 : 4;
    // points staged at a time, and held: two blocks, so that a run of 16 NB points
    // may start anywhere, where 2 workgroups per CU (FP64) then still fit
    static constexpr int block = 16 * NB;
    static constexpr int ring =
        DIM == 3 && WinRow<T, DIM, NS>::pitch * sizeof(T) * 4 * 64 <= 76 * 1024 ? 64 : block;
    static constexpr int HY = DIM == 2 ? 4 : win_interp_half(NS);
    static constexpr int HZ = DIM == 2 ? 1 : HY;
    // planes of cells in flight: all of a window where registers allow
    static constexpr int PF = DIM == 2 ? 1 : sizeof(T) == 4 || HZ == 4 ? HZ : 3;
    static constexpr int SX = 17 - NS, SY = DIM == 2 ? 17 - NS : 2 * HY - NS + 1,
                         SZ = DIM == 2 ? 1 : 2 * HZ - NS + 1;
};

template <typename T>
__device__ __forceinline__ cpx<T> load_cell(const __attribute__((address_space(1))) cpx<T> *p)
{
    cpx<T> v;
    v.x = p->x;
    v.y = p->y;
    return v;
}

// A window's cells as a lane reads them: first cell (y0, z0) of the window, the
// lane's own column gx, and for a window that does not wrap (inner) the lane's byte
// offset from the window's first row, so that an address is the offset plus a sum
// that the wave shares.
struct WinBox {
    int gx, y0, z0;
    unsigned off;
    bool inner;
};

// Sum of each of v[0..7] over a row of 16 lanes: lane i gets that of v[i / 2].  Each
// step halves the values a lane carries: it keeps one half, gives the other to the
// lane across (15 adds and 14 selects instead of 32 adds).
template <typename T>
__device__ __forceinline__ T row_sum8(const T *v)
{
    const int i = threadIdx.x;
    T a[4], b[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const T keep = i & 8 ? v[j + 4] : v[j], give = i & 8 ? v[j] : v[j + 4];
        a[j] = keep + dpp_mov<kDppRor + 8>(give);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const T keep = i & 4 ? a[j + 2] : a[j], give = i & 4 ? a[j] : a[j + 2];
        b[j] = keep + dpp_mov<kDppHalfMirror>(give);
    }
    const T keep = i & 2 ? b[1] : b[0], give = i & 2 ? b[0] : b[1];
    const T r = keep + dpp_mov<kDppQuadXor2>(give);
    return r + dpp_mov<kDppQuadXor1>(r);
}

template <typename T, int DIM, int NS, int NB, bool INNER>
__device__ __forceinline__ void win_interp_run(int s, int npt, const WinBox &w, const BinGeom &g,
                                               int M, int ntr, cpx<T> *__restrict__ c,
                                               const cpx<T> *__restrict__ fw, long long nftot,
                                               double back, const T *rows, const unsigned *sh,
                                               const int *ids)
{
    using W = InterpWin<T, DIM, NS>;
    using Row = WinRow<T, DIM, NS>;
    using Acc = typename Mfma<T>::Acc;
    constexpr int HY = W::HY, HZ = W::HZ, PF = W::PF;
    // the empty asm statements keep the compiler from forming addresses and lane
    // numbers ahead of the loops, which it would then spill
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int q = lane >> 4, i16 = lane & 15;
    int nx = g.nf[0];
    asm volatile("" : "+s"(nx));
    constexpr int E = sizeof(cpx<T>);
    const long long plane = (long long)nx * g.nf[1];
    // (address space 1: global memory, which the statements would hide)
    using Bytes = const __attribute__((address_space(1))) char *;
    using Cells = const __attribute__((address_space(1))) cpx<T> *;
    Bytes ft = (Bytes)(fw), pl;  // transform, next plane
    if (INNER) ft += (w.z0 * plane + (long long)w.y0 * nx) * E;
    unsigned row[HY];
#pragma unroll
    for (int k = 0; k < HY; ++k) row[k] = w.off + k * (DIM == 2 ? 4 : 1) * (unsigned)nx * E;
    cpx<T> v[PF][HY];
    // plane kk (2D: the rows) of the transform at ft
    auto load = [&](int kk) {
        if (INNER) {
            pl = kk ? pl + plane * E : ft;
            asm volatile("" : "+s"(pl));
#pragma unroll
            for (int k = 0; k < HY; ++k)
                v[kk % PF][k] = load_cell<T>((Cells)(pl + row[k]));
        } else {
            int y0 = w.y0;
            asm volatile("" : "+s"(y0));
            const int z = DIM == 3 ? win_wrap(w.z0 + (q >> 1) * HZ + kk, g.nf[2]) : 0;
            const Cells f = (Cells)ft + z * plane + w.gx;
#pragma unroll
            for (int k = 0; k < HY; ++k)
                v[kk % PF][k] = load_cell<T>(f + (long long)nx * win_wrap(
                    y0 + (DIM == 2 ? 4 * k + q : (q & 1) * HY + k), g.nf[1]));
        }
    };
#pragma unroll
    for (int kk = 0; kk < PF; ++kk) load(kk);
    T ky[NB][HY], kz[NB][HZ];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int p = (s + min(16 * b + i16, npt - 1)) & (W::ring - 1);
        const T *row = rows + __umul24(p, Row::pitch);
        const unsigned u = sh[p];
        const int y = (DIM == 2 ? q : (q & 1) * HY) - (int)(u >> 8 & 255);
#pragma unroll
        for (int k = 0; k < HY; ++k) ky[b][k] = row[Row::Y + Row::tap(y + (DIM == 2 ? 4 * k : k))];
        if (DIM == 3) {
            // the z taps have no zero behind them: the one of y stands in
            const int z = (q >> 1) * HZ - (int)(u >> 16);
#pragma unroll
            for (int k = 0; k < HZ; ++k)
                kz[b][k] = row[(unsigned)(z + k) < (unsigned)NS ? Row::Z + z + k : Row::Y + NS];
        }
    }
    for (int t = 0; t < ntr; ++t) {
        // keep the ky kz products inside the loop over transforms (hoisted
        // out of it they would take HY HZ registers per batch)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int k = 0; k < HY; ++k) asm volatile("" : "+v"(ky[b][k]));
        Acc ar[NB], ai[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) ar[b] = ai[b] = Acc{0, 0, 0, 0};
        // PF planes of cells in flight ahead of the one that is multiplied
#pragma unroll
        for (int kk = 0; kk < HZ; ++kk) {
#pragma unroll
            for (int k = 0; k < HY; ++k)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const T a = DIM == 3 ? ky[b][k] * kz[b][kk] : ky[b][k];
                    ar[b] = Mfma<T>::mac(a, v[kk % PF][k].x, ar[b]);
                    ai[b] = Mfma<T>::mac(a, v[kk % PF][k].y, ai[b]);
                }
            if (kk + PF < HZ) load(kk + PF);
            __builtin_amdgcn_sched_barrier(0);
        }
        ft += nftot * E;
        if (t + 1 < ntr)
#pragma unroll
            for (int kk = 0; kk < PF; ++kk) load(kk);
        // the x weights, and the sums over the cells of a row: lane i of quarter q
        // gets component (i / 2) % 2 of result row i / 4
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            int p[4];
            unsigned u[4];
            T r[8];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                p[k] = (s + min(16 * b + mfma_row<T>(q, k), npt - 1)) & (W::ring - 1);
                u[k] = sh[p[k]];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const T kx = rows[__umul24(p[k], Row::pitch) + Row::tap(i16 - (int)(u[k] & 255))];
                r[2 * k] = ar[b][k] * kx;
                r[2 * k + 1] = ai[b][k] * kx;
            }
            const T o = (T)((double)row_sum8(r) * back);
            const int pd = 16 * b + mfma_row<T>(q, i16 >> 2);
            if (!(i16 & 1) && pd < npt)
                reinterpret_cast<T *>(c + (long long)t * M + ids[(s + pd) & (W::ring - 1)])
                    [i16 >> 1 & 1] = o;
        }
    }
}

// Workgroups of 4 independent waves, one range of the order each; each XCD takes
// a contiguous part of it.
//
// Bounds per 16 points: 64 HY HZ (FP32) or 128 HY HZ clocks of the matrix cores for
// each transform, 1500 and more of the VALU, and below a few points per window the
// latency of its cells: all their loads are in flight at once, from addresses that
// the wave shares but for one offset per row.  That, the sums by row_sum8 and 3
// FP32 workgroups per CU instead of 4 that spill took two FP32 volumes of 160^3, 4e6
// points, ns 6, from 1.85 to 1.20 ms, 1e7 clustered FP64 points, ns 10, from 3.27
// to 2.46 ms and 3e6 2D FP64 points, ns 13, from 0.35 to 0.30 ms.
template <typename T, int DIM, int NS>
__global__ void __launch_bounds__(256, sizeof(T) == 4 ? 3 : 2)
k_win_interp(int M, WinPts wp, cpx<T> *__restrict__ c, const cpx<T> *__restrict__ fw, BinGeom g,
             WinGeom wg, KerParams<T> kp, int ntr, long long nftot)
{
    using W = InterpWin<T, DIM, NS>;
    using Row = WinRow<T, DIM, NS>;
    constexpr int F = (NS + 1) / 2 + 1;
    __shared__ T srow[4 * W::ring * Row::pitch];
    __shared__ unsigned ssh[4 * W::ring];
    __shared__ int sids[4 * W::ring];
    const int lane = threadIdx.x & 63, q = lane >> 4, i16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    T *rows = srow + wave * W::ring * Row::pitch;
    unsigned *sh = ssh + wave * W::ring;
    int *ids = sids + wave * W::ring;
    const T *x1 = static_cast<const T *>(wp.x);
    const JobRange jr = xcd_jobs(gridDim.x);
    const int rng = (int)jr.begin * 4 + wave;
    if (rng >= wg.ranges) return;
    const int2 r0 = wp.range[rng];
    int p = r0.x;
    const int pe = wp.range[rng + 1].x;
    if (p >= pe) return;
    const double back = exp((double)DIM * (double)kp.beta);
    WinKeys keys;
    keys.load(wp, wg.nkeys, r0.y);
    Row::clear(rows, W::ring, lane);
    // 3D: blocks of 32 points, lane l has point l % 32 and, half h of the wave,
    // axis h and a half of the z weights.  2D: blocks of 64, both axes.  The next
    // block is in flight while one is worked on.
    const int h = DIM == 3 ? lane >> 5 : 0, pl = lane & (W::block - 1);
    T xa[2];
    unsigned sa;
    int ia;
    auto load = [&](int i) {
        const int k = min(i, pe - 1);
        xa[0] = x1[h * wp.stride + k];
        xa[1] = x1[(DIM - 1) * wp.stride + k];
        sa = wp.sh[k];
        ia = wp.idx[k];
    };
    int b0 = p, se = p;  // the range's first point, the staged points' end
    auto stage = [&]() {
        __builtin_amdgcn_wave_barrier();
        const int at = (se - b0 + pl) & (W::ring - 1);
        T *row = rows + at * Row::pitch;
        Row::axis(row + h * Row::Y, xa[0], kp);
        if (DIM == 3)
            Row::half(row + Row::Z, h, xa[1], kp);
        else
            Row::axis(row + Row::Y, xa[1], kp);
        sh[at] = sa;
        ids[at] = ia;
        se += W::block;
        load(se + pl);
        __builtin_amdgcn_wave_barrier();
    };
    load(p + pl);
    while (p < pe) {
        const int key = keys.key_of(wp, wg.nkeys, p);
        const int ke = min(pe, keys.key_end(key));
        const int st = DIM == 3 ? key / wg.nw[2] : key;
        const int kz = DIM == 3 ? key - st * wg.nw[2] : 0;
        const int ky = st / wg.nw[0], kx = st - ky * wg.nw[0];
        WinBox w;
        w.y0 = ky * W::SY - F;
        w.z0 = DIM == 3 ? kz * W::SZ - F : 0;
        w.gx = win_wrap(kx * W::SX - F + i16, g.nf[0]);
        const long long plane = (long long)g.nf[0] * g.nf[1];
        w.inner = w.y0 >= 0 && w.y0 + (DIM == 2 ? 16 : 2 * W::HY) <= g.nf[1] &&
                  (DIM == 2 ? g.nf[0] < 1 << 24  // offsets fit 32 bits
                            : w.z0 >= 0 && w.z0 + 2 * W::HZ <= g.nf[2] && plane < 1 << 25);
        w.off = (unsigned)((w.gx + (DIM == 2 ? q : (q & 1) * W::HY) * (long long)g.nf[0] +
                            (DIM == 3 ? (q >> 1) * W::HZ * plane : 0)) *
                           (long long)sizeof(cpx<T>));
        while (p < ke) {
            int npt = min(ke - p, 16 * W::NB);
            if (W::ring > W::block ? p + npt > se : p >= se) stage();
            // (the first run of a range needs at most one block, a later one finds
            // its first point's staged)
            if (W::ring == W::block) npt = min(npt, se - p);
#define CFA_RUN(NB)                                                                                \
    do {                                                                                         \
        if (w.inner)                                                                             \
            win_interp_run<T, DIM, NS, NB, true>(p - b0, npt, w, g, M, ntr, c, fw, nftot, back,  \
                                                 rows, sh, ids);                                 \
        else                                                                                     \
            win_interp_run<T, DIM, NS, NB, false>(p - b0, npt, w, g, M, ntr, c, fw, nftot, back, \
                                                  rows, sh, ids);                                \
    } while (0)
            if (npt <= 16)
                CFA_RUN(1);
            else if (W::NB == 2 || npt <= 32)
                CFA_RUN(2);
            else
                CFA_RUN(W::NB);
#undef CFA_RUN
            p += npt;
        }
    }
}

}  // namespace cfa
