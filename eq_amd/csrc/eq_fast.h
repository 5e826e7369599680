// eq_fast.h -- the fast direct solver's plans, transforms and row kernels
// (eq_fast.hip has the method).  The transform kernels are instantiated in one
// translation unit per precision and kind of rows (eq_fast_*.hip): together
// they take minutes to compile.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <new>
#include <type_traits>
#include <utility>
#include <vector>

#include "eq_internal.h"

namespace eqk {


// ------------------------------------------------------------ plans

constexpr int kFastMaxStages = 12;
constexpr int kFastValues = 8;        // complex values a thread holds per transform pass (16 above 8192 points:
constexpr int kFastValuesWide = 16;   // more registers, fewer waves in flight)
static_assert(kFastValuesWide == 2 * kFastValues, "a class of twice 1024 threads runs 1024 of twice the values");
constexpr int kFastModes = 16;        // modes (columns) a block of the line solve takes
constexpr int kFastRowsMax = 4096;    // rows the line solve holds in one block
constexpr int64_t kFastLds = 150 * 1024;
constexpr int kFastGiveUp = 32;       // applications before the multigrid solver takes over,
constexpr int kChebMax = 64;          // and where the coefficients vary

enum FastEnds { kEndsNN = 0, kEndsDD = 1, kEndsND = 2, kEndsDN = 3 };

// One transform length: rows of N cells, 2N points (n), on a smooth length M
// (M == n, or the chirp's).  Tables are complex, in the solve's precision.
struct FastPlan {
    int32_t N, n, M, chirp;
    int32_t nstages;
    struct Pass {
        int32_t R, m, Ns, step; // radix, M / R, product of the radices before, m / Ns
    } pass[kFastMaxStages];
    int64_t tw;     // M: exp(-2 pi i k / M)
    int64_t quart;  // N + 1: exp(-pi i j / (2 N))
    int64_t ch;     // chirp: n values exp(-pi i j^2 / n)
    int64_t hh;     // chirp: M values, the transformed kernel / M
};

struct FastProb {
    int32_t plan, ends;
    int32_t pair0, npairs;  // this problem's slots of row-pair partials
    int64_t mode0;          // its modes' records
    double gain;            // what an application leaves of the error at most, squared (constant coefficients)
    double unit;            // an update's size in the right-hand side's units, squared
};

// A mode's tridiagonal inverse along y (k_fast_lines), laid out once: forming
// it takes a thread more time than the sweeps of 16 rows do.
struct FastMode {
    double rho, irho; // the decay of both recursions, and 1 / rho
    double scale;     // c and both transforms' factors
    double a0, a1;    // A = a0 w_0 + a1 w_ny
    double b0, b1;    // B = b0 w_ny + b1 A
    double w, wl;     // rho to the rows of a chunk, and of the last one
};

// The rows of a problem's operator and right-hand side by place: bottom row,
// between, top row by left column, between, right column.  A node at a wall
// then costs the same loads as any other (the frame around a field is zero),
// only other coefficients; evaluating the element counts there made the few
// blocks of wall rows the last to finish, at twice the launch's time.
struct FastRows {
    Row<double> a[3][3];
    double b[3][3][8]; // c, w, e, s, n, sw, ne of M, and the sources
};

// a block's work: problem and row pair (forward, backward) or mode group
struct FastJob {
    int32_t prob, at;
};

struct FastClass {
    int threads = 0;        // of the transform blocks
    size_t lds = 0;
    int32_t job0 = 0, njobs = 0;
    double nodes = 0.0;
};

struct FastSolver {
    std::vector<FastClass> classes;
    int32_t nline = 0, line_c = 0, line_rows = 0;
    FastPlan* d_plans = nullptr;
    FastProb* d_probs = nullptr;
    FastRows* d_rows = nullptr;
    FastJob* d_jobs = nullptr;   // row pairs, class by class
    FastJob* d_lines = nullptr;  // mode groups
    FastMode* d_modes = nullptr;
    void* d_tables = nullptr;
    double* d_partial = nullptr; // 3 per row pair: residual, right-hand side, last update
    bool robin_x = false; // some left or right wall is a Robin wall
    // beyond the constant operator (tensor field, advection, Robin walls
    // across x): per problem kChebMax
    // pairs (weight of the correction, weight of the one before); whether
    // every problem's bounds allow the solver; the applications they predict
    double2* d_cheb = nullptr;
    int32_t* d_extra = nullptr;  // per problem: applications after the tolerance is met,
    int32_t* d_met = nullptr;    // and where it first was (-1: not yet)
    bool general_ok = false;
    int rest = 0, last_rest = 0; // steps that leave the solver out after it gave up, and how many the last time
    std::vector<uint8_t> chirp; // per problem: its transforms are chirps
    // tensor fields: the stiffness weights of every node to its W, S and SW
    // neighbour (three arrays of level 0's layout, zero in the frame), formed
    // anew by each solve
    double* d_stiff = nullptr;
    int64_t stiff_stride = 0;
    int recent[2][4] = {{3, 3, 3, 3}, {3, 3, 3, 3}}; // application counts of the last solves, constant and varying
    int at[2] = {0, 0};
    static constexpr int kGraphs = 49;
    hipGraphExec_t graph[kGraphs] = {}; // a solve's first chunk of that many applications
    Acct acct[kGraphs];
};

// ------------------------------------------------------------ complex values

template <typename T>
struct alignas(2 * sizeof(T)) Cx {
    T x, y;
};
template <typename T>
__device__ __forceinline__ Cx<T> operator+(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> operator-(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> mul(Cx<T> a, Cx<T> b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// a * conj(b)
template <typename T>
__device__ __forceinline__ Cx<T> mulc(Cx<T> a, Cx<T> b) { return {a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y}; }
// -i a
template <typename T>
__device__ __forceinline__ Cx<T> mi(Cx<T> a) { return {a.y, -a.x}; }

// ------------------------------------------------------------ small transforms (in registers, exp(-2 pi i jk/R))

template <typename T>
__device__ __forceinline__ void dft2(Cx<T>& a, Cx<T>& b)
{
    const Cx<T> t = a - b;
    a = a + b;
    b = t;
}

template <typename T>
__device__ __forceinline__ void dft4(Cx<T>& a, Cx<T>& b, Cx<T>& c, Cx<T>& d)
{
    const Cx<T> s = a + c, t = a - c, u = b + d, v = mi(b - d);
    a = s + u;
    b = t + v;
    c = s - u;
    d = t - v;
}

template <typename T, int R>
__device__ __forceinline__ void dft(Cx<T> (&v)[R])
{
    if constexpr (R == 2) {
        dft2(v[0], v[1]);
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        const T h = (T)0.70710678118654752440;
        dft4(v[0], v[2], v[4], v[6]);
        dft4(v[1], v[3], v[5], v[7]);
        const Cx<T> w1 = {(v[3].x + v[3].y) * h, (v[3].y - v[3].x) * h};
        const Cx<T> w2 = mi(v[5]);
        const Cx<T> w3 = {(v[7].y - v[7].x) * h, -(v[7].x + v[7].y) * h};
        const Cx<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
        v[0] = e0 + o0;
        v[4] = e0 - o0;
        v[1] = e1 + w1;
        v[5] = e1 - w1;
        v[2] = e2 + w2;
        v[6] = e2 - w2;
        v[3] = e3 + w3;
        v[7] = e3 - w3;
    } else if constexpr (R == 3) {
        const T c = (T)-0.5, s = (T)0.86602540378443864676;
        const Cx<T> a = v[1] + v[2], b = v[1] - v[2];
        const Cx<T> m = {v[0].x + c * a.x, v[0].y + c * a.y};
        v[0] = v[0] + a;
        v[1] = {m.x + s * b.y, m.y - s * b.x};
        v[2] = {m.x - s * b.y, m.y + s * b.x};
    } else if constexpr (R == 5) {
        const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
        const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
        const Cx<T> a1 = v[1] + v[4], b1 = v[1] - v[4], a2 = v[2] + v[3], b2 = v[2] - v[3];
        const Cx<T> m1 = {v[0].x + c1 * a1.x + c2 * a2.x, v[0].y + c1 * a1.y + c2 * a2.y};
        const Cx<T> m2 = {v[0].x + c2 * a1.x + c1 * a2.x, v[0].y + c2 * a1.y + c1 * a2.y};
        const Cx<T> n1 = {s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y};
        const Cx<T> n2 = {s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y};
        v[0] = v[0] + a1 + a2;
        v[1] = {m1.x + n1.y, m1.y - n1.x};
        v[4] = {m1.x - n1.y, m1.y + n1.x};
        v[2] = {m2.x + n2.y, m2.y - n2.x};
        v[3] = {m2.x - n2.y, m2.y + n2.x};
    } else if constexpr (R == 6 || R == 10) {
        // 2 x R/2 with coprime factors (Good-Thomas): no twiddles
        constexpr int H = R / 2;
        Cx<T> e[H], o[H];
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const Cx<T> a = v[(2 * q) % R], b = v[(2 * q + H) % R];
            e[q] = a + b;
            o[q] = a - b;
        }
        dft<T, H>(e);
        dft<T, H>(o);
        // output k: residues (k mod 2, k mod H)
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = (k & 1) ? o[k % H] : e[k % H];
    } else if constexpr (R == 9) {
        const T c1 = (T)0.76604444311897803520, s1 = (T)0.64278760968653932632;
        const T c2 = (T)0.17364817766693034885, s2 = (T)0.98480775301220805937;
        const T c4 = (T)-0.93969262078590838405, s4 = (T)0.34202014332566873304;
        Cx<T> a[3], b[3], c[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            a[q] = v[3 * q];
            b[q] = v[3 * q + 1];
            c[q] = v[3 * q + 2];
        }
        dft<T, 3>(a);
        dft<T, 3>(b);
        dft<T, 3>(c);
        b[1] = mul(b[1], Cx<T>{c1, -s1});
        b[2] = mul(b[2], Cx<T>{c2, -s2});
        c[1] = mul(c[1], Cx<T>{c2, -s2});
        c[2] = mul(c[2], Cx<T>{c4, -s4});
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            Cx<T> t[3] = {a[q], b[q], c[q]};
            dft<T, 3>(t);
            v[q] = t[0];
            v[q + 3] = t[1];
            v[q + 6] = t[2];
        }
    } else {
        static_assert(R == 7, "radix");
        const T c1 = (T)0.62348980185873353053, c2 = (T)-0.22252093395631440429, c3 = (T)-0.90096886790241912624;
        const T s1 = (T)0.78183148246802980871, s2 = (T)0.97492791218182360702, s3 = (T)0.43388373911755812048;
        const Cx<T> a1 = v[1] + v[6], b1 = v[1] - v[6], a2 = v[2] + v[5], b2 = v[2] - v[5];
        const Cx<T> a3 = v[3] + v[4], b3 = v[3] - v[4], z = v[0];
        const Cx<T> m1 = {z.x + c1 * a1.x + c2 * a2.x + c3 * a3.x, z.y + c1 * a1.y + c2 * a2.y + c3 * a3.y};
        const Cx<T> m2 = {z.x + c2 * a1.x + c3 * a2.x + c1 * a3.x, z.y + c2 * a1.y + c3 * a2.y + c1 * a3.y};
        const Cx<T> m3 = {z.x + c3 * a1.x + c1 * a2.x + c2 * a3.x, z.y + c3 * a1.y + c1 * a2.y + c2 * a3.y};
        const Cx<T> n1 = {s1 * b1.x + s2 * b2.x + s3 * b3.x, s1 * b1.y + s2 * b2.y + s3 * b3.y};
        const Cx<T> n2 = {s2 * b1.x - s3 * b2.x - s1 * b3.x, s2 * b1.y - s3 * b2.y - s1 * b3.y};
        const Cx<T> n3 = {s3 * b1.x - s1 * b2.x + s2 * b3.x, s3 * b1.y - s1 * b2.y + s2 * b3.y};
        v[0] = z + a1 + a2 + a3;
        v[1] = {m1.x + n1.y, m1.y - n1.x};
        v[6] = {m1.x - n1.y, m1.y + n1.x};
        v[2] = {m2.x + n2.y, m2.y - n2.x};
        v[5] = {m2.x - n2.y, m2.y + n2.x};
        v[3] = {m3.x + n3.y, m3.y - n3.x};
        v[4] = {m3.x - n3.y, m3.y + n3.x};
    }
}

// ------------------------------------------------------------ transforms in LDS

// One Stockham pass of radix R in place: every value is held in registers
// across the barrier between its read and its write.  M <= V NT.  Output
// element i goes to store(i, value).  The passes run odd and singly even
// radices first (see make_plan), so the strided writes of the early ones
// spread over the LDS banks without padding.
template <typename T, int R, int NT, int V, typename S>
__device__ __forceinline__ void fft_pass(Cx<T>* s, const FastPlan::Pass& ps, const Cx<T>* __restrict__ tw, S&& store)
{
    constexpr int B = (V + R - 1) / R;
    const int m = ps.m, Ns = ps.Ns;
    const float inv = 1.0f / (float)Ns;
    const uint32_t step = (uint32_t)ps.step * (uint32_t)sizeof(Cx<T>);
    Cx<T> v[B][R];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int k = (int)threadIdx.x + b * NT;
        if (k < m)
#pragma unroll
            for (int r = 0; r < R; ++r) v[b][r] = s[k + r * m];
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int k = (int)threadIdx.x + b * NT;
        if (k < m) {
            // k = p Ns + q with q the position inside the finished sub-transforms
            const int p = (int)(((float)k + 0.5f) * inv), q = k - p * Ns;
            if (Ns > 1) {
                const uint32_t t = (uint32_t)q * step;
#pragma unroll
                for (int r = 1; r < R; ++r) v[b][r] = mul(v[b][r], *(const Cx<T>*)((const char*)tw + t * (uint32_t)r));
            }
            dft<T, R>(v[b]);
            const int o = p * Ns * R + q;
#pragma unroll
            for (int r = 0; r < R; ++r) store(o + r * Ns, v[b][r]);
        }
    }
}

// The pass's sizes come from its record: worked out in place, every radix's
// would be kept in registers through the loop over the passes.
template <typename T, int NT, int V, typename S>
__device__ __forceinline__ void fft_radix(Cx<T>* s, const FastPlan::Pass& ps, const Cx<T>* __restrict__ tw, S&& store)
{
    switch (ps.R) {
    case 10: fft_pass<T, 10, NT, V>(s, ps, tw, store); break;
    case 9: fft_pass<T, 9, NT, V>(s, ps, tw, store); break;
    case 8: fft_pass<T, 8, NT, V>(s, ps, tw, store); break;
    case 7: fft_pass<T, 7, NT, V>(s, ps, tw, store); break;
    case 6: fft_pass<T, 6, NT, V>(s, ps, tw, store); break;
    case 5: fft_pass<T, 5, NT, V>(s, ps, tw, store); break;
    case 4: fft_pass<T, 4, NT, V>(s, ps, tw, store); break;
    case 3: fft_pass<T, 3, NT, V>(s, ps, tw, store); break;
    default: fft_pass<T, 2, NT, V>(s, ps, tw, store); break;
    }
}

// The M-point transform of the row in LDS; the last pass hands its outputs to
// `last` (after a barrier behind the pass's reads, so it may write the row).
template <typename T, int NT, int V, typename S>
__device__ __forceinline__ void fft_lds(Cx<T>* s, const FastPlan& pl, const Cx<T>* __restrict__ tab, S&& last)
{
    const Cx<T>* tw = tab + pl.tw;
    const int n = pl.nstages - 1;
    for (int k = 0; k < n; ++k) {
        fft_radix<T, NT, V>(s, pl.pass[k], tw, [&](int i, Cx<T> v) { s[i] = v; });
        __syncthreads();
    }
    fft_radix<T, NT, V>(s, pl.pass[n], tw, last);
}

// The plan's n-point transform of the row placed with put_at, elements 0 .. N
// to out(k, value): the smooth length directly, or the chirp convolution (its
// second transform runs on the conjugate, so its result is conjugate).
template <typename T, int NT, int V, typename S>
__device__ __forceinline__ void row_transform(Cx<T>* s, const FastPlan& pl, const Cx<T>* __restrict__ tab, S&& out)
{
    const int N = pl.N;
    __syncthreads();
    if (!pl.chirp) {
        fft_lds<T, NT, V>(s, pl, tab, [&](int k, Cx<T> v) {
            if (k <= N) out(k, v);
        });
        return;
    }
    const Cx<T>* h = tab + pl.hh;
    fft_lds<T, NT, V>(s, pl, tab, [&](int k, Cx<T> v) {
        const Cx<T> p = mul(v, h[k]);
        s[k] = {p.x, -p.y};
    });
    __syncthreads();
    const Cx<T>* ch = tab + pl.ch;
    fft_lds<T, NT, V>(s, pl, tab, [&](int k, Cx<T> v) {
        if (k <= N) out(k, mul(Cx<T>{v.x, -v.y}, ch[k]));
    });
}
// element j of the period-n row, -n/2 <= j <= n/2
template <typename T>
__device__ __forceinline__ void put_at(Cx<T>* s, const FastPlan& pl, const Cx<T>* __restrict__ tab, int j, Cx<T> v)
{
    if (pl.chirp) v = mul(v, tab[pl.ch + (j < 0 ? -j : j)]);
    s[j < 0 ? j + pl.M : j] = v;
}
// the chirp's gap between the placed rows: elements a .. b are zero
template <typename T, int NT>
__device__ __forceinline__ void clear_gap(Cx<T>* s, const FastPlan& pl, int a, int b)
{
    if (!pl.chirp) return;
    for (int k = a + (int)threadIdx.x; k <= b; k += NT) s[k] = {(T)0, (T)0};
}

// The residual's scale.  Single precision holds the residual of a solve, from
// about the right-hand side to 1e-12 of it, only within its own range of
// exponents, so it is transformed times 2^-e (exact), e the exponent of the
// problem's first residual and right-hand side, and what comes back is added
// times 2^e.  The first launch of a solve takes the e of the solve before, and
// finds its own norms: within kFastScaleOff of them e stays (the 250 exponents
// leave room), else that launch's transform is dropped, the next one starts
// with the new e.  The results are the same bits whatever e is.
constexpr int kFastScaleOff = 32;

// (an exponent in a scalar register: a factor took two more vector registers
// of the forward transform, 34.4 -> 37.0 us at 2000x1000)
template <typename T>
__device__ __forceinline__ T scaled(double v, int e)
{
    return sizeof(T) == 4 ? (T)ldexp(v, e) : (T)v;
}

// Whether a solve is over: the residual rr within the tolerance and, with
// constant coefficients, the error within kFastError of it.  The residual alone
// does not tell the error: where the last application just got there the error
// is 3e-3 to 5e-2 of the residual (smooth fields, small dt D), up to 2e-12 of a
// field where the V-cycle CG left 2e-14 to 1e-12; and rounding (4e-12 at
// 2000x1000) hides how far below the tolerance the error is.  But the last
// update is the error before it, and an application leaves the part of it that
// the residuals show, at most `gain`.  All squared: prev the residual before
// the last application (< 0: there was none), upd that update in the
// right-hand side's units.  (varying: a fixed number of applications follow
// instead, fast_refresh)
constexpr double kFastError = 1e-4;
// A right-hand side without a finite norm makes every residual pass: only a
// kept solution is one then, as for the V-cycle solvers, which take the others.
__device__ __forceinline__ bool within(double rr, double tol, double prev, double upd, double gain, bool varying,
                                       bool kept)
{
    return rr <= tol && (rr < HUGE_VAL || kept) &&
           (varying || prev < 0.0 || upd * fmin(gain, rr / prev) <= kFastError * kFastError * tol);
}

// waves per SIMD the transform kernels are compiled for
constexpr int fast_waves(size_t elem, int NT, int V) { return V > kFastValues ? 4 : elem == 4 ? 8 : 4; }

// ------------------------------------------------------------ residual rows

__device__ __forceinline__ int swizzled_block()
{
    // workgroups are dealt round-robin to the 8 XCDs: each takes a contiguous
    // run of the jobs, so the rows two blocks share are in one L2
    const int per = gridDim.x >> 3;
    const int b = blockIdx.x;
    return (b & 7) * per + (b >> 3);
}

__device__ __forceinline__ double wave_add(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

struct PairWindow { // rows i0-1 .. i0+2 of column j, and of its neighbours as far as the two rows need them
    double m[4], w[3], e[3];
    __device__ __forceinline__ void load(const double* __restrict__ v, int j, const int (&row)[4])
    {
#pragma unroll
        for (int q = 0; q < 4; ++q) m[q] = v[row[q] + j];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            w[q] = v[row[q] + j - 1];
            e[q] = v[row[q + 1] + j + 1];
        }
    }
    // any row's coefficients
    __device__ __forceinline__ double apply(const Row<double>& r, int k) const
    {
        return row_apply<false>(r, m[k + 1], w[k + 1], e[k], m[k], m[k + 2], w[k], e[k + 1]);
    }
    __device__ __forceinline__ double rhs(const double* c, int k) const
    {
        return c[0] * m[k + 1] + ((c[1] * w[k + 1] + c[2] * e[k]) + (c[3] * m[k] + c[4] * m[k + 2])) +
               (c[5] * w[k] + c[6] * e[k + 1]) + c[7];
    }
    // a row off the walls: its neighbours' weights are equal, or equal by axis
    __device__ __forceinline__ double apply_inner(double mc, double mo, double kx, double ky, int k) const
    {
        const double c = m[k + 1];
        return (kx * ((c - w[k + 1]) + (c - e[k])) + ky * ((c - m[k]) + (c - m[k + 2]))) + rhs_inner(mc, mo, k);
    }
    // any row's coefficients, the diagonal neighbours' stiffness with them
    __device__ __forceinline__ double apply_full(const Row<double>& r, int k) const
    {
        return row_apply<true>(r, m[k + 1], w[k + 1], e[k], m[k], m[k + 2], w[k], e[k + 1]);
    }
    // a row off the walls from its stiffness weights: s points at the row's
    // node in the weights to W, to S and to SW (the others are theirs)
    __device__ __forceinline__ double apply_stiff(double mc, double mo, const double* __restrict__ s, int64_t st, int pt,
                                                  int k) const
    {
        const double c = m[k + 1];
        const double y = (s[0] * (c - w[k + 1]) + s[1] * (c - e[k])) + (s[st] * (c - m[k]) + s[st + pt] * (c - m[k + 2])) +
                         (s[2 * st] * (c - w[k]) + s[2 * st + pt + 1] * (c - e[k + 1]));
        return y + rhs_inner(mc, mo, k);
    }
    // convection of a row off the walls (difference form: add_convection_v)
    __device__ __forceinline__ double convect(double a, double b, double d, int k) const
    {
        return a * (e[k] - w[k + 1]) + (b * (m[k] - w[k]) + d * (e[k + 1] - m[k + 2]));
    }
    __device__ __forceinline__ double rhs_inner(double mc, double mo, int k) const
    {
        return mc * m[k + 1] + mo * (((w[k + 1] + e[k]) + (m[k] + m[k + 2])) + (w[k] + e[k + 1]));
    }
};

// Rows i0 and i0 + 1 of the residual b - A x, b = M u + sources, column by
// column; f(j, r0, r1) takes them (0 on held nodes, where x holds the wall
// value).  Sums r^2, and with want_b the row-replaced b^2, into acc.
// GEN: problems of the batch have a tensor field or advection.
template <int NT, bool GEN, typename F>
__device__ __forceinline__ void residual_pair(const LevelProb& P, const FastRows& tab, int i0,
                                              const double* __restrict__ u, const double* __restrict__ x,
                                              const double* __restrict__ stiff, int64_t sst, bool want_b,
                                              double (&acc)[2], F&& f)
{
    const int nx = P.nx, ny = P.ny, pt = P.pitch;
    const bool in1 = i0 + 1 <= ny;
    const double* __restrict__ ur = u + P.origin + (int64_t)i0 * pt;
    const double* __restrict__ xr = x + P.origin + (int64_t)i0 * pt;
    const int row[4] = {-pt, 0, pt, in1 ? 2 * pt : pt}; // (the frame ends at row ny + 1)
    const bool inner = i0 > 0 && i0 + 1 < ny;
    // one column with the table's rows (column class cc)
    auto by_table = [&](int j, int cc) {
        const int c0 = i0 == 0 ? 0 : i0 == ny ? 2 : 1, c1 = i0 + 1 >= ny ? 2 : 1;
        PairWindow U, X;
        U.load(ur, j, row);
        X.load(xr, j, row);
        double b0 = U.rhs(tab.b[c0][cc], 0), b1 = in1 ? U.rhs(tab.b[c1][cc], 1) : 0.0;
        double r0, r1;
        if (GEN && (P.aniso || P.vel)) {
            // (one lane's chain at the wall columns, so a short one: the
            // table's masses with the node's own stiffness)
            auto row_of = [&](int c, int q) {
                Row<double> r = tab.a[c][cc];
                if (P.aniso) {
                    const double* s = stiff + P.origin + (int64_t)(i0 + q) * pt + j;
                    r.kw = s[0];
                    r.ke = s[1];
                    r.ks = s[sst];
                    r.kn = s[sst + pt];
                    r.ksw = s[2 * sst];
                    r.kne = s[2 * sst + pt + 1];
                }
                if (P.vel) add_convection<double>(P, i0 + q, j, P.vel_d, r);
                return r;
            };
            r0 = b0 - X.apply_full(row_of(c0, 0), 0);
            r1 = in1 ? b1 - X.apply_full(row_of(c1, 1), 1) : 0.0;
        } else {
            r0 = b0 - X.apply(tab.a[c0][cc], 0);
            r1 = in1 ? b1 - X.apply(tab.a[c1][cc], 1) : 0.0;
        }
        if (is_dirichlet(P, i0, j)) {
            r0 = 0.0;
            b0 = want_b ? dirichlet_value(P, i0, j) : 0.0;
        }
        if (in1 && is_dirichlet(P, i0 + 1, j)) {
            r1 = 0.0;
            b1 = want_b ? dirichlet_value(P, i0 + 1, j) : 0.0;
        }
        acc[0] += r0 * r0 + r1 * r1;
        acc[1] += b0 * b0 + b1 * b1;
        f(j, r0, r1);
    };
    // the wall columns: one lane of a wave each, first
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
#pragma unroll 1
    for (int e = wave; e < 2; e += NT / 64)
        if ((threadIdx.x & 63) == 0) by_table(e ? nx : 0, e ? 2 : 0);
    if (inner) {
        const Row<double>& ra = tab.a[1][1];
        const double mc = ra.mc, mo = ra.mw, kx = ra.kw, ky = ra.ks;
        const double c0 = tab.b[1][1][0], c1 = tab.b[1][1][1], cs = tab.b[1][1][7];
        double ca[2] = {0.0, 0.0}, cb[2] = {0.0, 0.0}, cd[2] = {0.0, 0.0};
        const bool vel = GEN && P.vel;
        if (vel)
            for (int q = 0; q < 2; ++q) {
                const double* v = P.vel_d + i0 + q;
                ca[q] = P.cw * (6.0 * v[0] + v[-1] + v[1]);
                cb[q] = P.cw * 2.0 * (v[0] + v[-1]);
                cd[q] = P.cw * 2.0 * (v[0] + v[1]);
            }
#pragma unroll 1
        for (int j = 1 + (int)threadIdx.x; j < nx; j += NT) {
            PairWindow U, X;
            U.load(ur, j, row);
            X.load(xr, j, row);
            const double b0 = U.rhs_inner(c0, c1, 0) + cs, b1 = U.rhs_inner(c0, c1, 1) + cs;
            double r0, r1;
            if (GEN && P.aniso) {
                const double* s = stiff + P.origin + (int64_t)i0 * pt + j;
                r0 = b0 - X.apply_stiff(mc, mo, s, sst, pt, 0);
                r1 = b1 - X.apply_stiff(mc, mo, s + pt, sst, pt, 1);
            } else {
                r0 = b0 - X.apply_inner(mc, mo, kx, ky, 0);
                r1 = b1 - X.apply_inner(mc, mo, kx, ky, 1);
            }
            if (vel) {
                r0 -= X.convect(ca[0], cb[0], cd[0], 0);
                r1 -= X.convect(ca[1], cb[1], cd[1], 1);
            }
            acc[0] += r0 * r0 + r1 * r1;
            acc[1] += b0 * b0 + b1 * b1;
            f(j, r0, r1);
        }
    } else {
#pragma unroll 1
        for (int j = 1 + (int)threadIdx.x; j < nx; j += NT) by_table(j, 1);
    }
}

// block sums of two values in wave order; valid in thread 0
template <int NT>
__device__ __forceinline__ void block_pair(double (&v)[2])
{
    __shared__ double red[NT / 64][2];
    v[0] = wave_add(v[0]);
    v[1] = wave_add(v[1]);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6][0] = v[0];
        red[threadIdx.x >> 6][1] = v[1];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        v[0] = v[1] = 0.0;
        for (int w = 0; w < NT / 64; ++w) {
            v[0] += red[w][0];
            v[1] += red[w][1];
        }
    }
}

// ------------------------------------------------------------ kernels

// Residual of the iterate and its transform along x, two rows a block.
// k: applications done so far in this solve (0: the first residual, which
// also takes ||b||^2).  start: this launch begins a chunk of the host's loop.
template <typename T, int NT, int V, bool GEN>
__global__ __launch_bounds__(NT, GEN ? 4 : fast_waves(sizeof(T), NT, V)) void k_fast_forward(const FastJob* __restrict__ jobs, int njobs,
                                                     const LevelProb* __restrict__ probs,
                                                     const FastProb* __restrict__ fp, const FastRows* __restrict__ rows,
                                                     const FastPlan* __restrict__ plans, const Cx<T>* __restrict__ tab,
                                                     const double* __restrict__ u,
                                                     const double* __restrict__ x, const double* __restrict__ stiff,
                                                     int64_t sst, T* __restrict__ out,
                                                     double* __restrict__ partial, CgState* st, int k, int start)
{
    extern __shared__ char lds_raw[];
    Cx<T>* s = (Cx<T>*)lds_raw;
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    CgState& cs = st[P.prob];
    if (k > 0 && cs.done) {
        // a problem that an earlier chunk finished has its field already
        if (start && job.at == 0 && threadIdx.x == 0) cs.done = 2;
        return;
    }
    const FastProb f = fp[job.prob];
    const FastPlan& pl = plans[f.plan];
    const int N = pl.N, i0 = 2 * job.at;
    double acc[2] = {0.0, 0.0};
    const int ends = f.ends;
    const T two = (T)2;
    const int e = k == 0 ? -cs.fast_e0 : -cs.fast_e;
    clear_gap<T, NT>(s, pl, N + 1, pl.M - N);
    residual_pair<NT, GEN>(P, rows[job.prob], i0, u, x, stiff, sst, k == 0, acc, [&](int j, double r0, double r1) {
        Cx<T> v = {scaled<T>(r0, e), scaled<T>(r1, e)};
        if (ends == kEndsNN) {
            if (j == 0 || j == N) {
                put_at(s, pl, tab, j, Cx<T>{two * v.x, two * v.y});
            } else {
                put_at(s, pl, tab, j, v);
                put_at(s, pl, tab, pl.chirp ? -j : 2 * N - j, v);
            }
        } else if (ends == kEndsDD) {
            // odd: zero at both ends (v is zero on held nodes)
            put_at(s, pl, tab, j, v);
            if (j > 0 && j < N) put_at(s, pl, tab, pl.chirp ? -j : 2 * N - j, Cx<T>{-v.x, -v.y});
        } else {
            const int jj = ends == kEndsDN ? N - j : j;
            const Cx<T> q = tab[pl.quart + jj];
            if (jj == 0) {
                put_at(s, pl, tab, 0, Cx<T>{two * v.x, two * v.y});
            } else {
                put_at(s, pl, tab, jj, jj == N ? Cx<T>{(T)0, (T)0} : mul(v, q));
                if (jj < N) put_at(s, pl, tab, pl.chirp ? -jj : 2 * N - jj, mulc(v, q));
            }
        }
    });
    block_pair<NT>(acc);
    if (threadIdx.x == 0) {
        partial[3 * (int64_t)(f.pair0 + job.at)] = acc[0];
        partial[3 * (int64_t)(f.pair0 + job.at) + 1] = acc[1];
    }
    T* __restrict__ o0 = out + P.origin + (int64_t)i0 * P.pitch;
    const bool second = i0 + 1 <= P.ny;
    const int pitch = P.pitch;
    row_transform<T, NT, V>(s, pl, tab, [&](int q, Cx<T> v) {
        const Cx<T> w = ends == kEndsDD ? Cx<T>{-v.y, v.x} : v;
        o0[q] = w.x;
        if (second) o0[q + pitch] = w.y;
    });
}

// Transform back along x and x += z, two rows a block, and the update's square
// sum.  GEN: one application of the Chebyshev iteration, d <- alpha z + beta d,
// x += d, with d in FP64 (as the directions of BiCGStab are).
template <typename T, int NT, int V, bool GEN>
__global__ __launch_bounds__(NT, fast_waves(sizeof(T), NT, V)) void k_fast_backward(const FastJob* __restrict__ jobs, int njobs,
                                                      const LevelProb* __restrict__ probs,
                                                      const FastProb* __restrict__ fp,
                                                      const FastPlan* __restrict__ plans,
                                                      const Cx<T>* __restrict__ tab, const T* __restrict__ in,
                                                      double* __restrict__ x, const CgState* __restrict__ st,
                                                      double* __restrict__ d, const double2* __restrict__ cheb,
                                                      double* __restrict__ partial, int k)
{
    extern __shared__ char lds_raw[];
    Cx<T>* s = (Cx<T>*)lds_raw;
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    const CgState& cs = st[P.prob];
    if (cs.done) return;
    const int app = k - cs.fast_void; // the application of this solve
    if (app < 0) return;
    const int up = sizeof(T) == 4 ? cs.fast_e : 0;
    const FastProb f = fp[job.prob];
    const FastPlan& pl = plans[f.plan];
    const int N = pl.N, i0 = 2 * job.at, ends = f.ends;
    const bool second = i0 + 1 <= P.ny;
    const T* __restrict__ r0 = in + P.origin + (int64_t)i0 * P.pitch;
    const T* __restrict__ r1 = second ? r0 + P.pitch : r0;
    clear_gap<T, NT>(s, pl, ends >= kEndsND ? N : N + 1, ends >= kEndsND ? pl.M - N - 1 : pl.M - N);
    for (int q = threadIdx.x; q <= N; q += NT) {
        const Cx<T> v = {r0[q], second ? r1[q] : (T)0};
        if (ends == kEndsNN) {
            put_at(s, pl, tab, q, v);
            if (q > 0 && q < N) put_at(s, pl, tab, pl.chirp ? -q : 2 * N - q, v);
        } else if (ends == kEndsDD) {
            put_at(s, pl, tab, q, (q > 0 && q < N) ? v : Cx<T>{(T)0, (T)0});
            if (q > 0 && q < N) put_at(s, pl, tab, pl.chirp ? -q : 2 * N - q, Cx<T>{-v.x, -v.y});
        } else if (q < N) {
            put_at(s, pl, tab, q, v);
            put_at(s, pl, tab, pl.chirp ? -q - 1 : 2 * N - 1 - q, v);
        }
    }
    double* __restrict__ xr = x + P.origin + (int64_t)i0 * P.pitch;
    const int pitch = P.pitch;
    const bool held0 = i0 == 0 && (P.dmask & (1 << kBottom)), held1 = i0 + 1 == P.ny && (P.dmask & (1 << kTop));
    const bool top0 = i0 == P.ny && (P.dmask & (1 << kTop));
    [[maybe_unused]] double* __restrict__ dr = GEN ? d + P.origin + (int64_t)i0 * P.pitch : nullptr;
    [[maybe_unused]] double al = 1.0, be = 0.0;
    if constexpr (GEN) {
        const double2 w = cheb[(int64_t)job.prob * kChebMax + min(app, kChebMax - 1)];
        al = ldexp(w.x, up);
        be = w.y;
    }
    const int jlo = (P.dmask & (1 << kLeft)) ? 1 : 0, jhi = (P.dmask & (1 << kRight)) ? N - 1 : N;
    double acc[2] = {0.0, 0.0};
    row_transform<T, NT, V>(s, pl, tab, [&](int jj, Cx<T> v) {
        const int j = ends == kEndsDN ? N - jj : jj;
        if (ends == kEndsDD)
            v = Cx<T>{-v.y, v.x};
        else if (ends >= kEndsND)
            v = mul(v, tab[pl.quart + jj]);
        if (j < jlo || j > jhi) return;
        double v0 = (double)v.x, v1 = (double)v.y;
        if constexpr (GEN) {
            v0 *= al;
            v1 *= al;
            if (app > 0) {
                v0 += be * dr[j];
                if (second) v1 += be * dr[j + pitch];
            }
            dr[j] = v0;
            if (second) dr[j + pitch] = v1;
        }
        if (!held0 && !top0) {
            xr[j] += GEN || sizeof(T) == 8 ? v0 : ldexp(v0, up);
            acc[0] += v0 * v0;
        }
        if (second && !held1) {
            xr[j + pitch] += GEN || sizeof(T) == 8 ? v1 : ldexp(v1, up);
            acc[1] += v1 * v1;
        }
    });
    block_pair<NT>(acc);
    if (threadIdx.x == 0) partial[3 * (int64_t)(f.pair0 + job.at) + 2] = GEN ? acc[0] + acc[1] : ldexp(acc[0] + acc[1], 2 * up);
}

// ------------------------------------------------------------ launches

template <typename F>
inline void by_threads(int nt, F&& f)
{
    switch (nt) {
    case 64: f(std::integral_constant<int, 64>{}); break;
    case 128: f(std::integral_constant<int, 128>{}); break;
    case 256: f(std::integral_constant<int, 256>{}); break;
    case 512: f(std::integral_constant<int, 512>{}); break;
    case 1024: f(std::integral_constant<int, 1024>{}); break;
    default: f(std::integral_constant<int, 2048>{}); break;
    }
}

// one application's forward and backward transforms, class by class, and the
// LDS their kernels may use
template <typename T, bool GEN>
void fast_forward(eq_batch* b, int k, bool start);
template <typename T, bool GEN>
void fast_backward(eq_batch* b, int k);
template <typename T, bool GEN>
int fast_allow_lds(const FastSolver* F);

inline int grid8(int n) { return 8 * ((n + 7) / 8); }

} // namespace eqk
