// eq_fast.hip -- the constant-coefficient field step by a fast direct solver.
//
// With constant coefficients the P1 operator on the uniform "right"-diagonal
// mesh is separable but for one term: the stiffness is Kx (x) Ly + Lx (x) Ky
// with trapezoidal L, the consistent mass couples the SW and NE neighbours
// where a separable matrix would spread that weight over all four diagonal
// ones.  That difference is of relative size h^2 / (12 dt D): it acts like a
// mixed derivative of that strength.  So the separable matrix P is inverted
// exactly and the step is
//     x <- x + P^-1 (b - A x),      b = M u + sources,
// whose error falls by about h^2 / (12 dt D) a time (1e-4 to 1e-6 on the grids
// the step meets: two to four applications from the last step's solution,
// where the V-cycle needed nine to ten iterations of five times the cost).
// The residual b - A x is formed in FP64 from u and x themselves every time,
// so the stop test is on the true residual and nothing is carried along.
// The finite-difference scheme is separable exactly.
//
// Measured per time step, couple + solve + fields out, against the V-cycle
// CG: 2000x1000, 2 species 2.58 -> 0.40 ms (FP64 3.04 -> 0.46), 1237x611 (a
// chirp length) 2.02 -> 0.34, 12 uneven traps 3.32 -> 1.02, 512 uneven traps
// 69.4 -> 28.0; errors against a 64-bit solve 4e-15 to 6e-13.
//
// What bounds the transforms: vector issue and latency, not bandwidth
// (2000x1000: forward 34 us, backward 28, where the bytes take 18 and 14).
// They are compiled for 64 registers, eight waves a SIMD: at 82 to 119
// registers the same launch took two rounds of blocks and 59 and 34 us.
//
// P^-1: trigonometric transform along x (the eigenvectors of the x matrices:
// cosines for closed walls, sines for held ones, quarter-wave cosines for one
// of each), one tridiagonal solve along y per mode (which also carries Robin
// walls), transform back.  Three launches an application:
//   k_fast_forward   two rows a block: their residual (read through the
//                    caches from u and x), packed as one complex row,
//                    extended to period 2 nx, transformed in LDS
//   k_fast_lines     16 modes a block: all rows of a mode in registers, the
//                    two one-sided recursions of the tridiagonal inverse
//   k_fast_backward  two rows a block: transformed back in LDS, added to x
// Lengths whose factors are 2, 3, 5 and 7 take a Stockham transform of 2 nx
// points; the others Bluestein's chirp convolution (Bluestein, IEEE Trans.
// Audio Electroacoust. 18, 1970) on the next such length of at least 3 nx + 1.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
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
constexpr int kFastGiveUp = 32;       // applications before the multigrid solver takes over

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
    void* d_tables = nullptr;
    double* d_partial = nullptr; // 2 per row pair
    int recent[4] = {3, 3, 3, 3}; // application counts of the last solves
    int at = 0;
    static constexpr int kGraphs = 9;
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
    __device__ __forceinline__ double rhs_inner(double mc, double mo, int k) const
    {
        return mc * m[k + 1] + mo * (((w[k + 1] + e[k]) + (m[k] + m[k + 2])) + (w[k] + e[k + 1]));
    }
};

// Rows i0 and i0 + 1 of the residual b - A x, b = M u + sources, column by
// column; f(j, r0, r1) takes them (0 on held nodes, where x holds the wall
// value).  Sums r^2, and with want_b the row-replaced b^2, into acc.
template <int NT, typename F>
__device__ __forceinline__ void residual_pair(const LevelProb& P, const FastRows& tab, int i0,
                                              const double* __restrict__ u, const double* __restrict__ x, bool want_b,
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
        double r0 = b0 - X.apply(tab.a[c0][cc], 0), r1 = in1 ? b1 - X.apply(tab.a[c1][cc], 1) : 0.0;
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
#pragma unroll 1
        for (int j = 1 + (int)threadIdx.x; j < nx; j += NT) {
            PairWindow U, X;
            U.load(ur, j, row);
            X.load(xr, j, row);
            const double b0 = U.rhs_inner(c0, c1, 0) + cs, b1 = U.rhs_inner(c0, c1, 1) + cs;
            const double r0 = b0 - X.apply_inner(mc, mo, kx, ky, 0), r1 = b1 - X.apply_inner(mc, mo, kx, ky, 1);
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
template <typename T, int NT, int V>
__global__ __launch_bounds__(NT, fast_waves(sizeof(T), NT, V)) void k_fast_forward(const FastJob* __restrict__ jobs, int njobs,
                                                     const LevelProb* __restrict__ probs,
                                                     const FastProb* __restrict__ fp, const FastRows* __restrict__ rows,
                                                     const FastPlan* __restrict__ plans, const Cx<T>* __restrict__ tab,
                                                     const double* __restrict__ u,
                                                     const double* __restrict__ x, T* __restrict__ out,
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
    clear_gap<T, NT>(s, pl, N + 1, pl.M - N);
    residual_pair<NT>(P, rows[job.prob], i0, u, x, k == 0, acc, [&](int j, double r0, double r1) {
        Cx<T> v = {(T)r0, (T)r1};
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
        partial[2 * (int64_t)(f.pair0 + job.at)] = acc[0];
        partial[2 * (int64_t)(f.pair0 + job.at) + 1] = acc[1];
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

// The residual alone: the confirmation after a chunk of applications.
__global__ __launch_bounds__(256) void k_fast_check(const FastJob* __restrict__ jobs, int njobs,
                                                    const LevelProb* __restrict__ probs,
                                                    const FastProb* __restrict__ fp, const FastRows* __restrict__ rows,
                                                    const double* __restrict__ u, const double* __restrict__ x,
                                                    double* __restrict__ partial,
                                                    const CgState* __restrict__ st)
{
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    if (st[P.prob].done) return;
    double acc[2] = {0.0, 0.0};
    residual_pair<256>(P, rows[job.prob], 2 * job.at, u, x, false, acc, [](int, double, double) {});
    block_pair<256>(acc);
    if (threadIdx.x == 0) partial[2 * (int64_t)(fp[job.prob].pair0 + job.at)] = acc[0];
}

// Sums a problem's row-pair partials: the same order in every block of the
// launch.  Result in every thread.
__device__ __forceinline__ void sum_pairs(const double* __restrict__ partial, int npairs, double* red, double& rr,
                                          double& bb)
{
    double a = 0.0, b = 0.0;
    for (int q = threadIdx.x; q < npairs; q += blockDim.x) {
        a += partial[2 * q];
        b += partial[2 * q + 1];
    }
    a = wave_add(a);
    b = wave_add(b);
    const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[2 * w] = a;
        red[2 * w + 1] = b;
    }
    __syncthreads();
    rr = bb = 0.0;
    for (int q = 0; q < nw; ++q) {
        rr += red[2 * q];
        bb += red[2 * q + 1];
    }
}

__device__ __forceinline__ double ipow(double a, int n)
{
    double r = 1.0;
    for (; n > 0; n >>= 1) {
        if (n & 1) r *= a;
        a *= a;
    }
    return r;
}

// The tridiagonal solves along y, 16 modes a block, C chunks of rows each in
// the registers of one thread.  Per mode the matrix is (sigma + tau Lambda)
// with Lambda the second difference: its inverse on the whole line is
//   w = c (F + G),  F_i = rho F_(i-1) + f_i,  G_i = rho (G_(i+1) + f_(i+1)),
// c = 1 / (tau (1/rho - rho)), and a wall reflects: it adds A rho^i (bottom)
// and B rho^(ny - i) (top) with A = R0 (w_0 + B rho^ny), B = R1 (w_ny + A rho^ny),
// R = 1 for a closed wall, -1 for a held one and between for Robin.  All
// recursions decay, in FP64.  First every block takes its problem's residual
// norm from the row pairs' sums and stops where it converged.
template <typename T, int L>
__global__ void k_fast_lines(const FastJob* __restrict__ jobs, int njobs, const LevelProb* __restrict__ probs,
                             const FastProb* __restrict__ fp, T* __restrict__ io, const double* __restrict__ partial,
                             CgState* st, int k)
{
    extern __shared__ char lds_raw[];
    double* red = (double*)lds_raw;            // 32 doubles of sums, then the flag
    double* carry = red + 40;                  // [2][C][16] chunk ends
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    const FastProb f = fp[job.prob];
    CgState& cs = st[P.prob];
    const int m = threadIdx.x & (kFastModes - 1), c = threadIdx.x / kFastModes, C = blockDim.x / kFastModes;
    const int N = P.nx, ny = P.ny;
    const int rows = ny + 1, Lp = (rows + C - 1) / C; // rows of a chunk, <= L
    const int q = job.at * kFastModes + m;            // the mode
    const int a = c * Lp;
    const int nl = max(0, min(Lp, rows - a));
    const bool on = q <= N;
    T* __restrict__ col = io + P.origin + (int64_t)a * P.pitch + q;
    T v[L];
#pragma unroll
    for (int l = 0; l < L; ++l) v[l] = (on && l < nl) ? col[(int64_t)l * P.pitch] : (T)0;
    if (threadIdx.x == 0) ((int*)(red + 36))[0] = k > 0 ? cs.done : 0;
    double rr, bb;
    sum_pairs(partial + 2 * (int64_t)f.pair0, f.npairs, red, rr, bb);
    if (((int*)(red + 36))[0]) return;
    if (k > 0) bb = cs.bb;
    const bool conv = rr <= cs.tol2 * bb, stop = conv || k >= cs.max_iter;
    if (job.at == 0 && threadIdx.x == 0) {
        if (k == 0) cs.bb = bb;
        cs.done = stop ? 1 : 0;
        if (stop) {
            cs.fast_iter = k;
            cs.rr_true = rr;
        }
    }
    if (stop) return;
    // the mode's matrix
    const bool half = f.ends >= kEndsND;
    const double cx = cospi((half ? q + 0.5 : (double)q) / N), lx = 2.0 * (1.0 - cx);
    double sigma, tau, k0 = 0.0, k1 = 0.0;
    if (P.fd) {
        sigma = P.fdm + P.fkx * lx;
        tau = P.fky;
        k0 = P.frob[kBottom];
        k1 = P.frob[kTop];
    } else {
        const double ms = 12.0 * P.mh;
        sigma = ms * (2.0 + cx) / 3.0 + 2.0 * P.sa * lx;
        tau = 2.0 * P.sb - ms * (1.0 + cx) / 12.0;
        k0 = P.rob[kBottom] * 2.0 * (2.0 + cx) / 3.0;
        k1 = P.rob[kTop] * 2.0 * (2.0 + cx) / 3.0;
    }
    const double sh = sigma / tau;
    const double rho = 1.0 / (1.0 + 0.5 * sh + sqrt(sh + 0.25 * sh * sh));
    const double del = 1.0 / rho - rho;
    const double R0 = (P.dmask & (1 << kBottom)) ? -1.0 : (del - k0 / tau) / (del + k0 / tau);
    const double R1 = (P.dmask & (1 << kTop)) ? -1.0 : (del - k1 / tau) / (del + k1 / tau);
    const double scale = 1.0 / (tau * del * 2.0 * N); // both transforms' factors with it
    // chunk ends from zero carries: F at the chunk's last row, G before its first
    double F = 0.0, G = 0.0;
#pragma unroll
    for (int l = 0; l < L; ++l)
        if (l < nl) F = rho * F + (double)v[l];
#pragma unroll
    for (int l = L - 1; l >= 0; --l)
        if (l < nl) G = rho * (G + (double)v[l]);
    double* cF = carry + c * kFastModes + m;
    double* cG = cF + C * kFastModes;
    *cF = F;
    *cG = G;
    __syncthreads();
    // carries across the chunks: a thread per mode up, another down
    if (threadIdx.x < 2 * kFastModes) {
        const int mm = threadIdx.x & (kFastModes - 1);
        const double w = ipow(rho, Lp); // (a thread's own mode is mm)
        double* p = carry + mm + (threadIdx.x < kFastModes ? 0 : C * kFastModes);
        double in = 0.0;
        if (threadIdx.x < kFastModes) {
            for (int e = 0; e < C; ++e) {
                const double own = p[e * kFastModes];
                p[e * kFastModes] = in;
                in = w * in + own;
            }
        } else {
            for (int e = C - 1; e >= 0; --e) {
                const double own = p[e * kFastModes];
                p[e * kFastModes] = in;
                in = w * in + own; // rows past the last are zero: their chunk's power only scales zero
            }
        }
    }
    __syncthreads();
    // w on the whole line at the two walls (in units of c): bottom f_0 + G_0,
    // top F_ny; their threads publish them
    double* ends = red; // [2][16]
    F = *cF;
    G = *cG;
    if (a == 0) {
        double g = G;
#pragma unroll
        for (int l = L - 1; l >= 1; --l)
            if (l < nl) g = rho * (g + (double)v[l]);
        ends[m] = (double)v[0] + g;
    }
    if (nl > 0 && a + nl == rows) {
        double e = F;
#pragma unroll
        for (int l = 0; l < L; ++l)
            if (l < nl) e = rho * e + (double)v[l];
        ends[kFastModes + m] = e;
    }
    __syncthreads();
    if (!on || nl == 0) return;
    const double pn = ipow(rho, ny);
    const double w0 = ends[m], wn = ends[kFastModes + m];
    const double A = R0 * (w0 + pn * R1 * wn) / (1.0 - R0 * R1 * pn * pn);
    const double B = R1 * (wn + pn * A);
    // the walls' terms ride on the recursions' carries: F gets A rho^i, G gets B rho^(ny - i)
    F += A * ipow(rho, a) / rho;                     // at row a - 1
    G += B * ipow(rho, rows - (a + nl));             // at the chunk's last row
    // both directions through the registers: G_i kept, then F_i + G_i
    T g[L];
#pragma unroll
    for (int l = L - 1; l >= 0; --l)
        if (l < nl) {
            g[l] = (T)G;
            G = rho * (G + (double)v[l]);
        }
#pragma unroll
    for (int l = 0; l < L; ++l)
        if (l < nl) {
            F = rho * F + (double)v[l];
            col[(int64_t)l * P.pitch] = (T)(scale * (F + (double)g[l]));
        }
}

// Transform back along x and x += z, two rows a block.
template <typename T, int NT, int V>
__global__ __launch_bounds__(NT, fast_waves(sizeof(T), NT, V)) void k_fast_backward(const FastJob* __restrict__ jobs, int njobs,
                                                      const LevelProb* __restrict__ probs,
                                                      const FastProb* __restrict__ fp,
                                                      const FastPlan* __restrict__ plans,
                                                      const Cx<T>* __restrict__ tab, const T* __restrict__ in,
                                                      double* __restrict__ x, const CgState* __restrict__ st)
{
    extern __shared__ char lds_raw[];
    Cx<T>* s = (Cx<T>*)lds_raw;
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    const CgState& cs = st[P.prob];
    if (cs.done) return;
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
    const int jlo = (P.dmask & (1 << kLeft)) ? 1 : 0, jhi = (P.dmask & (1 << kRight)) ? N - 1 : N;
    row_transform<T, NT, V>(s, pl, tab, [&](int jj, Cx<T> v) {
        const int j = ends == kEndsDN ? N - jj : jj;
        if (ends == kEndsDD)
            v = Cx<T>{-v.y, v.x};
        else if (ends >= kEndsND)
            v = mul(v, tab[pl.quart + jj]);
        if (j < jlo || j > jhi) return;
        if (!held0 && !top0) xr[j] += (double)v.x;
        if (second && !held1) xr[j + pitch] += (double)v.y;
    });
}

// The chunk's end: every block takes its problem's residual norm, and where
// the solve is over (converged or out of iterations) the iterate becomes the
// field.  The first block of a problem keeps its state.
__global__ __launch_bounds__(256) void k_fast_commit(const FastJob* __restrict__ jobs, int njobs,
                                                     const LevelProb* __restrict__ probs,
                                                     const FastProb* __restrict__ fp, double* __restrict__ u,
                                                     const double* __restrict__ x, const double* __restrict__ partial,
                                                     CgState* st, int k)
{
    __shared__ double red[16];
    __shared__ int was;
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    const FastProb f = fp[job.prob];
    CgState& cs = st[P.prob];
    if (threadIdx.x == 0) was = cs.done;
    double rr, bb;
    sum_pairs(partial + 2 * (int64_t)f.pair0, f.npairs, red, rr, bb);
    if (was == 2) return;
    // (a block that already reads the first block's `done` takes the same way)
    const bool conv = rr <= cs.tol2 * cs.bb, over = was || conv || k >= cs.max_iter;
    if (job.at == 0 && threadIdx.x == 0) {
        if (!was) {
            cs.fast_iter = k;
            cs.rr_true = rr;
        }
        cs.rr = cs.rr_true;
        cs.iter = cs.fast_iter;
        if (over) {
            cs.done = 1;
            cs.have_prev = 1;
        }
    }
    if (!over) return;
    for (int w = 0; w < 2; ++w) {
        const int i = 2 * job.at + w;
        if (i > P.ny) break;
        const int64_t r = P.origin + (int64_t)i * P.pitch;
        for (int j = threadIdx.x; j <= P.nx; j += 256) u[r + j] = x[r + j];
    }
}

// A solve's start: the iterate takes the wall values on held nodes, and zero
// elsewhere where no solution is kept.
__global__ __launch_bounds__(256) void k_fast_start(const FastJob* __restrict__ jobs, int njobs,
                                                    const LevelProb* __restrict__ probs, double* __restrict__ x,
                                                    const CgState* __restrict__ st)
{
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    const bool kept = st[P.prob].have_prev != 0;
    for (int w = 0; w < 2; ++w) {
        const int i = 2 * job.at + w;
        if (i > P.ny) break;
        const int64_t r = P.origin + (int64_t)i * P.pitch;
        const bool wall = (i == 0 && (P.dmask & (1 << kBottom))) || (i == P.ny && (P.dmask & (1 << kTop)));
        if (kept && !wall) {
            // two columns at most
            const int j = threadIdx.x == 0 ? 0 : P.nx;
            if (threadIdx.x < 2 && is_dirichlet(P, i, j)) x[r + j] = dirichlet_value(P, i, j);
            continue;
        }
        for (int j = threadIdx.x; j <= P.nx; j += 256)
            x[r + j] = is_dirichlet(P, i, j) ? dirichlet_value(P, i, j) : 0.0;
    }
}

// tables: exp(-2 pi i k / M), exp(-pi i j / 2N), the chirp and its kernel
template <typename T>
__global__ void k_fast_tables(const FastPlan* __restrict__ plans, Cx<T>* __restrict__ tab)
{
    const FastPlan& pl = plans[blockIdx.x];
    const int at = blockIdx.y * blockDim.x + threadIdx.x, step = gridDim.y * blockDim.x;
    double sn, cs;
    for (int k = at; k < pl.M; k += step) {
        sincospi(-2.0 * k / pl.M, &sn, &cs);
        tab[pl.tw + k] = {(T)cs, (T)sn};
    }
    for (int k = at; k <= pl.N; k += step) {
        sincospi(-0.5 * k / pl.N, &sn, &cs);
        tab[pl.quart + k] = {(T)cs, (T)sn};
    }
    if (!pl.chirp) return;
    for (int k = at; k < pl.n; k += step) {
        const int64_t q = ((int64_t)k * k) % (2 * (int64_t)pl.n);
        sincospi(-(double)q / pl.n, &sn, &cs);
        tab[pl.ch + k] = {(T)cs, (T)sn};
    }
}
template <typename T, int NT, int V>
__global__ __launch_bounds__(NT) void k_fast_kernel(const FastPlan* __restrict__ plans, Cx<T>* __restrict__ tab)
{
    extern __shared__ char lds_raw[];
    Cx<T>* s = (Cx<T>*)lds_raw;
    const FastPlan& pl = plans[blockIdx.x];
    if (!pl.chirp) return;
    // conj(chirp) at -N .. 2N, which M >= 3N + 1 keeps apart
    for (int k = threadIdx.x; k < pl.M; k += NT) {
        const int d = k <= 2 * pl.N ? k : k - pl.M;
        Cx<T> v = {(T)0, (T)0};
        if (d >= -pl.N) {
            const int e = (d < 0 ? -d : d) % pl.n;
            v = tab[pl.ch + e];
            v.y = -v.y;
        }
        s[k] = v;
    }
    __syncthreads();
    const T r = (T)(1.0 / pl.M);
    Cx<T>* h = tab + pl.hh;
    fft_lds<T, NT, V>(s, pl, tab, [&](int k, Cx<T> v) { h[k] = {v.x * r, v.y * r}; });
}

// ------------------------------------------------------------ host: which batches, plans

// Passes of an M-point transform: as few as factors of at most 10 allow, odd
// and singly even radices first (their strided LDS writes spread over the
// banks; radix 8 first would put a wave on four of them).  False where M has
// a prime factor above 7.
static bool smooth_factors(int M, FastPlan& pl)
{
    int c[4] = {0, 0, 0, 0}, rest = M;
    const int primes[4] = {2, 3, 5, 7};
    for (int k = 0; k < 4; ++k)
        while (rest % primes[k] == 0) {
            rest /= primes[k];
            ++c[k];
        }
    if (rest != 1) return false;
    int& two = c[0];
    std::vector<int> odd, even;
    for (; c[3]; --c[3]) odd.push_back(7);
    for (; c[1] >= 2; c[1] -= 2) odd.push_back(9);
    // pair fives (and a last three) with twos while that leaves the twos in
    // eights and fours
    for (; c[2]; --c[2]) {
        const bool pair = two % 3 == 1 || (two > 0 && c[2] > 1) || (two % 3 == 2 && two > 2) || two == 1;
        odd.push_back(pair && two > 0 ? (--two, 10) : 5);
    }
    if (c[1]) odd.push_back(two % 3 == 1 ? (--two, 6) : 3);
    for (; two > 4 || two == 3; two -= 3) even.push_back(8);
    for (; two > 1; two -= 2) even.push_back(4);
    if (two) (odd.empty() ? odd : even).push_back(2);
    std::sort(odd.rbegin(), odd.rend());
    odd.insert(odd.end(), even.begin(), even.end());
    if (odd.empty() || (int)odd.size() > kFastMaxStages) return false;
    pl.nstages = 0;
    int Ns = 1;
    for (int r : odd) {
        pl.pass[pl.nstages++] = FastPlan::Pass{r, M / r, Ns, M / r / Ns};
        Ns *= r;
    }
    return true;
}

static size_t fast_lds_bytes(int M, size_t elem) { return (size_t)M * elem; }

// the plan of rows of N cells, or false where they do not fit a block
static bool make_plan(int N, size_t elem, FastPlan& pl)
{
    std::memset(&pl, 0, sizeof(pl));
    pl.N = N;
    pl.n = 2 * N;
    pl.M = pl.n;
    if (!smooth_factors(pl.n, pl)) {
        // the chirp's length: the cheapest (passes times points) up to an
        // eighth above the least
        pl.chirp = 1;
        FastPlan best{};
        for (int M = 3 * N + 1; best.M == 0 || M <= (3 * N + 1) + (3 * N + 1) / 8; ++M) {
            FastPlan t = pl;
            if (!smooth_factors(M, t)) continue;
            t.M = M;
            if (best.M == 0 || (int64_t)t.M * t.nstages < (int64_t)best.M * best.nstages) best = t;
        }
        pl = best;
    }
    return pl.M <= kFastValuesWide * 1024 && (int64_t)fast_lds_bytes(pl.M, elem) <= kFastLds;
}

// Whether the batch's grids and walls allow the solver: x walls closed or
// held (their transforms diagonalise the x matrices), rows that fit a block,
// and dt D of at least the square of the larger spacing, where the
// separable matrix is within a tenth of the operator.
static bool fast_shape(const eq_batch* b)
{
    const size_t elem = b->mixed ? sizeof(Cx<float>) : sizeof(Cx<double>);
    std::map<int, bool> fits;
    for (const eq_field_desc& d : b->descs) {
        for (int w : {EQ_WALL_LEFT, EQ_WALL_RIGHT})
            if (d.wall[w].kind == EQ_BC_ROBIN) return false;
        if (d.ny + 1 > kFastRowsMax || d.nx > (1 << 15)) return false;
        const double hx = d.width / d.nx, hy = d.height / d.ny, h = std::max(hx, hy);
        if (!(d.dt * d.D >= (1.0 + d.dt * d.gamma) * h * h) || h > 4.0 * std::min(hx, hy)) return false;
        auto it = fits.find(d.nx);
        if (it == fits.end()) {
            FastPlan pl;
            it = fits.emplace(d.nx, make_plan(d.nx, elem, pl)).first;
        }
        if (!it->second) return false;
    }
    return true;
}

void fast_free(eq_batch* b)
{
    FastSolver* F = b->fast;
    if (!F) return;
    for (hipGraphExec_t g : F->graph)
        if (g) hipGraphExecDestroy(g);
    hipFree(F->d_plans);
    hipFree(F->d_probs);
    hipFree(F->d_rows);
    hipFree(F->d_jobs);
    hipFree(F->d_lines);
    hipFree(F->d_tables);
    hipFree(F->d_partial);
    delete F;
    b->fast = nullptr;
}

void fast_drop_graphs(eq_batch* b)
{
    if (!b->fast) return;
    for (hipGraphExec_t& g : b->fast->graph) {
        if (g) hipGraphExecDestroy(g);
        g = nullptr;
    }
}

template <typename V>
static int put_table(V** d, const std::vector<V>& h, hipStream_t s)
{
    if (hipMalloc((void**)d, sizeof(V) * std::max<size_t>(1, h.size())) != hipSuccess)
        return set_error(EQ_ERR_NOMEM, "fast solver tables");
    EQ_HIP(hipMemcpyAsync(*d, h.data(), sizeof(V) * h.size(), hipMemcpyHostToDevice, s));
    return EQ_OK;
}

template <typename F>
static void by_threads(int nt, F&& f)
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

template <typename T>
static int allow_lds()
{
    int rc = EQ_OK;
    for (int nt = 64; nt <= 2048; nt *= 2)
        by_threads(nt, [&](auto c) {
            constexpr int NT = std::min(1024, decltype(c)::value), V = decltype(c)::value / NT * kFastValues;
            if (hipFuncSetAttribute((const void*)k_fast_forward<T, NT, V>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)kFastLds) != hipSuccess ||
                hipFuncSetAttribute((const void*)k_fast_backward<T, NT, V>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)kFastLds) != hipSuccess)
                rc = set_error(EQ_ERR_HIP, "hipFuncSetAttribute");
        });
    return rc;
}

template <typename T>
static int fast_build_t(eq_batch* b, FastSolver* F)
{
    hipStream_t s = b->stream;
    std::vector<FastPlan> plans;
    std::map<int, int> plan_of;
    std::vector<FastProb> fp(b->nprob);
    std::vector<FastRows> rows9(b->nprob);
    std::vector<int> thr(b->nprob);
    int64_t tab = 0;
    int32_t pairs = 0;
    int rows = 0, mmax = 1;
    for (int p = 0; p < b->nprob; ++p) {
        const LevelProb& P = b->levels[0].probs[p];
        auto it = plan_of.find(P.nx);
        if (it == plan_of.end()) {
            FastPlan pl;
            make_plan(P.nx, sizeof(Cx<T>), pl);
            pl.tw = tab;
            tab += pl.M;
            pl.quart = tab;
            tab += pl.N + 1;
            if (pl.chirp) {
                pl.ch = tab;
                tab += pl.n;
                pl.hh = tab;
                tab += pl.M;
                mmax = std::max(mmax, pl.M);
            }
            it = plan_of.emplace(P.nx, (int)plans.size()).first;
            plans.push_back(pl);
        }
        const bool l = P.dmask & (1 << kLeft), r = P.dmask & (1 << kRight);
        fp[p].plan = it->second;
        fp[p].ends = l ? (r ? kEndsDD : kEndsDN) : (r ? kEndsND : kEndsNN);
        fp[p].pair0 = pairs;
        fp[p].npairs = (P.ny + 2) / 2;
        pairs += fp[p].npairs;
        rows = std::max(rows, P.ny + 1);
        for (int ci = 0; ci < 3; ++ci)
            for (int cj = 0; cj < 3; ++cj) {
                const int i = ci == 0 ? 0 : ci == 1 ? 1 : P.ny, j = cj == 0 ? 0 : cj == 1 ? 1 : P.nx;
                rows9[p].a[ci][cj] = row_coefs_at<double>(P, i, j);
                double v[8] = {0, 0, 0, 0, 0, 0, 0, 0}, *o = rows9[p].b[ci][cj];
                o[7] = rhs_row(P, i, j, 0, 0, 0, 0, 0, 0, 0);
                for (int q = 0; q < 7; ++q) {
                    v[q] = 1.0;
                    o[q] = rhs_row(P, i, j, v[0], v[1], v[2], v[3], v[4], v[5], v[6]) - o[7];
                    v[q] = 0.0;
                }
            }
        int nt = 64;
        while (kFastValues * nt < plans[it->second].M && nt < 2048) nt *= 2;
        thr[p] = nt; // 2048: 1024 threads of twice the values
    }
    std::vector<FastJob> jobs, lines;
    for (int nt = 64; nt <= 2048; nt *= 2) {
        FastClass c;
        c.threads = nt;
        c.job0 = (int32_t)jobs.size();
        for (int p = 0; p < b->nprob; ++p) {
            if (thr[p] != nt) continue;
            const LevelProb& P = b->levels[0].probs[p];
            c.lds = std::max(c.lds, fast_lds_bytes(plans[fp[p].plan].M, sizeof(Cx<T>)));
            c.nodes += (double)(P.nx + 1) * (P.ny + 1);
            for (int q = 0; q < fp[p].npairs; ++q) jobs.push_back(FastJob{p, q});
        }
        c.njobs = (int32_t)jobs.size() - c.job0;
        if (c.njobs) F->classes.push_back(c);
    }
    for (int p = 0; p < b->nprob; ++p)
        for (int q = 0; q * kFastModes <= b->levels[0].probs[p].nx; ++q) lines.push_back(FastJob{p, q});
    F->nline = (int32_t)lines.size();
    F->line_rows = rows;
    // chunks of at most 16 rows a thread up to 1024 rows, then longer ones
    const int L = rows <= 1024 ? 16 : rows <= 2048 ? 32 : 64;
    F->line_c = std::max(4, (rows + L - 1) / L);
    F->line_c = (F->line_c + 3) / 4 * 4; // whole waves
    int rc;
    if ((rc = put_table(&F->d_plans, plans, s)) || (rc = put_table(&F->d_probs, fp, s)) ||
        (rc = put_table(&F->d_rows, rows9, s)) ||
        (rc = put_table(&F->d_jobs, jobs, s)) || (rc = put_table(&F->d_lines, lines, s)))
        return rc;
    if (hipMalloc(&F->d_tables, sizeof(Cx<T>) * tab) != hipSuccess ||
        hipMalloc((void**)&F->d_partial, sizeof(double) * 2 * pairs) != hipSuccess)
        return set_error(EQ_ERR_NOMEM, "fast solver tables");
    const int np = (int)plans.size();
    hipLaunchKernelGGL(k_fast_tables<T>, dim3(np, 4), dim3(256), 0, s, F->d_plans, (Cx<T>*)F->d_tables);
    if (mmax > 1) {
        const size_t lds = fast_lds_bytes(mmax, sizeof(Cx<T>));
        EQ_HIP(hipFuncSetAttribute((const void*)k_fast_kernel<T, 1024, kFastValuesWide>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFastLds));
        hipLaunchKernelGGL((k_fast_kernel<T, 1024, kFastValuesWide>), dim3(np), dim3(1024), lds, s, F->d_plans, (Cx<T>*)F->d_tables);
    }
    EQ_HIP(hipGetLastError());
    EQ_HIP(hipStreamSynchronize(s)); // the host tables above go out of scope
    return allow_lds<T>();
}

int fast_build(eq_batch* b)
{
    const eq_solver_desc& S = b->solver;
    if (S.kind != EQ_SOLVER_GMG_CG && S.kind != EQ_SOLVER_MIXED_GMG_CG) return EQ_OK;
    if (!fast_shape(b)) return EQ_OK;
    b->fast = new (std::nothrow) FastSolver();
    if (!b->fast) return set_error(EQ_ERR_NOMEM, "host allocation");
    return b->mixed ? fast_build_t<float>(b, b->fast) : fast_build_t<double>(b, b->fast);
}

// Whether this step takes the fast solver: constant coefficients, and the
// cycle options at their defaults (a caller that sets them asks for that
// multigrid cycle).
bool fast_applies(const eq_batch* b)
{
    if (!b->fast || b->any_tensor) return false;
    eq_solver_desc d;
    eq_solver_default(&d);
    const eq_solver_desc& S = b->solver;
    return S.mg_pre == d.mg_pre && S.mg_post == d.mg_post && S.mg_omega == d.mg_omega && S.mg_omega2 == d.mg_omega2 &&
           S.mg_coarse_max_nodes == d.mg_coarse_max_nodes && S.mg_max_levels == d.mg_max_levels &&
           S.mg_fuse_max_nodes == d.mg_fuse_max_nodes && S.mg_fuse_pre_max_nodes == d.mg_fuse_pre_max_nodes &&
           S.mg_bottom_lds_bytes == d.mg_bottom_lds_bytes && S.mg_fuse_pre_top == d.mg_fuse_pre_top &&
           S.tile4_min_nodes == d.tile4_min_nodes && S.tile8_min_nodes == d.tile8_min_nodes &&
           S.extrapolate == d.extrapolate && S.mg_level_fused == d.mg_level_fused;
}

// ------------------------------------------------------------ host: one solve

static int grid8(int n) { return 8 * ((n + 7) / 8); }

// Applications k0 .. k0 + n - 1, then the residual's check and the commit.
template <typename T>
static void fast_chunk(eq_batch* b, int k0, int n)
{
    FastSolver* F = b->fast;
    hipStream_t s = b->stream;
    const LevelProb* probs = b->levels[0].d_probs;
    const Cx<T>* tab = (const Cx<T>*)F->d_tables;
    T* z = (T*)b->z;
    const double nodes = b->levels[0].nodes_all;
    const size_t lds = sizeof(double) * (40 + 2 * (size_t)F->line_c * kFastModes);
    int32_t njobs = 0;
    for (const FastClass& c : F->classes) njobs += c.njobs;
    if (k0 == 0)
        launch(b, EQ_KERNEL_SOLVE_ONCE, 0.0, k_fast_start, dim3(grid8(njobs)), dim3(256), 0, s,
               (const FastJob*)F->d_jobs, njobs, probs, b->xprev, (const CgState*)b->d_state);
    for (int k = k0; k < k0 + n; ++k) {
        for (const FastClass& c : F->classes)
            by_threads(c.threads, [&](auto t) {
                constexpr int NT = std::min(1024, decltype(t)::value), V = decltype(t)::value / NT * kFastValues;
                launch(b, EQ_KERNEL_STENCIL64, c.nodes * (16.0 + sizeof(T)), k_fast_forward<T, NT, V>, dim3(grid8(c.njobs)),
                       dim3(NT), c.lds, s, (const FastJob*)F->d_jobs + c.job0, c.njobs, probs,
                       (const FastProb*)F->d_probs, (const FastRows*)F->d_rows, (const FastPlan*)F->d_plans, tab,
                       (const double*)b->u, (const double*)b->xprev, z, F->d_partial, b->d_state, k, k == k0 ? 1 : 0);
            });
        const dim3 lg(grid8(F->nline)), lb(F->line_c * kFastModes);
        auto lines = [&](auto kern) {
            launch(b, EQ_KERNEL_BOTTOM, nodes * 2 * sizeof(T), kern, lg, lb, lds, s, (const FastJob*)F->d_lines, F->nline,
                   probs, (const FastProb*)F->d_probs, z, (const double*)F->d_partial, b->d_state, k);
        };
        if (F->line_rows <= 1024)
            lines(k_fast_lines<T, 16>);
        else if (F->line_rows <= 2048)
            lines(k_fast_lines<T, 32>);
        else
            lines(k_fast_lines<T, 64>);
        for (const FastClass& c : F->classes)
            by_threads(c.threads, [&](auto t) {
                constexpr int NT = std::min(1024, decltype(t)::value), V = decltype(t)::value / NT * kFastValues;
                launch(b, EQ_KERNEL_CG_UPDATE, c.nodes * (16.0 + sizeof(T)), k_fast_backward<T, NT, V>,
                       dim3(grid8(c.njobs)), dim3(NT), c.lds, s, (const FastJob*)F->d_jobs + c.job0, c.njobs, probs,
                       (const FastProb*)F->d_probs, (const FastPlan*)F->d_plans, tab, (const T*)z, b->xprev,
                       (const CgState*)b->d_state);
            });
    }
    launch(b, EQ_KERNEL_SOLVE_ONCE, nodes * 16.0, k_fast_check, dim3(grid8(njobs)), dim3(256), 0, s,
           (const FastJob*)F->d_jobs, njobs, probs, (const FastProb*)F->d_probs, (const FastRows*)F->d_rows,
           (const double*)b->u, (const double*)b->xprev, F->d_partial, (const CgState*)b->d_state);
    launch(b, EQ_KERNEL_SOLVE_ONCE, nodes * 16.0, k_fast_commit, dim3(grid8(njobs)), dim3(256), 0, s,
           (const FastJob*)F->d_jobs, njobs, probs, (const FastProb*)F->d_probs, b->u, (const double*)b->xprev,
           (const double*)F->d_partial, b->d_state, k0 + n);
}

// One step's solve.  handled = false: the residual did not reach the tolerance
// in kFastGiveUp applications and iterations are left; the multigrid solver
// then continues from the kept iterate (the problems already solved are
// listed in `solved`, their fields final).
template <typename T>
static int fast_solve_t(eq_batch* b, bool profiling, bool* handled)
{
    FastSolver* F = b->fast;
    const eq_solver_desc& S = b->solver;
    hipStream_t s = b->stream;
    *handled = true;
    const bool graphs = S.use_graphs && !profiling;
    int chunk = *std::max_element(F->recent, F->recent + 4);
    chunk = std::max(1, std::min({chunk, S.max_iter, FastSolver::kGraphs - 1}));
    for (int k0 = 0;;) {
        if (k0 == 0 && graphs) {
            hipGraphExec_t& ge = F->graph[chunk];
            if (!ge) {
                hipGraph_t g = nullptr;
                EQ_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                F->acct[chunk] = Acct{};
                b->acct_to = &F->acct[chunk];
                fast_chunk<T>(b, 0, chunk);
                b->acct_to = &b->acct;
                EQ_HIP(hipStreamEndCapture(s, &g));
                const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
                hipGraphDestroy(g);
                if (e != hipSuccess) {
                    ge = nullptr;
                    return hip_check(e, "hipGraphInstantiate");
                }
            }
            EQ_HIP(hipGraphLaunch(ge, s));
            replayed(b, F->acct[chunk]);
        } else {
            fast_chunk<T>(b, k0, chunk);
        }
        k0 += chunk;
        EQ_HIP(hipMemcpyAsync(b->h_state, b->d_state, sizeof(CgState) * b->nprob, hipMemcpyDeviceToHost, s));
        EQ_HIP(hipGetLastError());
        EQ_HIP(hipStreamSynchronize(s));
        bool all = true;
        for (int p = 0; p < b->nprob; ++p) all = all && b->h_state[p].done;
        if (all) break;
        if (k0 >= kFastGiveUp && k0 < S.max_iter) {
            *handled = false;
            return EQ_OK;
        }
        chunk = std::max(1, std::min(2, S.max_iter - k0));
    }
    int most = 1;
    for (int p = 0; p < b->nprob; ++p) most = std::max(most, b->h_state[p].iter);
    F->recent[F->at] = std::min(most, FastSolver::kGraphs - 1);
    F->at = (F->at + 1) & 3;
    return EQ_OK;
}

int fast_solve(eq_batch* b, bool profiling, bool* handled)
{
    return b->mixed ? fast_solve_t<float>(b, profiling, handled) : fast_solve_t<double>(b, profiling, handled);
}

} // namespace eqk
