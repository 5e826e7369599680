// eq_fast.hip -- the field step by a fast direct solver (varying coefficients
// and Robin walls across x: as the operator of a Chebyshev iteration, fast_refresh).
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
// so the stop test is on the true residual, and on the error that the last
// update shows (within).
// The finite-difference scheme is separable exactly.
//
// Measured per time step, couple + solve + fields out, against the V-cycle
// CG: 2000x1000, 2 species 2.57 -> 0.40 ms (FP64 3.04 -> 0.50), 1237x611 (a
// chirp length) 2.00 -> 0.41, 12 uneven traps 3.31 -> 1.12, 512 uneven traps
// 69.6 -> 31.6; errors against a 64-bit solve 1e-15 to 2e-14, where the CG
// left 2e-14 to 1e-12.
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
#include "eq_fast.h"

namespace eqk {

// The residual alone: the confirmation after a chunk of applications.
template <bool GEN>
__global__ __launch_bounds__(256) void k_fast_check(const FastJob* __restrict__ jobs, int njobs,
                                                    const LevelProb* __restrict__ probs,
                                                    const FastProb* __restrict__ fp, const FastRows* __restrict__ rows,
                                                    const double* __restrict__ u, const double* __restrict__ x,
                                                    const double* __restrict__ stiff, int64_t sst,
                                                    double* __restrict__ partial, const CgState* __restrict__ st)
{
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    if (st[P.prob].done) return;
    double acc[2] = {0.0, 0.0};
    residual_pair<256, GEN>(P, rows[job.prob], 2 * job.at, u, x, stiff, sst, false, acc, [](int, double, double) {});
    block_pair<256>(acc);
    if (threadIdx.x == 0) partial[3 * (int64_t)(fp[job.prob].pair0 + job.at)] = acc[0];
}

// Sums a problem's row-pair partials: the same order in every block of the
// launch.  Result in every thread.
__device__ __forceinline__ void sum_pairs(const double* __restrict__ partial, int npairs, double* red, double (&sum)[3])
{
    double v[3] = {0.0, 0.0, 0.0};
    for (int q = threadIdx.x; q < npairs; q += blockDim.x)
#pragma unroll
        for (int e = 0; e < 3; ++e) v[e] += partial[3 * q + e];
    const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        v[e] = wave_add(v[e]);
        if ((threadIdx.x & 63) == 0) red[3 * w + e] = v[e];
        sum[e] = 0.0;
    }
    __syncthreads();
    for (int q = 0; q < nw; ++q)
#pragma unroll
        for (int e = 0; e < 3; ++e) sum[e] += red[3 * q + e];
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

// Every mode's record.
__global__ __launch_bounds__(256) void k_fast_modes(const LevelProb* __restrict__ probs,
                                                    const FastProb* __restrict__ fp, FastMode* __restrict__ modes, int C)
{
    const LevelProb& P = probs[blockIdx.x];
    const FastProb f = fp[blockIdx.x];
    const int N = P.nx, ny = P.ny, rows = ny + 1, Lp = (rows + C - 1) / C;
    const bool half = f.ends >= kEndsND;
    for (int q = threadIdx.x; q <= N; q += 256) {
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
        const double pn = ipow(rho, ny), den = 1.0 - R0 * R1 * pn * pn;
        FastMode m;
        m.rho = rho;
        m.irho = 1.0 / rho;
        m.scale = 1.0 / (tau * del * 2.0 * N); // both transforms' factors with it
        m.a0 = R0 / den;
        m.a1 = R0 * R1 * pn / den;
        m.b0 = R1;
        m.b1 = R1 * pn;
        m.w = ipow(rho, Lp);
        m.wl = ipow(rho, rows - (rows - 1) / Lp * Lp);
        modes[f.mode0 + q] = m;
    }
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
// Bound by latency (one block a CU at 2000x1000, 2 species): the carries go
// through four chunks of a wave by shuffles, then once through LDS; walked
// chunk by chunk by one thread a mode, and with the modes' constants formed in
// every thread, it took 21.7 us, now 16.6 (32 MB: 6 us); 800x400 14.3 -> 11.1.
// MANY: more blocks than the chip holds, so waves in flight count: the record
// is read where it is used (80 registers for 98; 512 uneven traps 865 -> 819
// us, where the 2000x1000 trap's one round of blocks takes 17.9 for 16.6).
template <typename T, int L, bool MANY>
__global__ __launch_bounds__(1024, MANY && sizeof(T) == 4 && L == 16 ? 6 : 4) void k_fast_lines(const FastJob* __restrict__ jobs, int njobs, const LevelProb* __restrict__ probs,
                             const FastProb* __restrict__ fp, const FastMode* __restrict__ modes, T* __restrict__ io,
                             const double* __restrict__ partial, CgState* st, const int32_t* __restrict__ extra,
                             int32_t* met_at, int k)
{
    __shared__ double red[50];                  // 48 doubles of sums, then the flags
    __shared__ double tot[2][16][kFastModes];   // the waves' totals, up and down
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
    std::conditional_t<MANY, const FastMode&, const FastMode> M = modes[f.mode0 + min(q, N)];
    if (threadIdx.x == 0) {
        ((int*)(red + 48))[0] = k > 0 ? cs.done : 0;
        ((int*)(red + 48))[1] = k > 0 ? met_at[P.prob] : -1;
    }
    double sum[3];
    sum_pairs(partial + 3 * (int64_t)f.pair0, f.npairs, red, sum);
    if (((int*)(red + 48))[0]) return;
    const double rr = sum[0], bb = k > 0 ? cs.bb : sum[1];
    // the first launch settles the scale (fast_e0 is not written here, so every block finds the same)
    int e = 0, drop = 0;
    if (sizeof(T) == 4 && k == 0) {
        const double msq = (rr + bb) / ((double)rows * (double)(N + 1));
        e = cs.fast_e0;
        if (msq > 0.0 && msq < HUGE_VAL) {
            const int own = ilogb(msq) / 2;
            drop = own > e + kFastScaleOff || own < e - kFastScaleOff;
            if (drop) e = own;
        }
    }
    const int app = k == 0 ? 0 : max(0, k - cs.fast_void); // applications done
    // (a block that already reads the first block's entry takes the same way)
    const bool conv = within(rr, cs.tol2 * bb, app > 0 ? cs.fast_rr[(k - 1) & 1] : -1.0, f.unit * sum[2], f.gain,
                             extra[job.prob] > 0, cs.have_prev != 0);
    int first = ((int*)(red + 48))[1];
    if (conv && first < 0) first = app;
    const bool stop = conv && app >= first + extra[job.prob];
    if (job.at == 0 && threadIdx.x == 0) {
        if (k == 0) {
            cs.bb = bb;
            cs.fast_void = drop;
            cs.fast_e = e;
        }
        cs.fast_rr[k & 1] = rr; // (the other one is being read)
        met_at[P.prob] = first;
        cs.done = stop ? 1 : 0;
        if (stop) {
            cs.fast_iter = app;
            cs.rr_true = rr;
        }
    }
    if (stop || drop) return;
    const double rho = M.rho;
    // chunk ends from zero carries: F at the chunk's last row, G before its first
    double F = 0.0, G = 0.0;
#pragma unroll
    for (int l = 0; l < L; ++l)
        if (l < nl) F = rho * F + (double)v[l];
#pragma unroll
    for (int l = L - 1; l >= 0; --l)
        if (l < nl) G = rho * (G + (double)v[l]);
    // carries across the chunks: inclusive over the wave's four, then the waves.
    // (Rows past the last are zero, so the powers there only scale zero.)
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6, cl = (threadIdx.x & 63) / kFastModes;
    const double w1 = M.w, w2 = w1 * w1, w4 = w2 * w2;
    double Fi = F, Gi = G;
    {
        double up = __shfl_up(Fi, kFastModes, 64), dn = __shfl_down(Gi, kFastModes, 64);
        if (cl >= 1) Fi += w1 * up;
        if (cl <= 2) Gi += w1 * dn;
        up = __shfl_up(Fi, 2 * kFastModes, 64);
        dn = __shfl_down(Gi, 2 * kFastModes, 64);
        if (cl >= 2) Fi += w2 * up;
        if (cl <= 1) Gi += w2 * dn;
    }
    if (cl == 3) tot[0][w][m] = Fi;
    if (cl == 0) tot[1][w][m] = Gi;
    __syncthreads();
    double fin = 0.0, gin = 0.0; // at the wave's edges
    for (int e = 0; e < w; ++e) fin = w4 * fin + tot[0][e][m];
    for (int e = nw - 1; e > w; --e) gin = w4 * gin + tot[1][e][m];
    {
        const double up = __shfl_up(Fi, kFastModes, 64), dn = __shfl_down(Gi, kFastModes, 64);
        const double own = F, owng = G, wc[4] = {1.0, w1, w2, w1 * w2};
        F = cl == 0 ? fin : up + (cl == 1 ? wc[1] : cl == 2 ? wc[2] : wc[3]) * fin;
        G = cl == 3 ? gin : dn + (cl == 2 ? wc[1] : cl == 1 ? wc[2] : wc[3]) * gin;
        // w on the whole line at the two walls (in units of c): bottom f_0 +
        // G_0, top F_ny; their threads publish them
        if (c == 0) red[m] = (owng + w1 * G) * M.irho;
        if (nl > 0 && a + nl == rows) red[kFastModes + m] = own + M.wl * F;
    }
    __syncthreads();
    if (!on || nl == 0) return;
    const double w0 = red[m], wn = red[kFastModes + m];
    const double A = M.a0 * w0 + M.a1 * wn, B = M.b0 * wn + M.b1 * A;
    // the walls' terms ride on the recursions' carries: F gets A rho^i, G gets B rho^(ny - i)
    const int last = (rows - 1) / Lp;
    F += A * ipow(w1, c) * M.irho;                              // at row a - 1
    G += c == last ? B : B * ipow(w1, last - c - 1) * M.wl;     // at the chunk's last row
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
            col[(int64_t)l * P.pitch] = (T)(M.scale * (F + (double)g[l]));
        }
}

// The chunk's end: every block takes its problem's residual norm, and where
// the solve has converged the iterate becomes the field (any other field stays
// as the step found it).  The first block of a problem keeps its state.
__global__ __launch_bounds__(256) void k_fast_commit(const FastJob* __restrict__ jobs, int njobs,
                                                     const LevelProb* __restrict__ probs,
                                                     const FastProb* __restrict__ fp, double* __restrict__ u,
                                                     const double* __restrict__ x, const double* __restrict__ partial,
                                                     CgState* st, const int32_t* __restrict__ extra, int32_t* met_at, int k)
{
    __shared__ double red[12];
    __shared__ int was, met, have;
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    const FastProb f = fp[job.prob];
    CgState& cs = st[P.prob];
    if (threadIdx.x == 0) {
        was = cs.done;
        met = met_at[P.prob];
        have = cs.have_prev;
    }
    double sum[3];
    sum_pairs(partial + 3 * (int64_t)f.pair0, f.npairs, red, sum);
    if (was == 2) return;
    const double rr = sum[0];
    const bool kept = have != 0;
    // (a block that already reads the first block's `done` takes the same way)
    const int app = k - cs.fast_void;
    const bool conv = within(rr, cs.tol2 * cs.bb, app > 0 ? cs.fast_rr[(k - 1) & 1] : -1.0, f.unit * sum[2], f.gain,
                             extra[job.prob] > 0, kept);
    const int first = conv && met < 0 ? app : met;
    const bool over = was || (conv && app >= first + extra[job.prob]);
    if (job.at == 0 && threadIdx.x == 0) {
        cs.fast_e0 = cs.fast_e;
        if (!was) {
            cs.fast_iter = app;
            met_at[P.prob] = first;
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

// The stiffness weights of the problems with a tensor field.  Formed in the
// residual from 21 tensor entries a node they made it the largest launch of a
// solve (800x400, 2 species: 39 us an application, now 20; the wall columns, one
// lane's chain of such rows, were half of that).
__global__ __launch_bounds__(256) void k_fast_stiff(const FastJob* __restrict__ jobs, int njobs,
                                                    const LevelProb* __restrict__ probs, double* __restrict__ stiff,
                                                    int64_t sst)
{
    const int t = swizzled_block();
    if (t >= njobs) return;
    const FastJob job = jobs[t];
    const LevelProb& P = probs[job.prob];
    if (!P.aniso) return;
    for (int w = 0; w < 2; ++w) {
        const int i = 2 * job.at + w;
        if (i > P.ny) break;
        for (int j = threadIdx.x; j <= P.nx; j += 256) {
            const int64_t k = P.origin + (int64_t)i * P.pitch + j;
            const double* d = P.tens_d + k;
            Row<double> r;
            aniso_stiffness<double>(P, i, j, d, d + P.tstride, d + 2 * P.tstride, P.pitch, r);
            stiff[k] = r.kw;
            stiff[k + sst] = r.ks;
            stiff[k + 2 * sst] = r.ksw;
        }
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

static bool robin_x(const eq_field_desc& d)
{
    return d.wall[EQ_WALL_LEFT].kind == EQ_BC_ROBIN || d.wall[EQ_WALL_RIGHT].kind == EQ_BC_ROBIN;
}

// The Robin walls across x, which P takes as closed: their part of the operator
// is at most this times P (|u(0)|^2 sqrt((1 + dt gamma) dt D) tanh(W / 2l) is
// the least energy of P with that end value, l = sqrt(dt D / (1 + dt gamma))).
static double robin_part(const eq_field_desc& d)
{
    const double react = 1.0 + d.dt * d.gamma;
    double r = 0.0;
    for (int w : {EQ_WALL_LEFT, EQ_WALL_RIGHT})
        if (d.wall[w].kind == EQ_BC_ROBIN) r = d.wall[w].r >= 0.0 ? std::max(r, d.wall[w].r) : HUGE_VAL;
    if (r == 0.0) return 0.0;
    return d.dt * r / (std::sqrt(react * d.dt * d.D) * std::tanh(0.5 * d.width * std::sqrt(react / (d.dt * d.D))));
}

// Whether the batch's grids and walls allow the solver: x walls closed or
// held (their transforms diagonalise the x matrices) or Robin walls of at most
// twice the closed operator (over 20 applications there), rows that fit a
// block, and dt D of at least the square of the larger spacing, where the
// separable matrix is within a tenth of the operator.  Robin walls across x in
// some problems only would go the same way (the weights are per problem); such
// batches are left to the multigrid solvers, whose fused and separate levels
// are compared with one another on one, by their iteration counts.
static bool fast_shape(const eq_batch* b)
{
    const size_t elem = b->mixed ? sizeof(Cx<float>) : sizeof(Cx<double>);
    std::map<int, bool> fits;
    for (const eq_field_desc& d : b->descs) {
        if (!(robin_part(d) <= 2.0) || robin_x(d) != robin_x(b->descs[0])) return false;
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
    hipFree(F->d_modes);
    hipFree(F->d_stiff);
    hipFree(F->d_tables);
    hipFree(F->d_partial);
    hipFree(F->d_cheb);
    hipFree(F->d_extra);
    hipFree(F->d_met);
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
    int64_t modes = 0;
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
        fp[p].mode0 = modes;
        // the mass couplings that P spreads (sin a sin b / 6 h^2 of the mass
        // against 2 (1 - cos a) + 2 (1 - cos b) of dt D), or the transforms'
        // rounding (FP64: 1e-15 to 4e-15 of the field)
        const eq_field_desc& D = b->descs[p];
        const double mass = P.fd ? 0.0 : (1.0 + D.dt * D.gamma) * P.hx * P.hy / (12.0 * D.dt * D.D);
        const double gain = std::max(mass, sizeof(T) == 4 ? 5e-7 : 3e-15);
        fp[p].gain = gain * gain;
        const double unit = (1.0 + D.dt * D.gamma) * P.hx * P.hy;
        fp[p].unit = unit * unit;
        modes += P.nx + 1;
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
    for (int p = 0; p < b->nprob; ++p) F->chirp.push_back((uint8_t)plans[fp[p].plan].chirp);
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
        hipMalloc((void**)&F->d_partial, sizeof(double) * 3 * pairs) != hipSuccess ||
        hipMalloc((void**)&F->d_modes, sizeof(FastMode) * modes) != hipSuccess ||
        hipMalloc((void**)&F->d_extra, sizeof(int32_t) * b->nprob) != hipSuccess ||
        hipMalloc((void**)&F->d_met, sizeof(int32_t) * b->nprob) != hipSuccess)
        return set_error(EQ_ERR_NOMEM, "fast solver tables");
    EQ_HIP(hipMemsetAsync(F->d_extra, 0, sizeof(int32_t) * b->nprob, s));
    hipLaunchKernelGGL(k_fast_modes, dim3(b->nprob), dim3(256), 0, s, (const LevelProb*)b->levels[0].d_probs,
                       (const FastProb*)F->d_probs, F->d_modes, (int)F->line_c);
    const int np = (int)plans.size();
    hipLaunchKernelGGL(k_fast_tables<T>, dim3(np, 4), dim3(256), 0, s, F->d_plans, (Cx<T>*)F->d_tables);
    if (mmax > 1) {
        const size_t lds = fast_lds_bytes(mmax, sizeof(Cx<T>));
        EQ_HIP(hipFuncSetAttribute((const void*)k_fast_kernel<T, 1024, kFastValuesWide>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFastLds));
        hipLaunchKernelGGL((k_fast_kernel<T, 1024, kFastValuesWide>), dim3(np), dim3(1024), lds, s, F->d_plans, (Cx<T>*)F->d_tables);
    }
    EQ_HIP(hipGetLastError());
    EQ_HIP(hipStreamSynchronize(s)); // the host tables above go out of scope
    const int rg = fast_allow_lds<T, true>(F);
    return rg ? rg : fast_allow_lds<T, false>(F);
}

// The cycle options at their defaults: a caller that sets them asks for that
// multigrid cycle.
static bool default_cycle(const eq_solver_desc& S)
{
    eq_solver_desc d;
    eq_solver_default(&d);
    // (an application is a refinement step, and those are few)
    if (S.kind == EQ_SOLVER_IR_GMG_CG && (S.ir_max_outer != d.ir_max_outer || S.ir_inner_rtol != d.ir_inner_rtol))
        return false;
    return S.mg_pre == d.mg_pre && S.mg_post == d.mg_post && S.mg_omega == d.mg_omega && S.mg_omega2 == d.mg_omega2 &&
           S.mg_coarse_max_nodes == d.mg_coarse_max_nodes && S.mg_max_levels == d.mg_max_levels &&
           S.mg_fuse_max_nodes == d.mg_fuse_max_nodes && S.mg_fuse_pre_max_nodes == d.mg_fuse_pre_max_nodes &&
           S.mg_bottom_lds_bytes == d.mg_bottom_lds_bytes && S.mg_fuse_pre_top == d.mg_fuse_pre_top &&
           S.tile4_min_nodes == d.tile4_min_nodes && S.tile8_min_nodes == d.tile8_min_nodes &&
           S.extrapolate == d.extrapolate && S.mg_level_fused == d.mg_level_fused;
}

// Varying coefficients: not by refinement steps, and an iteration limit that
// leaves room for the applications.
static bool may_vary(const eq_solver_desc& S) { return S.kind != EQ_SOLVER_IR_GMG_CG && S.max_iter >= kChebMax; }

// The plans of a batch that may take the solver (its options, grids and walls
// allow it), or none; where the device has no room for them, none either.
int fast_build(eq_batch* b)
{
    if (b->solver.kind == EQ_SOLVER_JACOBI_CG || !default_cycle(b->solver) || !fast_shape(b)) return EQ_OK;
    if (robin_x(b->descs[0]) && !may_vary(b->solver)) return EQ_OK;
    b->fast = new (std::nothrow) FastSolver();
    if (!b->fast) return set_error(EQ_ERR_NOMEM, "host allocation");
    b->fast->robin_x = robin_x(b->descs[0]); // (all of them)
    const int rc = b->mixed ? fast_build_t<float>(b, b->fast) : fast_build_t<double>(b, b->fast);
    if (rc == EQ_ERR_NOMEM) {
        hipStreamSynchronize(b->stream);
        hipGetLastError();
        fast_free(b);
        return EQ_OK;
    }
    return rc || !(b->fast->robin_x || b->any_tensor) ? rc : fast_refresh(b);
}

// Whether the Chebyshev iteration of fast_refresh is faster than the Krylov
// solver, which takes 5 to 6 iterations for a flow of any strength and 8 for
// Robin walls: microseconds a step as measured from 404x154 to 3000x1800, 2
// species (m: millions of nodes of the batch).  An application takes 28, and a million nodes in it 28 + m (FP32) or
// 32 + 2 m (FP64; the vectors outgrow the caches), by chirp 60 or 80; problems
// drop out one by one, and a kept solution saves 0.15 of the applications.
// Measured, fast against Krylov: flow of s = 0.8 in FP64 900x450 1.48 ms for
// 3.17, 901x449 (chirp) 2.14 for 3.12, 1237x611 (chirp) 3.8 for 3.5, 3000x1800
// 13.2 for 10.8, 2999x1800 (chirp) 22.6 for 10.1; s = 0.25 at 3000x1800 7.1 for
// 8.5; Robin walls at 2999x1800 (chirp) 5.5 for 4.7.  With tensor fields the CG
// takes 11 to 35 iterations on seven-point tensor rows: the fast solver was 1.5
// to 8 times faster on every size.
static bool worth(const eq_batch* b, const std::vector<int>& apps)
{
    bool flow = false;
    double m = 0.0;
    for (const LevelProb& P : b->levels[0].probs) {
        if (P.aniso) return true;
        flow = flow || P.vel;
        m += 1e-6 * (P.nx + 1) * (P.ny + 1);
    }
    const bool f32 = b->mixed;
    double most = 0.0, work = 0.0;
    for (int p = 0; p < b->nprob; ++p) {
        const LevelProb& P = b->levels[0].probs[p];
        const double n = apps[p] > 3 ? 0.85 * apps[p] : apps[p], large = std::min(m, 10.0);
        const double each = b->fast->chirp[p] ? (f32 ? 60.0 : 80.0) : (f32 ? 28.0 + large : 32.0 + 2.0 * large);
        most = std::max(most, n);
        work += n * each * 1e-6 * (P.nx + 1) * (P.ny + 1);
    }
    const double krylov = flow ? (f32 ? 1950.0 + 570.0 * m : 2300.0 + 750.0 * m) : 880.0 + (f32 ? 225.0 : 325.0) * m;
    return 150.0 + 28.0 * most + work <= 0.92 * krylov;
}

// Varying coefficients: the spectrum of P^-1 A, with P the constant operator
// (tensor 1, no flow), is known beforehand.  The stiffness of a tensor field
// lies between its eigenvalues' bounds times the isotropic one, triangle by
// triangle; convection by |v| <= w is skew (up to its ends) and at most
//   s = w dt / (2 sqrt((1 + dt gamma) dt D))
// times P: |S(u, u)| <= dt w |u'| |u| against (1 + dt gamma) |u|^2 + dt D |u'|^2.
// So x <- x + d, d <- alpha z + beta d with the Chebyshev weights of that
// ellipse (Manteuffel, Numer. Math. 28, 1977) converges at a known rate, with
// no inner products: three launches an application, as without them.
// Per step against the V-cycle CG and BiCGStab: a cell tensor of contrast 2 on
// 800x400 4.46 -> 1.07 ms (19 applications), a flow of s = 0.8 on 901x449 2.54
// -> 2.02 (32).
// Robin walls at a rate of 1.5 on the left and right, 900x450 in FP64: 1.20 ->
// 0.47 (nine applications).
// Beyond a rate of 1/2 an application the multigrid solvers are taken (a
// contrast of 9, s = 4/3): there are over 35 applications to a solve.
int fast_refresh(eq_batch* b)
{
    FastSolver* F = b->fast;
    if (!F) return EQ_OK;
    F->general_ok = false; // until everything below is in place
    const bool bicg = b->solver.kind == EQ_SOLVER_GMG_BICGSTAB || b->solver.kind == EQ_SOLVER_MIXED_GMG_BICGSTAB;
    std::vector<double2> tab((size_t)b->nprob * kChebMax, make_double2(1.0, 0.0));
    std::vector<int32_t> extra(b->nprob, 0);
    std::vector<int> apps(b->nprob, 3);
    // from a residual of about the right-hand side to the tolerance
    const double todo = std::log(1.0 / std::max(b->solver.rtol, 1e-15));
    auto needed = [&](double rate) { return rate > 0.0 ? (int)(todo / std::log(1.0 / rate)) + 1 : 3; };
    double worst = 0.0;
    int most = 0;
    for (int p = 0; p < b->nprob; ++p) {
        const LevelProb& P = b->levels[0].probs[p];
        const eq_field_desc& D = b->descs[p];
        const double robin = robin_part(D);
        if (!P.aniso && !P.vel && robin == 0.0) continue;
        const double h = std::max(P.hx, P.hy), react = 1.0 + D.dt * D.gamma;
        const double off = react * h * h / (6.0 * D.dt * D.D); // the mass couplings that P leaves out
        double lo = 1.0, hi = 1.0, s = 0.0;
        if (P.aniso) {
            if ((int)b->tens_bounds.size() <= p) return EQ_OK;
            lo = std::min(lo, b->tens_bounds[p][0]);
            hi = std::max(hi, b->tens_bounds[p][1]);
            if (P.celltens) { // a coupling may write over a field that was set
                lo = std::min(lo, b->cell_bounds[p][0]);
                hi = std::max(hi, b->cell_bounds[p][1]);
            }
        }
        if (P.vel) {
            double w = 0.0;
            for (double v : b->vel_host[p][0]) w = std::max(w, std::isfinite(v) ? std::fabs(v) : HUGE_VAL);
            s = 0.5 * w * std::sqrt(D.dt / (react * D.D));
        }
        hi += robin;
        const double d = 0.5 * (lo + hi), a = 0.5 * (hi - lo) + off, c2 = a * a - s * s;
        const double rate = (a + s) / (d + std::sqrt(d * d - c2));
        if (!(lo > 0.0) || !(rate <= 0.5) || (P.vel && !bicg)) return EQ_OK;
        worst = std::max(worst, rate);
        // The residual has a floor of rounding (the iterate's own, times the
        // largest eigenvalue) that the error does not share, so a tighter
        // tolerance may be out of reach: a fixed number of applications takes
        // the error down to what the multigrid solvers leave at best: another
        // factor of 1e5 with flow (BiCGStab overshoots: 4e-14 to 1e-11 of the
        // field; a factor of 1000 left 2e-13), 300 with a tensor (CG: 2e-14 to
        // 3e-13; 100 left up to 1e-13) and 1e4 for Robin walls alone, whose
        // rate is small: two or three (one left 1e-13).
        extra[p] = rate > 0.0 ? (int)std::ceil(std::log(P.vel ? 1e5 : P.aniso ? 3e2 : 1e4) / std::log(1.0 / rate)) : 0;
        most = std::max(most, extra[p]);
        apps[p] = needed(rate) + extra[p];
        double2* w = tab.data() + (size_t)p * kChebMax;
        double al = 1.0 / d;
        w[0] = make_double2(al, 0.0);
        for (int k = 1; k < kChebMax; ++k) {
            al = k == 1 ? 2.0 * d / (2.0 * d * d - c2) : 1.0 / (d - 0.25 * c2 * al);
            w[k] = make_double2(al, d * al - 1.0);
        }
    }
    if ((worst > 0.0) && !worth(b, apps)) return EQ_OK;
    for (int& r : F->recent[1]) r = std::min(needed(worst) + most, FastSolver::kGraphs - 1);
    EQ_HIP(hipStreamSynchronize(b->stream));
    bool aniso = false;
    for (const LevelProb& P : b->levels[0].probs) aniso = aniso || P.aniso;
    if (aniso != (F->d_stiff != nullptr)) {
        fast_drop_graphs(b); // they hold the old address
        hipFree(F->d_stiff);
        F->d_stiff = nullptr;
        F->stiff_stride = b->levels[0].pool;
        if (aniso && hipMalloc((void**)&F->d_stiff, sizeof(double) * 3 * F->stiff_stride) != hipSuccess) {
            F->d_stiff = nullptr;
            hipGetLastError();
            return EQ_OK; // no room: the multigrid solvers need none
        }
        if (aniso) EQ_HIP(hipMemset(F->d_stiff, 0, sizeof(double) * 3 * F->stiff_stride));
    }
    if (!F->d_cheb && hipMalloc((void**)&F->d_cheb, sizeof(double2) * tab.size()) != hipSuccess) {
        F->d_cheb = nullptr;
        hipGetLastError();
        return EQ_OK;
    }
    EQ_HIP(hipMemcpy(F->d_cheb, tab.data(), sizeof(double2) * tab.size(), hipMemcpyHostToDevice));
    EQ_HIP(hipMemcpy(F->d_extra, extra.data(), sizeof(int32_t) * extra.size(), hipMemcpyHostToDevice));
    F->general_ok = true;
    return EQ_OK;
}

// A change of tensor fields or velocities that fails part of the way leaves
// problems with coefficients that the tables here do not cover (a tensor
// without stiffness weights): until fast_refresh has seen it through, steps
// with varying coefficients take the multigrid solvers.
void fast_forget(eq_batch* b)
{
    if (b->fast) b->fast->general_ok = false;
}

// Whether this step takes the fast solver: the cycle options are at their
// defaults (autotune may have changed them since the batch was created), and
// where coefficients vary their bounds and the iteration limit allow it.
bool fast_applies(const eq_batch* b)
{
    if (!b->fast || b->fast->rest > 0) return false;
    const bool varying = b->any_tensor || b->fast->robin_x;
    return default_cycle(b->solver) && (!varying || (b->fast->general_ok && may_vary(b->solver)));
}

// ------------------------------------------------------------ host: one solve

// Applications k0 .. k0 + n - 1, then the residual's check and the commit.
template <typename T, bool GEN>
static void fast_chunk(eq_batch* b, int k0, int n)
{
    FastSolver* F = b->fast;
    hipStream_t s = b->stream;
    const LevelProb* probs = b->levels[0].d_probs;
    T* z = (T*)b->z;
    const double nodes = b->levels[0].nodes_all;
    int32_t njobs = 0;
    for (const FastClass& c : F->classes) njobs += c.njobs;
    if (k0 == 0)
        launch(b, EQ_KERNEL_SOLVE_ONCE, 0.0, k_fast_start, dim3(grid8(njobs)), dim3(256), 0, s,
               (const FastJob*)F->d_jobs, njobs, probs, b->xprev, (const CgState*)b->d_state);
    if (GEN && k0 == 0 && F->d_stiff)
        launch(b, EQ_KERNEL_SOLVE_ONCE, nodes * 48.0, k_fast_stiff, dim3(grid8(njobs)), dim3(256), 0, s,
               (const FastJob*)F->d_jobs, njobs, probs, F->d_stiff, F->stiff_stride);
    for (int k = k0; k < k0 + n; ++k) {
        fast_forward<T, GEN>(b, k, k == k0);
        const dim3 lg(grid8(F->nline)), lb(F->line_c * kFastModes);
        auto lines = [&](auto kern) {
            launch(b, EQ_KERNEL_BOTTOM, nodes * 2 * sizeof(T), kern, lg, lb, 0, s, (const FastJob*)F->d_lines, F->nline,
                   probs, (const FastProb*)F->d_probs, (const FastMode*)F->d_modes, z, (const double*)F->d_partial, b->d_state, (const int32_t*)F->d_extra, F->d_met, k);
        };
        const bool many = F->nline > 1024; // four blocks a CU
        if (F->line_rows <= 1024)
            many ? lines(k_fast_lines<T, 16, true>) : lines(k_fast_lines<T, 16, false>);
        else if (F->line_rows <= 2048)
            many ? lines(k_fast_lines<T, 32, true>) : lines(k_fast_lines<T, 32, false>);
        else
            many ? lines(k_fast_lines<T, 64, true>) : lines(k_fast_lines<T, 64, false>);
        fast_backward<T, GEN>(b, k);
    }
    launch(b, EQ_KERNEL_SOLVE_ONCE, nodes * 16.0, k_fast_check<GEN>, dim3(grid8(njobs)), dim3(256), 0, s,
           (const FastJob*)F->d_jobs, njobs, probs, (const FastProb*)F->d_probs, (const FastRows*)F->d_rows,
           (const double*)b->u, (const double*)b->xprev, (const double*)F->d_stiff, F->stiff_stride, F->d_partial,
           (const CgState*)b->d_state);
    launch(b, EQ_KERNEL_SOLVE_ONCE, nodes * 16.0, k_fast_commit, dim3(grid8(njobs)), dim3(256), 0, s,
           (const FastJob*)F->d_jobs, njobs, probs, (const FastProb*)F->d_probs, b->u, (const double*)b->xprev,
           (const double*)F->d_partial, b->d_state, (const int32_t*)F->d_extra, F->d_met, k0 + n);
}

// One step's solve.  handled = false: some residual did not reach the tolerance
// in the applications given to it, at most the kind's iteration limit; those
// problems (h_state: not done) still hold the step's fields, for the multigrid
// solver to take, and the others their solutions.
template <typename T>
static int fast_solve_t(eq_batch* b, bool profiling, bool* handled)
{
    FastSolver* F = b->fast;
    const eq_solver_desc& S = b->solver;
    hipStream_t s = b->stream;
    *handled = true;
    const bool graphs = S.use_graphs && !profiling;
    const int gen = b->any_tensor || F->robin_x ? 1 : 0;
    auto applications = [&](int k0, int n) {
        if (gen)
            fast_chunk<T, true>(b, k0, n);
        else
            fast_chunk<T, false>(b, k0, n);
    };
    int* recent = F->recent[gen];
    int chunk = *std::max_element(recent, recent + 4);
    const int limit = S.kind == EQ_SOLVER_IR_GMG_CG ? S.ir_max_outer : S.max_iter;
    const int give_up = std::min(gen ? kChebMax : kFastGiveUp, limit);
    chunk = std::max(1, std::min({chunk, give_up, FastSolver::kGraphs - 1}));
    for (int k0 = 0;;) {
        if (k0 == 0 && graphs) {
            hipGraphExec_t& ge = F->graph[chunk];
            if (!ge) {
                hipGraph_t g = nullptr;
                EQ_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                F->acct[chunk] = Acct{};
                b->acct_to = &F->acct[chunk];
                applications(0, chunk);
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
            applications(k0, chunk);
        }
        k0 += chunk;
        EQ_HIP(hipMemcpyAsync(b->h_state, b->d_state, sizeof(CgState) * b->nprob, hipMemcpyDeviceToHost, s));
        EQ_HIP(hipGetLastError());
        EQ_HIP(hipStreamSynchronize(s));
        bool all = true;
        for (int p = 0; p < b->nprob; ++p) all = all && b->h_state[p].done;
        if (all) break;
        if (k0 >= give_up) {
            // what holds it back (a tolerance below rounding, say) may well
            // hold at the next step: twice as many without it each time
            F->last_rest = std::min(63, 2 * F->last_rest + 1);
            F->rest = F->last_rest;
            *handled = false;
            return EQ_OK;
        }
        chunk = std::min(2, give_up - k0);
    }
    F->last_rest = 0;
    int most = 1;
    for (int p = 0; p < b->nprob; ++p) most = std::max(most, b->h_state[p].iter);
    recent[F->at[gen]] = std::min(most, FastSolver::kGraphs - 1);
    F->at[gen] = (F->at[gen] + 1) & 3;
    return EQ_OK;
}

void fast_rest(eq_batch* b)
{
    if (b->fast && b->fast->rest > 0) --b->fast->rest;
}

int fast_solve(eq_batch* b, bool profiling, bool* handled)
{
    return b->mixed ? fast_solve_t<float>(b, profiling, handled) : fast_solve_t<double>(b, profiling, handled);
}

} // namespace eqk
